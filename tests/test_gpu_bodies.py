"""Free surface: tiles inside a body of fluid, whose masses and flags
stream-collide stores only when they are read, against runs without such tiles
(flb_set_fs_fields resets the work map every step, so every tile takes the
general path).  Same arithmetic in both: equal bit for bit.
"""
import numpy as np
import pytest

from flowlb_amd import core

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,storage", [(700, 200, "fp32"), (703, 201, "fp16s"),
                                           (641, 217, "bf16s"), (700, 200, "fp64")])
def test_bodies_equal_general_path(nx, ny, storage):
    flags, _, u0 = core.build_culvert(nx, ny, True, (core.WALL,) * 4, (int(nx * 0.7), int(nx * 0.75)),
                                      ny // 6, water=(int(nx * 0.6), int(ny * 0.8)))
    fl = flags.copy()
    fl[(fl & 7) == core.INTERFACE] = core.GAS
    fl.reshape(ny, nx)[60:66, 200:206] = core.GAS  # a bubble that collapses: bodies come and go
    flags = core.seed_free_surface(fl, nx, ny)
    rng = np.random.default_rng(nx)
    rho0 = (1 + 2e-4 * (rng.random(nx * ny) - 0.5)).astype(np.float32)
    o = core.default_options(tau=0.6, fx=5e-5, fy=-2e-4, use_force=1, problem=core.FREE_SURFACE,
                             storage=storage, gas_check_corrected=1)
    out = []
    for calls in ([1, 37, 2, 60, 50], [1] * 150):
        with core.Solver(flags, nx, ny, o, rho0=rho0, u0=u0) as s:
            s.set_fs_fields(*core.init_free_surface_fields(flags))
            for n in calls:
                s.step(n)
                if len(calls) > 5:
                    g = s.read64()
                    s.set_fs_fields64(g["mass"], g["phi"], g["excess"])
            out.append((s.read64(), s.populations64()))
    (a, fa), (b, fb) = out
    assert (a["flags"] != flags).sum() > 200  # the surface moved
    for k in ("flags", "mass", "excess", "phi", "u", "rho"):
        np.testing.assert_array_equal(a[k], b[k], err_msg=k)
    np.testing.assert_array_equal(fa, fb)
