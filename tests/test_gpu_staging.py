"""Host copies through the pinned buffers: fields written and read back are the
same bytes, for rows shorter and longer than the pitch, copies of one piece and
of several (8 MiB each), in both directions."""
import numpy as np
import pytest

from flowlb_amd import core

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(2, 2), (63, 5), (64, 5), (65, 7), (1999, 600), (2048, 1100),
                                   (1500, 1399)])
@pytest.mark.parametrize("storage", ["fp32", "fp64"])
def test_round_trip(nx, ny, storage):
    rng = np.random.default_rng(3)
    fl = np.full(nx * ny, core.FLUID, np.uint8)
    fl[: nx] = core.WALL
    rho0 = (1 + 0.1 * rng.random(nx * ny)).astype(np.float32)
    u0 = (0.1 * rng.random(2 * nx * ny)).astype(np.float32)
    with core.Solver(fl, nx, ny, core.default_options(problem=core.FREE_SURFACE, storage=storage),
                     rho0=rho0, u0=u0) as s:
        f = rng.random(9 * nx * ny)
        mass, phi, ex = (rng.random(nx * ny) for _ in range(3))
        s.write_populations64(f)
        s.set_fs_fields64(mass, phi, ex)
        g = s.read64()
        f2 = s.populations64()
    one = (lambda a: a) if storage == "fp64" else (lambda a: a.astype(np.float32).astype(np.float64))
    assert np.array_equal(g["flags"], fl)
    assert np.array_equal(g["rho"], rho0.astype(np.float64))
    assert np.array_equal(g["u"], u0.astype(np.float64))
    for k, a in (("mass", mass), ("phi", phi), ("excess", ex)):
        assert np.array_equal(g[k], one(a)), k
    # Populations are stored less their weight: a rounding each way.
    assert np.abs(f2 - f).max() <= (3e-16 if storage == "fp64" else 1.5e-7)
