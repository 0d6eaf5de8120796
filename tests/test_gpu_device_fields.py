"""Values a program writes into the device fields of a single-phase handle
(flb_device_fields): the velocity inlet cells prescribe and the density outlet
cells keep are read from there at every step, in passes of several steps as in
single ones (bit for bit), and nothing else is.
"""
import ctypes as C

import numpy as np
import pytest

from flowlb_amd import core
from test_gpu_march import _domain

pytestmark = pytest.mark.gpu
H2D, D2H = 1, 2


def _edit(s, ptr, planes, dtype, f):
    pitch, _ = s.layout
    a = np.empty((planes, s.ny, pitch), dtype)
    p = a.ctypes.data_as(C.c_void_p)
    s.sync()
    assert core.hip().hipMemcpy(p, C.c_void_p(ptr), a.nbytes, D2H) == 0
    f(a[:, :, :s.nx])
    assert core.hip().hipMemcpy(C.c_void_p(ptr), p, a.nbytes, H2D) == 0
    assert core.hip().hipDeviceSynchronize() == 0


@pytest.mark.parametrize("storage", ["fp32", "fp16s", "fp64"])
@pytest.mark.parametrize("kind,force", [("channel", False), ("channel", True),
                                        ("scattered", False)])
def test_written_inlet_velocity_and_outlet_density(storage, kind, force):
    dtype = np.float64 if storage == "fp64" else np.float32
    for nx, ny in [(131, 37), (9, 12)]:
        rng = np.random.default_rng(31)
        fl, rho0, u0 = _domain(nx, ny, kind, rng)
        opt = dict(use_force=1, fx=1e-5) if force else {}
        out = []
        for calls in ([1] * 18, [2, 7, 5, 4]):
            new = np.random.default_rng(32)
            with core.Solver(fl, nx, ny, core.default_options(tau=0.6, storage=storage, **opt),
                             rho0=rho0, u0=u0) as s:
                done = 0
                for n in calls:
                    if done in (2, 9):
                        u, rho = s.device_fields()[:2]
                        du = 0.02 * new.random((2, ny, nx)).astype(dtype)
                        dr = 1e-3 * new.random((1, ny, nx)).astype(dtype)
                        _edit(s, u, 2, dtype, lambda a: a.__iadd__(du))
                        _edit(s, rho, 1, dtype, lambda a: a.__iadd__(dr))
                    s.step(n)
                    done += n
                out.append(dict(f=s.populations64(), **s.read64()))
        inlet = (fl & core.INLET) != 0
        assert np.abs(out[0]["u"][:nx * ny][inlet] - u0[:nx * ny][inlet]).max() > 1e-3
        for k in ("f", "rho", "u"):
            assert np.isfinite(out[0][k]).mean() > 0.95
            assert np.array_equal(out[0][k], out[1][k], equal_nan=True), (nx, ny, k)
