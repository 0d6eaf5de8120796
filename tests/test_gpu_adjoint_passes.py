"""Gradients by passes of several steps against the same gradients step by step.

With a checkpoint at every step each forward and reverse sweep takes one step;
with wider intervals they take two to four in a pass.  Both evaluate every cell
with the same arithmetic, and the discharge and dJ/dalpha are summed in the order
of the steps, so these have to be equal bit for bit.  dJ/du_inlet is an FP64 sum
whose order varies: up to 24 x 2000 terms, 5e-12 relative to the sum of their
magnitudes, of which cancellation may leave half a percent.
"""
import numpy as np
import pytest

from flowlb_amd import core
from test_gpu_march import _domain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage", ["fp32", "fp64"])
@pytest.mark.parametrize("nx,ny,kind", [
    (131, 37, "channel"), (9, 5, "channel"), (58, 17, "channel"), (61, 300, "channel"),
    (131, 37, "scattered"), (61, 33, "scattered"), (5, 70, "scattered"), (70, 9, "open")])
def test_gradient_by_passes(storage, nx, ny, kind):
    rng = np.random.default_rng(nx * 1000 + ny)
    fl, rho0, u0 = _domain(nx, ny, kind, rng)
    steps, t0, t1 = 24, 5, 21  # neither end of the average is a multiple of a pass
    alpha = np.where(rng.random(nx * ny) < 0.3, rng.random(nx * ny), 0).astype(np.float32)
    for drag, force, column in ((True, False, nx // 2), (True, True, nx - 2), (False, True, 0)):
        opt = dict(use_force=1, fx=1e-5, fy=-2e-5) if force else {}
        out = []
        for ckpt, budget in ((1, 0), (steps, 0), (7, 1)):
            with core.Solver(fl, nx, ny, core.default_options(tau=0.6, storage=storage, **opt),
                             rho0=rho0, u0=u0) as s:
                if drag:
                    s.set_brinkman(alpha)
                J, g, duin, _ = s.adjoint(steps, column, t0, t1, ckpt=ckpt,
                                          trace_budget_bytes=budget)
                assert s.objective(steps, column, t0, t1) == J
            out.append((J, g, duin))
        J, g, duin = out[0]
        assert np.isfinite(J) and np.isfinite(g).all() and (not drag or g.any())
        for other in out[1:]:
            assert other[0] == J
            np.testing.assert_array_equal(other[1], g)
            assert abs(other[2] - duin) <= 1e-9 * abs(duin)
