"""Passes of every length (2, 3 and 4 steps forward, 2 and 3 in reverse) and of
many chunk heights, set by flb_test_pass_shape, against the same steps one by
one.  Small grids take passes of three steps and four rows by themselves (two in
reverse); the shapes here are those that the rules give larger grids.  Every cell
is evaluated with the same arithmetic: equal bit for bit.
"""
import numpy as np
import pytest

from flowlb_amd import core
from test_gpu_march import _domain

pytestmark = pytest.mark.gpu

# Steps and rows per chunk: one row, remainders of every kind, more rows than the domain.
SHAPES = [(2, 1), (2, 16), (3, 2), (3, 7), (4, 1), (4, 5), (4, 16), (4, 32), (4, 100)]


def shape(s, steps, rows, reverse=-1, reverse_rows=0):
    core.check(core.lib().flb_test_pass_shape(s.h, steps, rows, reverse, reverse_rows), s.h,
               "flb_test_pass_shape")


def run(domain, calls, steps, rows, alpha=None, **opt):
    nx, ny, (fl, rho0, u0) = domain
    with core.Solver(fl, nx, ny, core.default_options(tau=0.6, **opt), rho0=rho0, u0=u0) as s:
        shape(s, steps, rows)
        if alpha is not None:
            s.set_brinkman(alpha)
        for n in calls:
            s.step(n)
        return dict(s.read64(), f=s.populations64(), t=s.time)


def same(one, many, what):
    for k in ("f", "u", "rho", "flags"):
        assert np.isfinite(one[k]).mean() > 0.95, (what, k)
        assert np.array_equal(one[k], many[k], equal_nan=True), (what, k)


@pytest.mark.parametrize("storage", ["fp32", "fp16s", "bf16s", "fp64"])
@pytest.mark.parametrize("kind", ["open", "channel", "scattered"])
def test_every_shape(storage, kind):
    rng = np.random.default_rng(17)
    for nx, ny in [(131, 47), (61, 70), (300, 33), (9, 5)]:
        d = nx, ny, _domain(nx, ny, kind, rng)
        one = run(d, [1] * 22, 0, 0, storage=storage)
        for steps, rows in SHAPES:
            # Passes of `steps` from even and odd times, two in a row, a shorter one.
            calls = [steps, 1, 2 * steps, steps]
            calls.append(22 - sum(calls))
            many = run(d, [n for n in calls if n], steps, rows, storage=storage)
            assert one["t"] == many["t"] == 22
            same(one, many, (nx, ny, steps, rows))


@pytest.mark.parametrize("storage", ["fp32", "fp16s", "bf16s", "fp64"])
@pytest.mark.parametrize("opt", [dict(), dict(use_force=1, fx=1e-5), dict(collision=1),
                                 dict(collision=1, smagorinsky=1), dict(smagorinsky=1),
                                 dict(collision=1, use_force=1, fx=1e-5),
                                 dict(collision=2, use_force=1, fx=1e-5, fy=-2e-5, smagorinsky=1),
                                 dict(alpha=1), dict(alpha=1, use_force=1, fx=1e-5),
                                 dict(alpha=1, smagorinsky=1)])
def test_every_model(storage, opt):
    rng = np.random.default_rng(18)
    kw = {k: v for k, v in opt.items() if k != "alpha"}
    for kind in ("channel", "scattered"):
        nx, ny = 190, 41
        d = nx, ny, _domain(nx, ny, kind, rng)
        alpha = rng.random(nx * ny).astype(np.float32) if opt.get("alpha") else None
        one = run(d, [1] * 13, 0, 0, alpha, storage=storage, **kw)
        for steps, rows in ((2, 9), (3, 6), (4, 11)):
            same(one, run(d, [steps, 1, 12 - steps], steps, rows, alpha, storage=storage, **kw),
                 (kind, steps))


@pytest.mark.parametrize("nx,ny,storage", [(601, 601, "fp32"), (2048, 700, "fp32"),
                                           (2048, 700, "fp16s"), (3000, 1000, "bf16s"),
                                           (1201, 601, "fp64")])
def test_sizes_that_take_four_steps(nx, ny, storage):
    """Four steps per pass from 1.5 wavefronts per SIMD at more than three rows
    on: chunks of 5 to 32 rows with a remainder, by the rule's own choice."""
    assert -(-nx // 58) * ny > 3 * 6 * 256  # 256 CUs
    d = nx, ny, _domain(nx, ny, "channel", np.random.default_rng(19))
    one = run(d, [1] * 10, 0, 0, storage=storage)
    same(one, run(d, [4, 1, 5], -1, 0, storage=storage), (nx, ny))


@pytest.mark.parametrize("storage", ["fp32", "fp16s", "bf16s"])
@pytest.mark.parametrize("force", [False, True])
def test_batch_shapes(storage, force):
    rng = np.random.default_rng(20)
    inst = []
    for k, (nx, ny) in enumerate([(65, 9), (130, 41), (57, 4), (300, 33), (64, 64)]):
        fl, rho0, u0 = _domain(nx, ny, "channel" if k % 2 else "scattered", rng)
        fl[-1] = fl[0] = core.WALL
        inst.append(dict(nx=nx, ny=ny, tau=0.6 + 0.05 * k, flags=fl, rho0=rho0, u0=u0,
                         use_force=int(force and k != 2), fx=1e-5 * k, fy=-1e-5))

    def go(steps, rows, calls, chunk):
        with core.Batch(inst, storage=storage) as b:
            b._check(core.lib().flb_test_batch_pass_shape(b.h, steps, rows), "pass shape")
            b.configure(block_x=128, grid=0, graph_chunk=chunk)
            for n in calls:
                b.step(n)
            assert b.time == 41
            return [dict(f=b.populations(i), **b.read(i)) for i in range(len(inst))]

    one = go(0, 0, [41], 0)
    for steps, rows in SHAPES:
        for calls, chunk in (([41], 0), ([2 * steps, 1, 40 - 2 * steps], 6)):
            for i, (a, g) in enumerate(zip(one, go(steps, rows, calls, chunk))):
                for k in a:
                    assert np.isfinite(a[k]).mean() > 0.95
                    assert np.array_equal(a[k], g[k], equal_nan=True), (steps, rows, chunk, i, k)


@pytest.mark.parametrize("storage", ["fp32", "fp64"])
@pytest.mark.parametrize("nx,ny,kind", [(131, 37, "channel"), (61, 33, "scattered"),
                                        (5, 70, "scattered"), (70, 9, "open")])
def test_reverse_shapes(storage, nx, ny, kind):
    """Gradients by reverse passes of 2 and 3 steps, alone and mixed with single
    steps (segments that leave one or two), against single reverse steps.
    dJ/du_inlet is summed in an order that varies: see test_gpu_adjoint_passes.py."""
    rng = np.random.default_rng(nx * 100 + ny)
    fl, rho0, u0 = _domain(nx, ny, kind, rng)
    steps, t0, t1 = 23, 5, 20  # neither end of the average is a multiple of a pass
    alpha = np.where(rng.random(nx * ny) < 0.3, rng.random(nx * ny), 0).astype(np.float32)
    for drag, force in ((True, False), (True, True), (False, True)):
        opt = dict(use_force=1, fx=1e-5, fy=-2e-5) if force else {}

        def grad(reverse, rows, ckpt, budget):
            with core.Solver(fl, nx, ny, core.default_options(tau=0.6, storage=storage, **opt),
                             rho0=rho0, u0=u0) as s:
                shape(s, -1, 0, reverse, rows)
                if drag:
                    s.set_brinkman(alpha)
                return s.adjoint(steps, nx // 2, t0, t1, ckpt=ckpt, trace_budget_bytes=budget)[:3]

        J, g, duin = grad(0, 0, steps, 0)
        assert np.isfinite(J) and np.isfinite(g).all() and (not drag or g.any())
        for reverse, rows in ((2, 2), (2, 9), (3, 1), (3, 4), (3, 5), (3, 16)):
            for ckpt, budget in ((steps, 0), (5, 1), (7, 1), (4, 0)):
                other = grad(reverse, rows, ckpt, budget)
                assert other[0] == J, (reverse, rows, ckpt)
                np.testing.assert_array_equal(other[1], g, err_msg=str((reverse, rows, ckpt)))
                assert abs(other[2] - duin) <= 1e-9 * abs(duin)


@pytest.mark.parametrize("storage", ["fp32", "fp64"])
def test_gradient_of_the_size_that_takes_three(storage):
    nx, ny, steps = 1024, 256, 11
    fl, rho0, u0 = _domain(nx, ny, "channel", np.random.default_rng(21))
    alpha = np.where(np.random.default_rng(22).random(nx * ny) < 0.3, 0.5, 0).astype(np.float32)
    out = []
    for reverse in (0, -1):
        with core.Solver(fl, nx, ny, core.default_options(tau=0.6, storage=storage), rho0=rho0,
                         u0=u0) as s:
            shape(s, -1, 0, reverse, 0)
            s.set_brinkman(alpha)
            out.append(s.adjoint(steps, 4, 3, 9, ckpt=steps))
    assert out[0][0] == out[1][0] and out[0][1].any()
    np.testing.assert_array_equal(out[0][1], out[1][1])
    assert abs(out[0][2] - out[1][2]) <= 1e-9 * abs(out[0][2])


# Single steps, which domains and runs that take no passes still use: the batch's
# tile kernel with its orders, grids and graphs, and the block sizes of a handle.
@pytest.mark.parametrize("storage", ["fp32", "bf16s"])
@pytest.mark.parametrize("graph_chunk,grid,order", [(0, 512, "rows"), (10, 512, "rows"),
                                                    (10, 0, "rows"), (10, 0, "instance"),
                                                    (0, 512, "bands"), (4, 0, "bands")])
def test_batch_single_steps_equal_handles(storage, graph_chunk, grid, order):
    rng = np.random.default_rng(23)
    inst = []
    for k, (nx, ny) in enumerate([(65, 9), (130, 41), (57, 4), (300, 33), (640, 70)]):
        fl, rho0, u0 = _domain(nx, ny, "channel" if k % 2 else "scattered", rng)
        fl[:nx] = fl[-nx:] = core.WALL
        inst.append(dict(nx=nx, ny=ny, tau=0.6 + 0.05 * k, flags=fl, rho0=rho0, u0=u0))
    with core.Batch(inst, storage=storage) as b:
        b._check(core.lib().flb_test_batch_pass_shape(b.h, 0, 0), "pass shape")
        b.set_order(order)
        b.configure(block_x=128, grid=grid, graph_chunk=graph_chunk)
        b.step(37)
        got = [dict(f=b.populations(i), **b.read(i)) for i in range(len(inst))]
    for d, g in zip(inst, got):
        o = core.default_options(tau=d["tau"], storage=storage)
        with core.Solver(d["flags"], d["nx"], d["ny"], o, rho0=d["rho0"], u0=d["u0"]) as s:
            s.step(37)
            want = dict(s.read(), f=s.populations())
        for k in g:
            assert np.array_equal(g[k], want[k], equal_nan=True), (d["nx"], k)


@pytest.mark.parametrize("block_x", [64, 128, 512, 1024])
def test_block_sizes_of_single_steps(block_x):
    d = 700, 61, _domain(700, 61, "channel", np.random.default_rng(24))
    same(run(d, [13], 0, 0), run(d, [13], 0, 0, block_x=block_x), block_x)
