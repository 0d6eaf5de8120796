"""Several steps in one pass (flb_march.h) against the same steps one by one.

flb_step(n) runs passes of two to four steps, flb_step(1) the single-step
kernel.  Both evaluate every cell with the same arithmetic in the same order, so
the populations and fields have to be equal bit for bit: the tolerance is zero.
"""
import numpy as np
import pytest

from flowlb_amd import core

pytestmark = pytest.mark.gpu


def _domain(nx, ny, kind, rng):
    fl = np.full((ny, nx), core.FLUID, np.uint8)
    u0 = np.zeros((2, ny, nx), np.float32)
    if kind != "open":  # open: periodic both ways, no walls
        fl[0] = fl[-1] = core.WALL
    if kind == "channel":
        fl[1:-1, 0] = core.INLET
        fl[1:-1, -1] = core.OUTLET
    elif kind == "scattered":
        # Walls anywhere (whole rows of a strip among them), inlets and outlets
        # inside the domain: beside walls, beside each other, two deep.
        fl[rng.random((ny, nx)) < 0.2] = core.WALL
        fl[ny // 2, : max(1, nx - 2)] = core.WALL
        fl[rng.random((ny, nx)) < 0.02] = core.INLET
        fl[rng.random((ny, nx)) < 0.02] = core.OUTLET
        fl[:, 0][fl[:, 0] == core.OUTLET] = core.FLUID  # outside the pass's rule
        fl[:, -1][fl[:, -1] == core.INLET] = core.FLUID
    u0[0][fl == core.INLET] = 0.03
    rho0 = (1 + 1e-3 * (rng.random((ny, nx)) - 0.5)).astype(np.float32)
    return fl.ravel(), rho0.ravel(), u0.ravel()


def _run(fl, nx, ny, rho0, u0, calls, alpha=None, **opt):
    with core.Solver(fl, nx, ny, core.default_options(tau=0.6, **opt), rho0=rho0, u0=u0) as s:
        if alpha is not None:
            s.set_brinkman(alpha)
        for n in calls:
            s.step(n)
        g = s.read64()
        g["f"] = s.populations64()
        g["t"] = s.time
    return g


# Widths around the strips of 58, 60 and 62 columns and the 64 lanes, rows
# around the smallest a pass takes (4) and a chunk's remainder.
SIZES = [(2, 4), (5, 7), (57, 9), (58, 5), (59, 4), (63, 12), (64, 33), (65, 6), (117, 31),
         (129, 3), (190, 70)]


@pytest.mark.parametrize("storage", ["fp32", "fp16s", "bf16s", "fp64"])
@pytest.mark.parametrize("kind", ["open", "channel", "scattered"])
def test_passes_equal_single_steps(storage, kind):
    rng = np.random.default_rng(7)
    for nx, ny in SIZES:
        fl, rho0, u0 = _domain(nx, ny, kind, rng)
        if fl[-1] & core.INLET or fl[0] & core.OUTLET:
            continue
        one = _run(fl, nx, ny, rho0, u0, [1] * 14, storage=storage)
        # From even and odd times: passes of 4, 3 and 2 with single steps between.
        many = _run(fl, nx, ny, rho0, u0, [4, 1, 3, 1, 5], storage=storage)
        assert one["t"] == many["t"] == 14
        for k in ("f", "u", "rho", "flags"):
            assert np.array_equal(one[k], many[k], equal_nan=True), (nx, ny, k)


@pytest.mark.parametrize("storage", ["fp32", "bf16s", "fp64"])
@pytest.mark.parametrize("opt", [dict(collision=1), dict(collision=1, smagorinsky=1),
                                 dict(collision=2, use_force=1, fx=1e-5, fy=-2e-5),
                                 dict(use_force=1, fx=1e-5), dict(smagorinsky=1),
                                 dict(alpha=1, use_force=1, fx=1e-5)])
def test_passes_equal_single_steps_models(storage, opt):
    rng = np.random.default_rng(8)
    opt = dict(opt)
    for nx, ny in [(65, 9), (190, 70)]:
        fl, rho0, u0 = _domain(nx, ny, "channel", rng)
        alpha = rng.random(nx * ny).astype(np.float32) if opt.get("alpha") else None
        kw = {k: v for k, v in opt.items() if k != "alpha"}
        one = _run(fl, nx, ny, rho0, u0, [1] * 14, alpha, storage=storage, **kw)
        many = _run(fl, nx, ny, rho0, u0, [4, 1, 3, 1, 5], alpha, storage=storage, **kw)
        for k in ("f", "u", "rho"):
            assert np.array_equal(one[k], many[k], equal_nan=True), (nx, ny, k)


def test_inlet_in_the_last_column_keeps_single_steps():
    """An inlet at the end of a row reads the next row's first cell: such a
    domain is stepped one step at a time and still matches itself."""
    rng = np.random.default_rng(9)
    nx, ny = 66, 10
    fl, rho0, u0 = _domain(nx, ny, "channel", rng)
    fl = fl.reshape(ny, nx)
    fl[1:-1, -1] = core.INLET
    u0 = u0.reshape(2, ny, nx)
    u0[0][fl == core.INLET] = 0.01
    one = _run(fl.ravel(), nx, ny, rho0, u0.ravel(), [1] * 9)
    many = _run(fl.ravel(), nx, ny, rho0, u0.ravel(), [9])
    for k in ("f", "u", "rho"):
        assert np.array_equal(one[k], many[k]), k


@pytest.mark.parametrize("storage", ["fp32", "fp16s", "bf16s"])
@pytest.mark.parametrize("force", [False, True])
def test_batch_passes_equal_single_steps(storage, force):
    """A batch of uneven instances: passes, graphs of passes (8 steps, so that a
    replay starts from each of the two population arrays) and single steps."""
    rng = np.random.default_rng(10)
    inst = []
    for k, (nx, ny) in enumerate([(65, 9), (130, 41), (57, 4), (300, 33), (64, 64)]):
        fl, rho0, u0 = _domain(nx, ny, "channel" if k % 2 else "scattered", rng)
        fl[-1] = core.WALL
        fl[0] = core.WALL
        inst.append(dict(nx=nx, ny=ny, tau=0.6 + 0.05 * k, flags=fl, rho0=rho0, u0=u0,
                         use_force=int(force and k != 2), fx=1e-5 * k, fy=-1e-5))

    def run(calls, chunk):
        with core.Batch(inst, storage=storage) as b:
            b.configure(block_x=128, grid=0, graph_chunk=chunk)
            for n in calls:
                b.step(n)
            assert b.time == sum(calls)
            return [dict(f=b.populations(i), **b.read(i)) for i in range(len(inst))]

    one = run([1] * 48, 0)
    for calls, chunk in (([48], 0), ([7, 20, 21], 0), ([26, 1, 21], 4), ([3, 45], 10)):
        for i, (a, g) in enumerate(zip(one, run(calls, chunk))):
            for k in a:
                assert np.array_equal(a[k], g[k], equal_nan=True), (calls, chunk, i, k)


def test_batch_with_an_unfit_instance():
    """One instance under four rows: the whole batch keeps single steps."""
    rng = np.random.default_rng(11)
    inst = []
    for nx, ny in [(65, 9), (70, 3)]:
        fl, rho0, u0 = _domain(nx, ny, "channel", rng)
        inst.append(dict(nx=nx, ny=ny, tau=0.7, flags=fl, rho0=rho0, u0=u0))
    got = []
    for calls in ([1] * 9, [9]):
        with core.Batch(inst) as b:
            for n in calls:
                b.step(n)
            got.append([b.populations(i) for i in range(2)])
    for a, g in zip(*got):
        assert np.array_equal(a, g)
