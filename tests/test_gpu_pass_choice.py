"""Runs of several steps never take much longer than the same steps one by one:
domains and batches where passes are the slower way (every strip with inlet or
outlet cells, costly models in 16-bit storage) go in single steps.  flb_step(1) also
stores the fields each time, so the bound is lenient; passes took 1.3 to 2 times as
long here.  Results are those of single steps either way (bit for bit)."""
import numpy as np
import pytest

from flowlb_amd import core

pytestmark = pytest.mark.gpu


def _domain(nx, ny, top):
    fl = np.full((ny, nx), core.FLUID, np.uint8)
    fl[0] = core.WALL
    fl[-1] = core.OUTLET if top else core.WALL
    fl[1:-1, 0] = core.INLET
    fl[1:-1, -1] = core.OUTLET
    fl[-1, 0] = fl[-1, -1] = core.WALL
    u0 = np.zeros((2, ny, nx), np.float32)
    u0[0][fl == core.INLET] = 0.02
    return fl.ravel(), u0.ravel()


def _time(step, many):
    """ms of `many` steps in one call and in calls of one step."""
    out = []
    for f in (lambda: step(many), lambda: sum(step(1) for _ in range(many))):
        f()
        out.append(min(f() for _ in range(6)))
    return out


@pytest.mark.parametrize("nx,ny,top,storage,opt", [
    (4096, 1024, True, "bf16s", dict(use_force=1, fx=1e-6)),
    (2048, 512, True, "fp64", dict(use_force=1, fx=1e-6, smagorinsky=1)),
    (3000, 700, False, "fp16s", dict(collision=2, smagorinsky=1, use_force=1, fx=1e-6))])
def test_runs_are_not_slower_than_single_steps(nx, ny, top, storage, opt):
    fl, u0 = _domain(nx, ny, top)
    with core.Solver(fl, nx, ny, core.default_options(tau=0.6, storage=storage, **opt), u0=u0) as s:
        run, single = _time(s.step_timed, 24)
    print(run, single)
    assert run < 1.12 * single


@pytest.mark.parametrize("storage", ["fp16s", "bf16s"])
def test_batch_runs_are_not_slower_than_single_steps(storage):
    inst = []
    for k in range(12):
        nx, ny = 400 + 60 * k, 150 + 20 * k
        fl, u0 = _domain(nx, ny, True)
        inst.append(dict(nx=nx, ny=ny, tau=0.6, flags=fl, u0=u0))
    with core.Batch(inst, storage=storage) as b:
        b.set_order("bands")
        b.configure(block_x=256, grid=0, graph_chunk=0)
        run, single = _time(b.step_timed, 24)
    print(run, single)
    assert run < 1.12 * single
