"""flb_batch_autotune chooses between settings that differ: the single steps of
every tile order, block and grid, the persistent kernel, and the passes.  It used to
time the passes under 48 settings that change nothing of them."""
import numpy as np
import pytest

from flowlb_amd import core
from test_gpu_pass_choice import _domain

pytestmark = pytest.mark.gpu


def instances():
    out = []
    for k in range(12):
        nx, ny = 400 + 60 * k, 150 + 20 * k
        fl, u0 = _domain(nx, ny, True)
        out.append(dict(nx=nx, ny=ny, tau=0.6, flags=fl, u0=u0))
    return out


@pytest.mark.parametrize("storage", ["fp16s", "bf16s"])
def test_not_slower_than_a_setting_by_hand(storage):
    """Single steps in bands are the faster way here (passes took 1.4 times as long)."""
    with core.Batch(instances(), storage=storage) as a, core.Batch(instances(), storage=storage) as b:
        a.autotune(steps=24)
        b.set_order("bands")
        b.configure(block_x=256, grid=0, graph_chunk=0)
        took = []
        for run in (lambda: a.step_timed(24), lambda: sum(b.step_timed(1) for _ in range(24))):
            run()
            took.append(min(run() for _ in range(8)))
    print(took)
    assert took[0] < 1.12 * took[1]


@pytest.mark.parametrize("steps", [1, 2, 9])
@pytest.mark.parametrize("unfit", [False, True])
def test_state_and_settings(steps, unfit):
    """Every way leaves the state of as many steps; settings are those of the sweep."""
    inst = instances()[:4]
    if unfit:  # three rows: no passes
        fl, u0 = _domain(70, 3, False)
        inst.append(dict(nx=70, ny=3, tau=0.7, flags=fl, u0=u0))
    with core.Batch(inst) as a, core.Batch(inst) as b:
        bx, grid, ms = a.autotune(steps=steps)
        info = a.info()
        # Three orders with as many settings each, every one over 2 + steps steps, and
        # the passes once.
        assert a.time % (2 + steps) == 0
        assert a.time // (2 + steps) % 3 == int(steps > 1 and not unfit)
        assert bx in (64, 128, 256, 512) and ms > 0 and info["block_x"] == bx and info["grid"] == grid
        a.step(30)
        for _ in range(a.time):
            b.step(1)
        for i in range(len(inst)):
            np.testing.assert_array_equal(a.populations(i), b.populations(i))
