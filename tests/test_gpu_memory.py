"""Device memory held for speed alone (the second population array of the passes,
the buffers of the last gradient) takes nothing from what a program could allocate
without it: where an allocation of the library finds no room, idle handles and
batches give it back and go on by single steps with the same results.  The device is
filled with plain allocations (never touched) up to a few GB."""
import ctypes as C
import threading

import numpy as np
import pytest

from flowlb_amd import core

pytestmark = pytest.mark.gpu
GB = 1 << 30


def free_bytes():
    a, b = C.c_size_t(), C.c_size_t()
    assert core.hip().hipMemGetInfo(C.byref(a), C.byref(b)) == 0
    return a.value


@pytest.fixture(scope="module")
def filled():
    """All but 3 GB of the device taken."""
    hip, held = core.hip(), []
    for piece in (16 * GB, GB, 64 << 20):
        while free_bytes() > 3 * GB + piece:
            p = C.c_void_p()
            if hip.hipMalloc(C.byref(p), piece) != 0:
                break
            held.append(p)
    yield
    for p in held:
        hip.hipFree(p)


def box(nx, ny, fits=True):
    fl = np.full((ny, nx), core.FLUID, np.uint8)
    fl[0] = fl[-1] = core.WALL
    u0 = np.zeros((2, ny, nx), np.float32)
    if not fits:  # an inlet in the last column: such a domain takes no passes
        fl[ny // 2, -1] = core.INLET
    u0[0][1:-1] = 0.01
    return fl.ravel(), u0.ravel()


def as_many_as_fit(make):
    out = []
    try:
        while len(out) < 64:
            out.append(make())
    except core.FlbError as e:
        assert e.status == 3
    return out


NX, NY = 4096, 1024  # 357 MB, and 151 MB for the second array


def gradient(s, steps=200):
    return s.adjoint(steps, 300, steps // 2, steps - 1, ckpt=steps, trace_budget_bytes=1 << 50)


def test_what_handles_keep_together_is_bounded():
    fl, u0 = box(1024, 256)
    core.lib()
    start = free_bytes()
    hs = [core.Solver(fl, 1024, 256, core.default_options(tau=0.6), u0=u0) for _ in range(8)]
    made = free_bytes()
    total = C.c_size_t()
    core.hip().hipMemGetInfo(C.byref(C.c_size_t()), C.byref(total))
    for s in hs:
        gradient(s, 800)  # 2.5 GB of trace each
    kept = made - free_bytes()
    for s in hs:
        s.close()
    assert GB < kept <= total.value // 32 + (256 << 20)
    assert free_bytes() > start - (256 << 20)


def test_a_small_trace_budget_is_kept_to():
    fl, u0 = box(1024, 256)
    with core.Solver(fl, 1024, 256, core.default_options(tau=0.6), u0=u0) as s:
        made = free_bytes()
        a = gradient(s, 300)  # 0.9 GB of trace
        assert made - free_bytes() > 700 << 20
        b = s.adjoint(300, 300, 150, 299, ckpt=20, trace_budget_bytes=100 << 20)
        assert made - free_bytes() < 700 << 20
        assert a[0] == b[0]


def test_handles_fill_the_device_as_without_passes(filled):
    def make(fits):
        fl, u0 = box(NX, NY, fits)
        s = core.Solver(fl, NX, NY, core.default_options(tau=0.6), u0=u0)
        s.step(4)
        s.sync()
        return s

    plain = as_many_as_fit(lambda: make(False))
    n = len(plain)
    for s in plain:
        s.close()
    assert 4 <= n < 64
    full = as_many_as_fit(lambda: make(True))
    try:
        assert len(full) >= n
        # The first ones lost their second array, the state is the same.
        fl, u0 = box(NX, NY)
        for s in full:
            s.step(5)
    finally:
        for s in full[1:]:
            s.close()
    got = full[0].populations()
    full[0].close()
    with core.Solver(fl, NX, NY, core.default_options(tau=0.6), u0=u0) as s:
        s.step(9)
        np.testing.assert_array_equal(got, s.populations())


@pytest.mark.parametrize("steps", [6, 7])  # the state ends in either array
def test_batch_gives_its_second_array_back(steps, filled):
    fl, u0 = box(NX, NY)
    inst = [dict(nx=NX, ny=NY, tau=0.6, flags=fl, u0=u0), dict(nx=70, ny=30, tau=0.7, flags=box(70, 30)[0], u0=None)]
    with core.Batch(inst) as b:
        b.step(steps)
        b.sync()
        before = free_bytes()
        fill = as_many_as_fit(lambda: core.Solver(*box(NX, NY, False)[:1], NX, NY, core.default_options(tau=0.6)))
        size = (before - free_bytes()) // max(1, len(fill)) if fill else 0
        b.step(9)
        got = [b.populations(i) for i in range(1, 2)]
        for s in fill:
            s.close()
        got.insert(0, b.populations(0))
        # The batch's 151 MB are no longer held.
        assert free_bytes() > before + 100_000_000, size
    with core.Batch(inst) as b:
        b.step(steps + 9)
        for i in range(2):
            np.testing.assert_array_equal(got[i], b.populations(i))


def test_gradients_of_many_idle_handles(filled):
    """A gradient here keeps 0.7 GB; eight handles need less than they would keep."""
    fl, u0 = box(1024, 256)
    fl = fl.reshape(256, 1024)
    fl[1:-1, 0], fl[1:-1, -1] = core.INLET, core.OUTLET
    alpha = np.zeros(1024 * 256, np.float32)
    alpha[40000:60000] = 0.3
    hs = []
    try:
        for _ in range(8):
            s = core.Solver(fl.ravel(), 1024, 256, core.default_options(tau=0.6), u0=u0)
            s.set_brinkman(alpha)
            hs.append(s)
        out = [gradient(s) for s in hs]
        assert all(o[0] == out[0][0] and np.array_equal(o[1], out[0][1]) for o in out)
        assert hs[0].objective(200, 300, 100, 199) == out[0][0]
    finally:
        for s in hs:
            s.close()


def test_threads_that_step_while_others_run_out_of_room(filled):
    """Handles stepping in threads of their own while the main thread allocates
    until nothing is left: each either keeps its second array or gives it back
    between calls."""
    fl, u0 = box(NX, NY)
    errors, stop = [], threading.Event()

    def work(s, done):
        try:
            while not stop.is_set():
                s.step(4)
                s.step(3)
                s.sync()  # streams share queues: a backlog here would hold up every copy there
                done[0] += 7
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    hs = [core.Solver(fl, NX, NY, core.default_options(tau=0.6), u0=u0) for _ in range(3)]
    done = [[0] for _ in hs]
    ts = [threading.Thread(target=work, args=x) for x in zip(hs, done)]
    for t in ts:
        t.start()
    try:
        fill = as_many_as_fit(lambda: core.Solver(box(NX, NY, False)[0], NX, NY, core.default_options(tau=0.6)))
    finally:
        stop.set()
        for t in ts:
            t.join()
    for s in fill:
        s.close()
    assert not errors
    got = [(s.populations(), s.time) for s in hs]
    for s in hs:
        s.close()
    with core.Solver(fl, NX, NY, core.default_options(tau=0.6), u0=u0) as s:
        for (f, t), n in sorted(zip(got, done), key=lambda x: x[0][1]):
            assert t == n[0]
            s.step(t - s.time)
            np.testing.assert_array_equal(f, s.populations())
