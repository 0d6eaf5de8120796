"""Host copies from and to memory the caller pinned, which go straight to the
device, and pageable copies around the sizes where the runtime's own copy takes
over from the handle's buffers (16 KiB and 1 MiB to the host, 16 MiB to the
device): the same bytes, and no second copy for pinned memory."""
import ctypes as C
import time

import numpy as np
import pytest

from flowlb_amd import core

pytestmark = pytest.mark.gpu


class Pinned:
    def __init__(self, count, dtype=np.float32):
        hip = core.hip()
        hip.hipHostMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t, C.c_uint]
        self.p = C.c_void_p()
        nbytes = count * np.dtype(dtype).itemsize
        assert hip.hipHostMalloc(C.byref(self.p), nbytes, 0) == 0
        self.a = np.ctypeslib.as_array((C.c_uint8 * nbytes).from_address(self.p.value)).view(dtype)

    def __enter__(self):
        return self.a

    def __exit__(self, *a):
        core.hip().hipHostFree.argtypes = [C.c_void_p]
        core.hip().hipHostFree(self.p)


def solver(nx, ny, **opt):
    rng = np.random.default_rng(nx * ny)
    fl = np.full(nx * ny, core.FLUID, np.uint8)
    fl[:nx] = core.WALL
    return core.Solver(fl, nx, ny, core.default_options(**opt),
                       rho0=(1 + 0.1 * rng.random(nx * ny)).astype(np.float32),
                       u0=(0.1 * rng.random(2 * nx * ny)).astype(np.float32))


# Populations of 9 * 4 * nx * ny bytes: just below and above 16 KiB, 1 MiB and 16 MiB;
# fields in padded rows (strided copies) and in rows of 64 and 128 cells (contiguous).
@pytest.mark.parametrize("nx,ny", [(5, 91), (4, 114), (64, 7), (64, 8), (7, 4161), (53, 550),
                                   (128, 228), (682, 683), (684, 682), (1999, 300)])
def test_same_bytes(nx, ny):
    N = nx * ny
    rng = np.random.default_rng(5)
    new = [rng.random(N).astype(np.float32) for _ in range(3)]
    out = []
    for pinned in (False, True):
        with solver(nx, ny, problem=core.FREE_SURFACE) as s, Pinned(3 * N) as a, \
                Pinned(9 * N) as f, Pinned(3 * N) as b:
            if not pinned:
                a, f, b = np.empty(3 * N, np.float32), np.empty(9 * N, np.float32), np.empty(3 * N, np.float32)
            for k in range(3):
                a[k * N:(k + 1) * N] = new[k]
            P = [core.fptr(a[k * N:(k + 1) * N]) for k in range(3)]
            core.check(core.lib().flb_set_fs_fields(s.h, *P), s.h)
            core.check(core.lib().flb_read_populations(s.h, core.fptr(f)), s.h)
            core.check(core.lib().flb_read(s.h, core.fptr(b[:2 * N]), core.fptr(b[2 * N:]), None, None), s.h)
            a[:] = -1
            core.check(core.lib().flb_read_fs(s.h, P[0], P[2]), s.h)
            out.append([x.copy() for x in (f, b, a)])
            assert np.array_equal(a[:N], new[0]) and np.array_equal(a[2 * N:], new[2])
    for x, y in zip(*out):
        np.testing.assert_array_equal(x, y)
    rho0 = (1 + 0.1 * np.random.default_rng(N).random(N)).astype(np.float32)
    np.testing.assert_array_equal(out[0][1][2 * N:], rho0)


@pytest.mark.parametrize("nx,ny", [(1024, 1024), (1000, 1024)])
def test_pinned_memory_is_copied_once(nx, ny):
    """Through the buffers a readback into pinned memory took as long as one into
    pageable memory (650 us); straight it takes 240 us."""
    N = nx * ny
    with solver(nx, ny) as s, Pinned(3 * N) as pinned:
        took = {}
        for name, b in (("pageable", np.zeros(3 * N, np.float32)), ("pinned", pinned)):
            b[:] = 0
            best = 1e9
            for _ in range(25):
                t = time.perf_counter()
                core.check(core.lib().flb_read(s.h, core.fptr(b[:2 * N]), core.fptr(b[2 * N:]), None, None), s.h)
                best = min(best, time.perf_counter() - t)
            took[name] = best
        print(took)
        assert took["pinned"] < 0.75 * took["pageable"]
