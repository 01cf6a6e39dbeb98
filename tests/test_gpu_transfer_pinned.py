"""GPU: uploads from and downloads to memory the caller has pinned: the sizes
where the path of pageable memory changes, and that a large one is copied
directly (half the time of a pageable one)."""
import ctypes as C
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

mx = pytest.importorskip("mmsp_amd")

MIB = 1 << 20


@pytest.fixture
def pinned():
    """Makes pinned arrays, from the HIP runtime that libmmsp_amd.so has loaded."""
    hip, held = C.CDLL("libamdhip64.so.7"), []

    def make(n):
        p = C.c_void_p()
        assert hip.hipHostMalloc(C.byref(p), C.c_size_t(8 * n), 0) == 0
        held.append(p)
        return np.ctypeslib.as_array(C.cast(p, C.POINTER(C.c_double)), (n,))

    yield make
    for p in held:
        assert hip.hipHostFree(p) == 0


def copies(g, array):
    def call(f):
        t = time.perf_counter()
        mx.check(f(g._h, C.c_void_p(array.ctypes.data), mx.NODE_MAJOR))
        return time.perf_counter() - t

    return (lambda: call(mx.lib.mmspx_upload)), (lambda: call(mx.lib.mmspx_download))


@pytest.mark.parametrize("nbytes", [8, 128 * 1024, MIB * 3 // 2 - 8, 2 * MIB + 8, 17 * MIB + 4096])
def test_roundtrip(nbytes, pinned):
    n = nbytes // 8
    mine = pinned(n + 1)[1:]  # not the allocation's first element
    a = np.random.default_rng(nbytes).random(n)
    with mx.Grid((1, n)) as g:
        up, down = copies(g, mine)
        mine[:] = a
        up()
        assert np.array_equal(g.download().ravel(), a)
        mine[:] = 0.0
        down()
        assert np.array_equal(mine, a)


def test_a_large_pinned_copy_is_direct(pinned):
    n = 64 * MIB // 8
    with mx.Grid((1, n)) as g:
        down = copies(g, pinned(n))[1]
        pageable = copies(g, np.zeros(n))[1]
        times = [sorted(f() for _ in range(9))[4] for f in (pageable, down, pageable, down)]
    assert min(times[1], times[3]) < 0.75 * min(times[0], times[2]), times
