"""Uploads and downloads through pinned memory: the sizes where the path
changes, remainders of a piece, two threads at once, and teardown between."""

import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

mx = pytest.importorskip("mmsp_amd")

MIB = 1 << 20
# bytes around: staged upload, staged download, pieces, more threads
SIZES = [8, 128 * 1024, MIB // 2 + 8, MIB * 3 // 2 - 8, MIB * 3 // 2 + 8, 2 * MIB, 2 * MIB + 8, 15 * MIB + 8, 16 * MIB,
         17 * MIB + 4096, 49 * MIB - 8]


def _roundtrip(nbytes, seed):
    n = nbytes // 8
    a = np.random.default_rng(seed).integers(-1000, 1000, (1, n)).astype(np.float64)  # whole numbers: sums are exact
    with mx.Grid((1, n)) as g:
        g.upload(a)
        assert np.array_equal(g.download(), a)
        assert np.ravel(g.mass())[0] == a.sum()


@pytest.mark.parametrize("nbytes", SIZES)
def test_roundtrip(nbytes):
    _roundtrip(nbytes, nbytes)


def test_two_threads():
    errors = []

    def work(seed):
        try:
            for nbytes in (MIB, 5 * MIB + 8, 128 * 1024, 20 * MIB):
                _roundtrip(nbytes, seed)
        except BaseException as e:
            errors.append(e)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
