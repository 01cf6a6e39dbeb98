"""GPU: transfers before and after the library makes its pinned area (the ninth
that asks for one; at once from 8 MiB on), sizes mixed so that it grows, and
made again after the last state went."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

mx = pytest.importorskip("mmsp_amd")

MIB = 1 << 20


def transfers(nbytes, count, seed):
    n = nbytes // 8
    with mx.Grid((1, n)) as g:
        for k in range(count):
            a = np.random.default_rng(seed + k).random((1, n))
            g.upload(a)
            assert np.array_equal(g.download(), a), k


@pytest.mark.parametrize("nbytes", [8, 128 * 1024, MIB // 2 + 8, MIB * 3 // 2 - 8, MIB * 3 // 2 + 8, 2 * MIB, 2 * MIB + 8,
                                    5 * MIB + 8, 8 * MIB])
def test_one_size(nbytes):
    for life in range(2):
        transfers(nbytes, 12, 100 * life)


def test_sizes_mixed():
    with mx.Grid((1, 2)):  # the area outlives the states below
        for nbytes in (1024, MIB, 3 * MIB, 64, 9 * MIB, 512 * 1024, 3 * MIB):
            transfers(nbytes, 6, nbytes)
