"""GPU: the four-level march with a wave's lanes along axis 2 on 12 waves of four
rows (42 x 56 tiles, FP64: the default of large grids), bitwise against the
oracle's single steps."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

mx = pytest.importorskip("mmsp_amd")

AC, CH, DW = [1.0, 1.0, 1.3, 0.9, 0.01], [1.0, 1.0, 0.8, 1.0, 0.01], [1.0, 1.0, 0.005]
UNIT = {"ac": [1.0, 1.0, 1.0, 1.0, 0.01], "ch": [1.0, 1.0, 1.0, 1.0, 0.01], "ch_dw": DW}
# one node, grids thinner than the halo, one tile exactly, one node more than a
# tile in each in-plane axis, planes that leave a short last chunk
SHAPES = [(1, 1, 1), (2, 3, 5), (9, 42, 56), (7, 43, 57), (13, 47, 58)]


@pytest.mark.parametrize("model", ["ac", "ch", "ch_dw"])
def test_tall_tiles(model):
    """Chunks of 2, 3 and 7 planes, unit and other weights, whole passes and last
    passes of every shorter length."""
    for k, shape in enumerate(SHAPES):
        dx = [0.9, 1.1, 1.2] if k == 3 else None
        params = UNIT[model] if k % 2 else {"ac": AC, "ch": CH, "ch_dw": DW}[model]
        a = O.uniform(int(np.prod(shape)), 4200 + k, 0.3, 0.7).reshape(shape)
        for steps in (4, 5 + k % 3):
            if model == "ac":
                exp = O.ac(a, params, steps, dx=dx)
            else:
                exp = O.ch(a, params, steps, mu=O.MU_POLY if model == "ch" else O.MU_DW, dx=dx)
            with mx.Grid(shape, dx=dx) as g:
                g.set_variant(2)
                g.set_tile(42, 56, (2, 3, 7)[k % 3])
                g.upload(a)
                g.step(model, params, steps)
                t = g.get_kernel()
                assert (t["ty"], t["tz"], t["opt"]) == (42, 56, 15)
                assert np.array_equal(g.download(), exp), (shape, steps)
