"""GPU: the four-level march with a wave's lanes along axis 2 (tile body 15 on
26 x 56 and, in FP32, 30 x 56 tiles), bitwise against the oracle's single steps."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

mx = pytest.importorskip("mmsp_amd")

AC, CH, DW = [1.0, 1.0, 1.3, 0.9, 0.01], [1.0, 1.0, 0.8, 1.0, 0.01], [1.0, 1.0, 0.005]
UNIT = {"ac": [1.0, 1.0, 1.0, 1.0, 0.01], "ch": [1.0, 1.0, 1.0, 1.0, 0.01], "ch_dw": [1.0, 1.0, 0.005]}
# one node, grids thinner than the halo, one tile exactly, one node more than a
# tile in each in-plane axis, planes that leave a short last chunk
SHAPES = [(1, 1, 1), (2, 3, 5), (9, 26, 56), (7, 27, 57), (13, 31, 58)]


def expected(model, a, params, steps, prec, dx):
    if model == "ac":
        return O.ac(a, params, steps, form=prec, dx=dx)
    return O.ch(a, params, steps, mu=O.MU_POLY if model == "ch" else O.MU_DW, form=prec, dx=dx)


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("model", ["ac", "ch", "ch_dw"])
def test_lanes_along_axis_2(model, prec):
    """Both tiles, chunks of 2, 3 and 7 planes, unit and other weights, whole
    passes and last passes of every shorter length."""
    for k, shape in enumerate(SHAPES):
        dx = [0.9, 1.1, 1.2] if k == 3 else None
        params = UNIT[model] if k % 2 else {"ac": AC, "ch": CH, "ch_dw": DW}[model]
        a = O.uniform(int(np.prod(shape)), 2300 + k, 0.3, 0.7).reshape(shape)
        if prec == "f32":
            a = a.astype(np.float32)
        for steps in (4, 5 + k % 3):
            exp = expected(model, a, params, steps, prec, dx)
            for n, tile in enumerate([(26, 56)] + ([(30, 56)] if prec == "f32" else [])):
                with mx.Grid(shape, precision=prec, dx=dx) as g:
                    g.set_variant(2)
                    g.set_tile(tile[0], tile[1], (2, 3, 7)[(n + k) % 3])
                    t = g.get_tile()
                    assert (t["ty"], t["tz"], t["opt"]) == (tile[0], tile[1], 15)
                    g.upload(a)
                    g.step(model, params, steps)
                    assert np.array_equal(g.download(), exp), (shape, steps, tile)
