"""GPU: the batches' multi-step strips of both widths and their four-level march on
each of its tiles, bitwise against the oracle."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

mx = pytest.importorskip("mmsp_amd")

P, N = O.PERIODIC, O.NEUMANN
PAR = {"ac": [1.0, 1.0, 1.3, 0.9, 0.01], "ch": [1.0, 1.0, 0.8, 1.0, 0.01], "ch_dw": [0.9, 1.0, 0.005]}


def expected(model, a, steps, prec, bc=None):
    if model == "ac":
        return O.ac(a, PAR[model], steps, form=prec, bc=bc)
    return O.ch(a, PAR[model], steps, mu=O.MU_POLY if model == "ch" else O.MU_DW, form=prec, bc=bc)


def members(model, shapes, prec, bcs=None):
    b = mx.Batch(shapes, model, precision=prec, bcs=bcs)
    b.set_params(np.array([PAR[model]] * len(shapes)))
    inits = [O.uniform(int(np.prod(s)), 4100 + k, 0.3, 0.7).reshape(s).astype(b.dtype) for k, s in enumerate(shapes)]
    return b, inits


def check(b, inits, model, steps, prec, bcs=None, graph=0):
    for m, a in enumerate(inits):
        b.upload(m, a)
    b.step(steps, graph_steps=graph)
    for m, a in enumerate(inits):
        assert np.array_equal(b.download(m), expected(model, a, steps, prec, bcs[m] if bcs else None)), (steps, m)


def tile(b):
    t = b.get_tile()
    return t["strip_width"], t["rows_per_item"], t["blocks_per_cu"]


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("model,walls", [("ac", False), ("ac", True), ("ch", False), ("ch_dw", False)])
def test_strips_of_eight_and_four_levels(model, walls, prec):
    """Whole passes and a short last one of either width, chunks of 2 to 17 rows."""
    shapes = [(3, 5), (40, 57), (33, 49), (18, 200)]
    bcs = [[(N, N), (P, P)]] * 4 if walls else None
    b, inits = members(model, shapes, prec, bcs)
    with b:
        for width in (48, 56):
            for rows, steps, graph in ((2, 8, 0), (5, 13, 0), (17, 27, 6)):
                b.set_tile(width, rows, 0)
                assert tile(b) == (width, rows, 0)
                check(b, inits, model, steps, prec, bcs, graph)


# number and extents of members for which the cost model takes each tile (its
# columns last)
MARCHES = {"f64": [(2, (20, 20, 20), 16), (2, (30, 52, 52), 32), (4, (40, 60, 90), 32), (2, (32, 128, 128), 64),
                   (8, (30, 52, 52), 52)],
           "f32": [(2, (20, 20, 20), 16), (2, (30, 52, 52), 32), (16, (40, 60, 90), 32), (4, (32, 128, 128), 64),
                   (8, (30, 52, 52), 52)]}


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("k", range(5))
def test_march_tiles(k, prec):
    count, shape, columns = MARCHES[prec][k]
    b, inits = members("ch_dw" if k % 2 else "ch", [shape] * count, prec)
    with b:
        assert tile(b)[0] == columns and tile(b)[2] == 0
        check(b, inits, "ch_dw" if k % 2 else "ch", 5, prec)
