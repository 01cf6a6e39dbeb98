"""GPU: the 2-D four-step field strips (tile body 16) and the default that
chooses them, bitwise against the oracle's single steps."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

mx = pytest.importorskip("mmsp_amd")

P, N = O.PERIODIC, O.NEUMANN

# one node, fewer columns than the halo, a last strip of one column, exact
# strips; fewer rows than the halo, rows that end in every place of the march
SHAPES = [(1, 1), (3, 5), (7, 57), (13, 56), (26, 113), (17, 30)]


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("model", ["gg", "zener"])
@pytest.mark.parametrize("q", [2, 4, 8, 16, 32])
def test_four_step_field_strips(q, model, prec):
    """Whole passes and a last pass of every shorter length, unit and other
    grid weights, chunks of 2 to 8 rows and the default."""
    tiled = not (q == 32 and model == "zener" and prec == "f64")  # one thread per node there
    run = O.gg if model == "gg" else O.zener
    for k, shape in enumerate(SHAPES):
        dx = None if k % 2 else [0.9, 1.1]
        a = O.uniform(int(np.prod(shape)) * q, 700 + k, 0.0, 1.0).reshape(shape + (q,))
        if prec == "f32":
            a = a.astype(np.float32)
        for steps in (4, 9 + k % 3):
            exp = run(a, 0.01, steps, form=prec, dx=dx)
            for chunk in (0, 2, 3 + k) if tiled else (0,):  # 0: the default
                with mx.Grid(shape, fields=q, vector=True, precision=prec, dx=dx) as g:
                    if chunk:
                        g.set_variant(2)
                        g.set_tile(1, 56, chunk)
                        g.set_tile_options(body=16)
                    g.upload(a)
                    g.step(model, [0.01], steps)
                    assert np.array_equal(g.download(), exp), (shape, steps, chunk)
                    assert (g.get_tile()["opt"] == 16) == tiled


def test_four_step_field_strips_refuse_other_boundaries():
    with mx.Grid((20, 70), fields=8, vector=True, bc=[(N, N), (P, P)]) as g:
        g.upload(np.zeros((20, 70, 8)))
        g.step("gg", [0.01], 5)
        assert g.get_tile()["opt"] != 16
        g.set_variant(2)
        g.set_tile(1, 56, 8)
        g.set_tile_options(body=16)
        with pytest.raises(mx.MmspxError):
            g.step("gg", [0.01], 4)
