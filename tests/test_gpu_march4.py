"""GPU: the 3-D four-level march (tile body 15) and the default that chooses
it, bitwise against the oracle's single steps."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

mx = pytest.importorskip("mmsp_amd")

AC, CH, DW = [1.0, 1.0, 1.3, 0.9, 0.01], [1.0, 1.0, 0.8, 1.0, 0.01], [1.0, 1.0, 0.005]
TILES = {"f64": [(26, 52), (16, 64), (32, 32), (16, 32), (16, 16)],
         "f32": [(32, 64), (26, 52), (32, 32), (16, 32), (16, 16)]}
# one node, grids thinner than the halo, one tile exactly, one node more than
# a tile in each in-plane axis, planes that leave a short last chunk
SHAPES = [(1, 1, 1), (2, 3, 5), (9, 16, 32), (7, 17, 33), (13, 27, 65)]


def expected(model, a, steps, prec, dx):
    if model == "ac":
        return O.ac(a, AC, steps, form=prec, dx=dx)
    if model == "ch":
        return O.ch(a, CH, steps, mu=O.MU_POLY, form=prec, dx=dx)
    return O.ch(a, DW, steps, mu=O.MU_DW, form=prec, dx=dx)


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("model", ["ac", "ch", "ch_dw"])
def test_four_level_march(model, prec):
    """Every tile, chunks of 2, 3 and 7 planes, unit and other grid weights,
    whole passes and last passes of every shorter length, the default."""
    params = {"ac": AC, "ch": CH, "ch_dw": DW}[model]
    for k, shape in enumerate(SHAPES):
        dx = [0.9, 1.1, 1.2] if k == 3 else None
        a = O.uniform(int(np.prod(shape)), 1900 + k, 0.3, 0.7).reshape(shape)
        if prec == "f32":
            a = a.astype(np.float32)
        for steps in (4, 5 + k % 3):
            exp = expected(model, a, steps, prec, dx)
            for n, tile in enumerate([None] + TILES[prec]):
                with mx.Grid(shape, precision=prec, dx=dx) as g:
                    if tile:
                        g.set_variant(2)
                        g.set_tile(32, 64, (2, 3, 7)[(n + k) % 3])
                        g.set_tile_options(body=15)
                        g.set_tile(tile[0], tile[1], (2, 3, 7)[(n + k) % 3])
                        g.set_tile_options(body=15)
                        t = g.get_tile()
                        assert (t["ty"], t["tz"], t["opt"]) == (tile[0], tile[1], 15)
                    g.upload(a)
                    g.step(model, params, steps)
                    assert np.array_equal(g.download(), exp), (shape, steps, tile)


def test_four_level_march_refuses_what_it_cannot_run():
    """Non-periodic grids, the reference's float form, a tile of the other form."""
    for kw in (dict(bc=[(O.NEUMANN, O.NEUMANN), (O.PERIODIC, O.PERIODIC), (O.PERIODIC, O.PERIODIC)]),
               dict(precision="f32ref")):
        with mx.Grid((8, 10, 12), **kw) as g:
            g.set_variant(2)
            g.set_tile(16, 16, 4)
            g.upload(np.zeros((8, 10, 12)))
            with pytest.raises(mx.MmspxError):
                g.step("ac", AC, 4)
    with mx.Grid((8, 10, 12), precision="f32") as g:
        g.set_variant(2)
        g.set_tile(16, 64, 4)
        g.set_tile_options(body=15)  # 16 x 64 is an FP64 tile of this body: falls back to 16 x 32
        assert (g.get_tile()["ty"], g.get_tile()["tz"]) == (16, 32)
