"""GPU: the 3-D field march (tile body 17) and the default that chooses it,
bitwise against the oracle's single steps."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

mx = pytest.importorskip("mmsp_amd")

TILES = {("f32", 8): [(12, 58), (22, 60)], ("f32", 4): [(18, 56), (28, 58)], ("f32", 2): [(26, 56)],
         ("f64", 8): [(8, 60), (10, 60)], ("f64", 4): [(22, 60), (12, 58)], ("f64", 2): [(18, 56), (28, 58)]}
# one node, grids thinner than the halo, one node more than a tile in each
# in-plane axis, planes that leave a short last chunk
SHAPES = [(1, 1, 1), (2, 3, 5), (7, 23, 61), (11, 13, 59)]


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("model", ["gg", "zener"])
@pytest.mark.parametrize("q", [2, 4, 8])
def test_field_march(q, model, prec):
    """Every tile and the default, chunks of 2, 3 and 5 planes, unit and other
    grid weights, whole passes and last passes of every shorter length."""
    run = O.gg if model == "gg" else O.zener
    for k, shape in enumerate(SHAPES):
        dx = [0.9, 1.1, 1.2] if k % 2 else None
        a = O.uniform(int(np.prod(shape)) * q, 2700 + k, 0.0, 1.0).reshape(shape + (q,))
        if prec == "f32":
            a = a.astype(np.float32)
        for steps in (4, 5, 7):
            exp = run(a, 0.01, steps, form=prec, dx=dx)
            for n, tile in enumerate([None] + TILES[prec, q]):
                with mx.Grid(shape, fields=q, vector=True, precision=prec, dx=dx) as g:
                    if tile:
                        g.set_variant(2)
                        g.set_tile(16, 32, (2, 3, 5)[(n + k) % 3])
                        g.set_tile_options(body=17)
                        g.set_tile(tile[0], tile[1], (2, 3, 5)[(n + k) % 3])
                        t = g.get_tile()
                        assert (t["ty"], t["tz"], t["opt"]) == (tile[0], tile[1], 17)
                    g.upload(a)
                    g.step(model, [0.01], steps)
                    assert np.array_equal(g.download(), exp), (shape, steps, tile)


def test_field_march_is_the_default_where_tiles_would_be_padded():
    shape = (20, 41, 97)
    a = O.uniform(int(np.prod(shape)) * 8, 2790, 0.0, 1.0).reshape(shape + (8,))
    with mx.Grid(shape, fields=8, vector=True) as g:
        g.upload(a)
        g.step("gg", [0.01], 5)
        t = g.get_tile()
        assert (t["ty"], t["tz"]) in TILES["f64", 8]
        assert np.array_equal(g.download(), O.gg(a, 0.01, 5))


def test_field_march_refuses_other_boundaries():
    with mx.Grid((6, 20, 40), fields=4, vector=True, bc=[(O.NEUMANN, O.NEUMANN), (O.PERIODIC, O.PERIODIC),
                                                         (O.PERIODIC, O.PERIODIC)]) as g:
        g.set_variant(2)
        g.set_tile(16, 32, 4)
        g.set_tile_options(body=17)
        g.upload(np.zeros((6, 20, 40, 4)))
        with pytest.raises(mx.MmspxError):
            g.step("gg", [0.01], 4)
