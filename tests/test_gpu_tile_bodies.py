"""GPU: tiles and bodies set one after the other. A body keeps no tile that only
bodies 13 to 17 run; a body or tile no model of the grid runs is refused where
it is set; a field march's kernel read back can be set again."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

mx = pytest.importorskip("mmsp_amd")

N = O.NEUMANN
AC, DW, GGA = [1.0, 1.0, 1.0, 1.0, 0.01], [1.0, 1.0, 0.005], [0.01, 8.0, 1.0, 1.0]


def start(shape, q, seed=4000):
    return O.uniform(int(np.prod(shape)) * q, seed, 0.0, 1.0).reshape(shape + ((q,) if q > 1 else ()))


def run(a, q, model, params, bodies, bc=None, tile=None):
    shape = a.shape[:-1] if q > 1 else a.shape
    with mx.Grid(shape, fields=q, vector=q > 1, bc=bc) as g:
        g.set_variant(2)
        if tile:
            g.set_tile(*tile)
        for body in bodies:
            g.set_tile_options(body=body)
        g.upload(a)
        g.step(model, params, 5)
        return g.get_kernel(), g.download()


@pytest.mark.parametrize("first", [13, 14])
@pytest.mark.parametrize("body", [0, 1, 2])
def test_leaving_the_multi_step_strips(first, body):
    a, bc = start((40, 70), 1), [(N, N), (N, N)]
    ran, got = run(a, 1, "ac", AC, (first, body), bc)
    assert (ran["opt"], ran["tz"]) == (body, 64) and np.array_equal(got, O.ac(a, AC, 5, bc=bc))
    ran, got = run(a, 1, "ch_dw", DW, (first, body))
    assert (ran["opt"], ran["tz"]) == (body, 64) and np.array_equal(got, O.ch(a, DW, 5, mu=O.MU_DW))


def test_leaving_the_field_strips():
    a = start((40, 70), 4)
    ran, got = run(a, 4, "gg_aniso", GGA, (16, 2))
    assert (ran["opt"], ran["tz"]) == (2, 64) and np.array_equal(got, O.gg_aniso(a, GGA, 5))
    ran, got = run(a, 4, "zener", [0.01], (16, 2))
    assert ran["opt"] == 2 and np.array_equal(got, O.zener(a, 0.01, 5))


@pytest.mark.parametrize("tile", [(16, 16, 4), (26, 52, 4), (26, 56, 4)])
@pytest.mark.parametrize("body", [0, 1, 2, 3])
def test_leaving_the_four_level_march(tile, body):
    a = start((9, 20, 40), 1)
    ran, got = run(a, 1, "ch_dw", DW, (15, body), tile=tile)
    assert (ran["ty"], ran["tz"], ran["opt"]) == (32, 64, body) and np.array_equal(got, O.ch(a, DW, 5, mu=O.MU_DW))


@pytest.mark.parametrize("body", [8, 12])  # (grain growth runs no others)
def test_leaving_the_field_march(body):
    a = start((9, 20, 40), 4)
    ran, got = run(a, 4, "gg", [0.01], (17, body))
    assert ran["opt"] == body and np.array_equal(got, O.gg(a, 0.01, 5))


def test_what_no_model_of_the_grid_runs_is_refused():
    for shape, q, tiles, bodies in [((20, 70), 4, [(1, 48, 4)], (13, 14)), ((20, 70), 3, [(1, 48, 4), (1, 56, 4)], (13, 14, 16)),
                                    ((20, 70), 1, [], (16,)), ((8, 20, 40), 1, [(12, 58, 4), (28, 58, 4)], (17,)),
                                    ((8, 20, 40), 4, [(26, 52, 4), (16, 16, 4), (42, 56, 4)], (15,)),
                                    ((8, 20, 40), 3, [(12, 58, 4)], (15, 17))]:
        with mx.Grid(shape, fields=q, vector=q > 1) as g:
            before = g.get_tile()
            for t in tiles:
                with pytest.raises(mx.MmspxError):
                    g.set_tile(*t)
            for b in bodies:
                with pytest.raises(mx.MmspxError):
                    g.set_tile_options(body=b)
            assert g.get_tile() == before
    with mx.Grid((8, 20, 40), fields=4, vector=True, precision="f32ref") as g:
        with pytest.raises(mx.MmspxError):
            g.set_tile_options(body=17)


@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_a_field_march_read_back_is_set_again(prec):
    a = start((40, 50, 97), 8).astype(np.float64 if prec == "f64" else np.float32)
    kernels, states = [], []
    for k in range(2):
        with mx.Grid((40, 50, 97), fields=8, vector=True, precision=prec) as g:
            if k:
                g.set_tile(kernels[0]["ty"], kernels[0]["tz"], kernels[0]["chunk"])
                g.set_tile_options(body=kernels[0]["opt"])
            g.upload(a)
            g.step("gg", [0.01], 6)
            kernels.append(g.get_kernel())
            states.append(g.download())
    assert kernels[0]["opt"] == 17 and kernels[0] == kernels[1] and np.array_equal(*states)
