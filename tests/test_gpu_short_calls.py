"""GPU: calls of fewer steps than a pass, and the steps left over at a call's
end, on the kernel that is fastest for them, bitwise against the oracle (the
one-thread-per-node kernels where the grid is large)."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

mx = pytest.importorskip("mmsp_amd")

P, N, M = O.PERIODIC, O.NEUMANN, O.MIRROR
WALLS = [(N, M), (M, N)]
PARAMS = {"ac": [1.0, 1.0, 1.3, 0.9, 0.01], "ch": [1.0, 1.0, 0.8, 1.0, 0.01], "ch_dw": [1.0, 1.0, 0.005], "gg": [0.01],
          "zener": [0.01]}
# the body a call of 1, 2, 3, ... steps starts with (the multi-step bodies are 13 to 17)
CASES = [
    ("ac", (40, 60), 1, None, {1: (3,), 2: (3,), 3: (3,), 4: (13, 14), 5: (3,), 7: (3,), 9: (13, 14)}),
    ("ac", (40, 60), 1, WALLS, {1: (2,), 2: (13, 14), 5: (13, 14), 9: (13, 14)}),
    ("ch", (40, 60), 1, WALLS, {1: (0,), 2: (13, 14), 3: (13, 14), 5: (13, 14)}),
    ("ch_dw", (40, 60), 1, None, {1: (0,), 2: (13, 14), 3: (13, 14), 5: (13, 14)}),
    ("gg", (40, 60), 4, None, {1: (16,), 2: (16,), 3: (16,), 5: (16,), 6: (16,)}),
    ("gg", (270, 250), 32, None, {1: (10,), 2: (10,), 3: (16,), 5: (16,), 6: (16,)}),
    ("zener", (350, 380), 16, None, {1: (10,), 2: (10,), 3: (16,), 6: (16,)}),
    ("ac", (20, 30, 40), 1, None, {1: (15,), 2: (15,), 5: (15,)}),
    ("ac", (62, 66, 66), 1, None, {1: (8,), 2: (15,), 3: (15,), 5: (15,), 6: (15,)}),
    ("ch", (20, 30, 40), 1, None, {1: (15,), 2: (15,), 3: (15,)}),
]
# 3-D grain growth: the field march by precision; in FP64 its single step too,
# as the plane march would pad these rows
MARCHES = {"f64": {1: (17,), 2: (17,), 3: (17,)}, "f32": {1: (8,), 2: (17,), 3: (17,), 4: (17,), 5: (17,)}}


def start(shape, q, seed, prec):
    a = O.uniform(int(np.prod(shape)) * q, seed, 0.0, 1.0).reshape(shape + ((q,) if q > 1 else ()))
    return a if prec == "f64" else a.astype(np.float32)


def expected(model, a, steps, prec, bc):
    p = PARAMS[model]
    if model == "ac":
        return O.ac(a, p, steps, form=prec, bc=bc)
    if model in ("gg", "zener"):
        return (O.gg if model == "gg" else O.zener)(a, p[0], steps, form=prec, bc=bc)
    return O.ch(a, p, steps, mu=O.MU_POLY if model == "ch" else O.MU_DW, form=prec, bc=bc)


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("model,shape,q,bc,bodies", CASES)
def test_short_calls(model, shape, q, bc, bodies, prec):
    check(model, shape, q, bc, bodies, prec)


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("model", ["gg", "zener"])
def test_short_calls_on_the_field_march(model, prec):
    check(model, (40, 50, 97), 8, None, MARCHES[prec], prec)


def check(model, shape, q, bc, bodies, prec):
    a = start(shape, q, 3600, prec)
    for steps, opts in bodies.items():
        with mx.Grid(shape, fields=q, vector=q > 1, precision=prec, bc=bc) as g:
            g.upload(a)
            g.step(model, PARAMS[model], steps)
            assert g.get_kernel()["opt"] in opts, (steps, g.get_kernel())
            assert np.array_equal(g.download(), expected(model, a, steps, prec, bc)), steps


def test_one_step_of_small_single_precision_marches():
    a = start((62, 66, 66), 1, 3650, "f32")
    with mx.Grid(a.shape, precision="f32") as g:
        g.upload(a)
        g.step("ac", PARAMS["ac"], 5)  # a pass of four and one step
        g.step("ac", PARAMS["ac"], 1)
        k = g.get_kernel()
        assert (k["ty"], k["tz"], k["chunk"], k["opt"]) == (16, 32, 4, 8)
        assert np.array_equal(g.download(), expected("ac", a, 6, "f32", None))


# large grids: two steps of 3-D Allen-Cahn, one of 3-D Cahn-Hilliard, two of
# Allen-Cahn between walls; 2-D Allen-Cahn too large for the temporal blocks
@pytest.mark.parametrize("model,shape,bc,prec,steps,bodies", [
    ("ac", (64, 128, 128), None, "f64", 2, (12,)), ("ac", (64, 128, 128), None, "f32", 6, (15,)),
    ("ch_dw", (256, 256, 256), None, "f64", 1, (2,)), ("ch_dw", (256, 256, 256), None, "f32", 3, (15,)),
    ("ch_dw", (128, 128, 128), None, "f64", 1, (15,)),
    ("ac", (1024, 1024), WALLS, "f64", 2, (2,)), ("ac", (1100, 1000), None, "f64", 1, (13, 14))])
def test_short_calls_on_large_grids(model, shape, bc, prec, steps, bodies):
    a = start(shape, 1, 3700, prec)
    got = []
    for variant in (0, 1):
        with mx.Grid(shape, precision=prec, bc=bc) as g:
            g.set_variant(variant)
            g.upload(a)
            g.step(model, PARAMS[model], steps)
            if variant == 0:
                assert g.get_kernel()["opt"] in bodies, g.get_kernel()
            got.append(g.download())
    assert np.array_equal(*got)
