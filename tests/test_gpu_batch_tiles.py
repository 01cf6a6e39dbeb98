"""GPU: a batch's tile read back can be set again, and the multi-step kernels are
reached again after another tile, bitwise against the oracle."""
import re

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


@pytest.mark.parametrize("model,shapes", [("ac", [(40, 60), (33, 49)]), ("ch_dw", [(40, 60), (17, 33, 18)]),
                                          ("ch", [(17, 33, 18), (20, 16, 34)])])
def test_a_tile_read_back_is_set_again(model, shapes):
    b, inits = members(model, shapes, "f64")
    with b:
        default = tile(b)
        assert default[2] == 0  # the multi-step kernels
        for other in ((64, 16, 8), (128, 32, 4)) + (((48, 4, 4),) if model == "ac" else ()):
            b.set_tile(*other)
            assert tile(b) == other
            check(b, inits, model, 9, "f64")
            b.set_tile(*default)
            assert tile(b) == default
            check(b, inits, model, 9, "f64")
        b.set_tile(64, 16, 8)
        report = b.autotune(trial_steps=2)
        assert re.search("blocks_per_cu=0 ", report), report
        check(b, inits, model, 9, "f64")


def test_the_multi_step_kernels_are_refused_where_they_do_not_run():
    for model, kw in (("ac", dict(bcs=[[(P, N), (P, P)]] * 2)), ("ac", dict(precision="f32ref"))):
        with mx.Batch([(20, 30), (30, 20)], model, **kw) as b:
            before = tile(b)
            for t in ((48, 8, 0), (56, 8, 0), (64, 8, 0)):
                with pytest.raises(mx.MmspxError):
                    b.set_tile(*t)
            assert tile(b) == before and before[2] > 0
