"""GPU: the multi-step kernels leave out the addition that turns a laplacian of
-0 into +0: the signs of zeros (and every other bit) are the oracle's."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

mx = pytest.importorskip("mmsp_amd")

PARAMS = {"ac": [1.0, 1.0, 1.3, 0.9, 0.01], "ch": [1.0, 1.0, 0.8, 1.0, 0.01], "ch_dw": [0.9, 1.0, 0.005], "gg": [0.01],
          "zener": [0.01], "gg_aniso": [0.01, 8.0, 1.0, 1.0]}
UNIT = {"ac": [1.0, 1.0, 1.0, 1.0, 0.01], "ch": [1.0, 1.0, 1.0, 1.0, 0.01], "ch_dw": [1.0, 1.0, 0.005]}


def expected(model, a, p, steps, prec, dx):
    if model == "ac":
        return O.ac(a, p, steps, form=prec, dx=dx)
    if model in ("gg", "zener"):
        return (O.gg if model == "gg" else O.zener)(a, p[0], steps, form=prec, dx=dx)
    if model == "gg_aniso":
        return O.gg_aniso(a, p, steps, form=prec, dx=dx)
    return O.ch(a, p, steps, mu=O.MU_POLY if model == "ch" else O.MU_DW, form=prec, dx=dx)


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("shape,q", [((37, 101), 1), ((13, 29, 60), 1), ((40, 70), 4), ((40, 50, 97), 8)])
def test_signs_of_zero(shape, q, prec):
    n = int(np.prod(shape)) * q
    a = O.uniform(n, 4300, -0.9, 0.9)
    a[: n // 2] = np.where(np.arange(n // 2) // 3 % 5 < 3, -0.0, 0.0)  # runs of either zero
    a[n // 8: n // 4] = -0.0
    a[n // 2:: 7] = 0.0
    a[n // 2 + 3:: 11] = -0.0
    a = a.reshape(shape + ((q,) if q > 1 else ())).astype(np.float64 if prec == "f64" else np.float32)
    bits = np.uint64 if prec == "f64" else np.uint32
    for model in ("gg", "zener", "gg_aniso") if q > 1 else ("ac", "ch", "ch_dw"):
        for p in [PARAMS[model]] + ([UNIT[model]] if model in UNIT else []):
            for dx in (None, [0.9] * len(shape)):
                for steps in (1, 2, 4, 8):
                    with mx.Grid(shape, fields=q, vector=q > 1, precision=prec, dx=dx) as g:
                        g.upload(a)
                        g.step(model, p, steps)
                        got, exp = g.download(), expected(model, a, p, steps, prec, dx)
                    assert np.array_equal(got.view(bits), exp.view(bits)), (model, p, dx, steps)
