"""GPU: the multi-step kernels' forms without the multiplications by grid weights
and coefficients that are all one, and the forms beside them (only the weights
one, one coefficient not), bitwise against the oracle."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

mx = pytest.importorskip("mmsp_amd")

CASES = {"ac": ([1.0, 1.0, 1.0, 1.0, 0.01], [1.0, 1.0, 1.0, 0.5, 0.02], [1.0, 1.5, 1.0, 1.0, 0.01], [0.5, 1.0, 1.0, 1.0, 0.01],
                [1.0, 1.0, 0.7, 1.0, 0.01]),
         "ch": ([1.0, 1.0, 1.0, 1.0, 0.01], [1.0, 1.5, 1.0, 1.0, 0.01], [1.0, 1.0, 0.7, 1.0, 0.01]),
         "ch_dw": ([1.0, 1.0, 0.005], [0.6, 1.0, 0.005])}


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("shape", [(37, 101), (13, 29, 60)], ids=["2d", "3d"])
@pytest.mark.parametrize("model", list(CASES))
def test_unit_coefficients(model, shape, prec):
    a = O.uniform(int(np.prod(shape)), 3300, -0.9, 0.9).reshape(shape)
    a.flat[::7] = 0.0  # zero laplacians and zero values too
    a.flat[3::11] = -0.0
    if prec == "f32":
        a = a.astype(np.float32)
    for params in CASES[model]:
        for dx in (None, [0.9] * len(shape)):
            if model == "ac":
                exp = O.ac(a, params, 9, form=prec, dx=dx)
            else:
                exp = O.ch(a, params, 9, mu=O.MU_POLY if model == "ch" else O.MU_DW, form=prec, dx=dx)
            with mx.Grid(shape, precision=prec, dx=dx) as g:
                g.upload(a)
                g.step(model, params, 9)
                assert np.array_equal(g.download(), exp), (params, dx)
