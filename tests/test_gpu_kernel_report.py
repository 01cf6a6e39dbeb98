"""GPU: get_kernel names the kernel that ran, and that kernel set again on
another state runs again with the same bits."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

mx = pytest.importorskip("mmsp_amd")

AC, DW = [1.0, 1.0, 1.0, 1.0, 0.01], [1.0, 1.0, 0.005]


def advance(model, params, shape, q, prec, steps, kernel=None):
    a = O.uniform(int(np.prod(shape)) * q, 3500, 0.3, 0.7).reshape(shape + ((q,) if q > 1 else ()))
    with mx.Grid(shape, fields=q, vector=q > 1, precision=prec) as g:
        if kernel:
            g.set_variant(2)
            g.set_tile(kernel["ty"], kernel["tz"], kernel["chunk"])
            g.set_tile_options(body=kernel["opt"])
        g.upload(a if prec == "f64" else a.astype(np.float32))
        g.step(model, params, steps)
        return g.get_kernel(), g.download()


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("model,params,shape,q,bodies", [
    ("ac", AC, (60, 90), 1, (13, 14)), ("ch_dw", DW, (60, 90), 1, (13, 14)), ("gg", [0.01], (40, 60), 4, (16,)),
    ("ac", AC, (40, 41, 42), 1, (15,)), ("ch_dw", DW, (40, 41, 42), 1, (15,)), ("ch_dw", DW, (96, 100, 104), 1, (15,)),
])
def test_the_kernel_that_ran(model, params, shape, q, bodies, prec):
    ran, state = advance(model, params, shape, q, prec, 8)
    assert ran["variant"] == 2 and ran["opt"] in bodies, ran
    again, same = advance(model, params, shape, q, prec, 8, ran)
    assert again == ran and np.array_equal(same, state)
