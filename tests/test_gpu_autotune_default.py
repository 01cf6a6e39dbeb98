"""GPU: the autotuner times the default kernel too, and every tile of the
multi-step kernels, so a tuned state is no slower than an untuned one."""
import re

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

mx = pytest.importorskip("mmsp_amd")

PARAMS = {"ac": [1.0, 1.0, 1.0, 1.0, 0.01], "ch_dw": [1.0, 1.0, 0.005], "gg": [0.01], "zener": [0.01]}
MARCH = {"f64": {(26, 52), (16, 64), (32, 32), (16, 32), (16, 16), (26, 56), (42, 56)},
         "f32": {(32, 64), (26, 52), (32, 32), (16, 32), (16, 16), (26, 56), (30, 56)}}


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("model,shape,q", [("ac", (300, 200), 1), ("ch_dw", (300, 200), 1), ("gg", (150, 130), 8),
                                           ("zener", (150, 130), 4), ("ac", (60, 70, 80), 1), ("ch_dw", (60, 70, 80), 1),
                                           ("ch_dw", (96, 100, 104), 1), ("gg", (40, 50, 97), 8)])
def test_the_default_is_a_candidate(model, shape, q, prec):
    a = O.uniform(int(np.prod(shape)) * q, 3800, 0.3, 0.7).reshape(shape + ((q,) if q > 1 else ()))
    with mx.Grid(shape, fields=q, vector=q > 1, precision=prec) as g:
        a = a.astype(g.dtype)
        g.upload(a)
        g.step(model, PARAMS[model], 8)
        default, state = g.get_kernel(), g.download()
        g.upload(a)
        lines = [{k: float(v) for k, v in re.findall(r"(\w+)=([0-9.]+)", r)}
                 for r in g.autotune(model, PARAMS[model], trial_steps=3).splitlines()]
        same = [r for r in lines if all(r[k] == default[k] for k in ("variant", "ty", "tz", "chunk", "opt"))]
        assert same, default
        if len(shape) == 3 and q == 1:
            assert {(int(r["ty"]), int(r["tz"])) for r in lines if r["opt"] == 15} == MARCH[prec]
        assert min(r["mean_us"] for r in lines) <= same[0]["mean_us"]
        g.step(model, PARAMS[model], 8)
        assert np.array_equal(g.download(), state)
