"""GPU: a state tuned for one model runs the other models of its kind: a tile
the autotuner chose gives way where its body does not run them; a tile the
caller set is refused."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

mx = pytest.importorskip("mmsp_amd")

PARAMS = {"ac": [1.0, 1.0, 1.0, 1.0, 0.01], "ch": [1.0, 1.0, 1.0, 1.0, 0.01], "ch_dw": [1.0, 1.0, 0.005], "gg": [0.01],
          "zener": [0.01], "gg_aniso": [0.01, 8.0, 1.0, 1.0],
          "ostwald": [0.001, 1.0, 1.0, 0.05, 0.95, 2.0, 1.0, 3.0, 2.0],
          "ac_noise": [1.0, 1.0, 1.0, 1.0, 0.01, 1.4, 20260107], "ch_noise": [1.0, 1.0, 1.0, 1.0, 0.01, 1.4, 20260107]}
SCALAR = ["ac", "ch", "ch_dw", "ac_noise", "ch_noise"]
VECTOR = ["gg", "zener", "gg_aniso", "ostwald"]


@pytest.mark.parametrize("tuned,shape,q,body", [("ch_dw", (70, 90), 1, 13), ("ch", (24, 40, 60), 1, 15), ("ac", (24, 40, 60), 1, 15),
                                                ("gg", (60, 70), 4, 16), ("gg", (40, 50, 97), 4, 17)])
def test_other_models_on_a_tuned_state(tuned, shape, q, body):
    a = O.uniform(int(np.prod(shape)) * q, 3900, 0.0, 1.0).reshape(shape + ((q,) if q > 1 else ()))
    models = VECTOR if q > 1 else SCALAR if len(shape) == 3 else SCALAR[:3] + ["ch_noise"]
    for model in models:
        states = []
        for tune in (False, True):
            with mx.Grid(shape, fields=q, vector=q > 1) as g:
                if tune:
                    g.autotune(tuned, PARAMS[tuned], trial_steps=2)
                g.upload(a)
                g.step(model, PARAMS[model], 5)
                states.append(g.download())
        assert np.array_equal(*states), model
        if model.endswith("noise") or model in ("gg_aniso", "ostwald"):  # the body set by the caller
            with mx.Grid(shape, fields=q, vector=q > 1) as g:
                g.set_tile_options(body=body)
                g.upload(a)
                with pytest.raises(mx.MmspxError):
                    g.step(model, PARAMS[model], 5)
