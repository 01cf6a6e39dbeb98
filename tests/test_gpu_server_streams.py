"""GPU: rounds whose launches run on two streams: 2-D and 3-D requests in FP32
and FP64 together, in every combination that forks a round or does not."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

mx = pytest.importorskip("mmsp_amd")

PARAMS = [1.0, 1.0, 0.005]
WORK = {"2d32": ((40, 53), 30), "3d32": ((11, 17, 20), 25), "2d64": ((33, 61), 70), "3d64": ((9, 21, 18), 65)}


@pytest.mark.parametrize("kinds", ["2d32,3d32", "3d32,3d64", "2d32,2d64", "2d64,3d64", "2d32,3d64", "3d32,2d64",
                                   "2d32,3d32,2d64,3d64"])
def test_mixed_rounds(kinds):
    work = [WORK[k] for k in kinds.split(",") for _ in range(2)]
    inits = [np.random.default_rng(50 + k).uniform(0.4, 0.6, s) for k, (s, _) in enumerate(work)]
    sv = mx.Server("ch_dw", "f32", hbm_budget=1 << 30, max_slots=16, chunk_steps=10, fp64_above_steps=50)
    try:
        ids = [sv.submit(a, PARAMS, steps) for a, (_, steps) in zip(inits, work)]
        for i in ids:
            sv.wait(i)
        got = [sv.fetch(i) for i in ids]
    finally:
        sv.close()
    for a, (shape, steps), g in zip(inits, work, got):
        prec = "f64" if steps > 50 else "f32"
        with mx.Grid(shape, precision=prec) as ref:
            ref.upload(a.astype(np.float64 if prec == "f64" else np.float32))
            ref.step("ch_dw", PARAMS, steps)
            assert np.array_equal(np.asarray(g, dtype=np.float64), ref.download().astype(np.float64)), (shape, steps)
