"""GPU: batches on the multi-step kernels (their default), bitwise against the
oracle's single steps."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

mx = pytest.importorskip("mmsp_amd")

P, N, M = O.PERIODIC, O.NEUMANN, O.MIRROR


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("walls", [False, True])
def test_allen_cahn_batch_takes_several_steps_per_pass(prec, walls):
    """Members of one strip to several, narrower than the halo, unlike weights;
    whole passes, a short last one, graphs that leave the buffers swapped."""
    shapes = [(3, 5), (40, 48), (33, 49), (70, 130), (2, 200)]
    bcs = [[(N, M), (P, P)] if walls and k % 2 else [(P, P), (N, N)] if walls else [(P, P), (P, P)] for k in range(5)]
    dxs = [[1.0, 1.0], [0.9, 1.1], [1.0, 1.0], [1.0, 1.0], [1.2, 1.0]]
    params = np.array([[1.0, 1.0, 0.5 + 0.3 * k, 1.0, 0.01] for k in range(5)])
    inits = [O.uniform(s[0] * s[1], 2100 + k, -1.0, 1.0).reshape(s) for k, s in enumerate(shapes)]
    if prec == "f32":
        inits = [a.astype(np.float32) for a in inits]
    for steps, graph in ((8, 0), (13, 0), (53, 24), (53, 17)):
        with mx.Batch(shapes, "ac", precision=prec, bcs=bcs, dxs=dxs) as b:
            b.set_params(params)
            for m, a in enumerate(inits):
                b.upload(m, a)
            b.step(steps, graph_steps=graph)
            for m, a in enumerate(inits):
                exp = O.ac(a, params[m], steps, form=prec, bc=bcs[m], dx=dxs[m])
                assert np.array_equal(b.download(m), exp), (steps, graph, m)


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("model", ["ch", "ch_dw"])
def test_cahn_hilliard_batch_takes_several_steps_per_pass(model, prec):
    """2-D and 3-D members together: their passes differ in steps, so in the
    buffer each leaves its members in."""
    shapes = [(6, 7, 9), (30, 40), (17, 33, 18), (5, 100), (20, 16, 34)]
    par = [1.0, 1.0, 0.8, 1.0, 0.01] if model == "ch" else [0.9, 1.0, 0.005]
    inits = [O.uniform(int(np.prod(s)), 2200 + k, 0.3, 0.7).reshape(s) for k, s in enumerate(shapes)]
    if prec == "f32":
        inits = [a.astype(np.float32) for a in inits]
    mu = O.MU_POLY if model == "ch" else O.MU_DW
    for steps, graph in ((4, 0), (7, 0), (26, 6), (25, 5)):
        with mx.Batch(shapes, model, precision=prec) as b:
            b.set_params(np.array([par] * len(shapes)))
            for m, a in enumerate(inits):
                b.upload(m, a)
            b.step(steps, graph_steps=graph)
            for m, a in enumerate(inits):
                assert np.array_equal(b.download(m), O.ch(a, par, steps, mu=mu, form=prec)), (steps, graph, m)
