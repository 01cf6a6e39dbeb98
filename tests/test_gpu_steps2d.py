"""GPU: the 2-D multi-step wave strips (tile bodies 13 and 14) and the default
that chooses them, bitwise against the oracle's single steps."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

mx = pytest.importorskip("mmsp_amd")

P, N, M, D = O.PERIODIC, O.NEUMANN, O.MIRROR, O.DIRICHLET
AC, CH, DW = [1.0, 1.0, 1.3, 0.9, 0.01], [1.0, 1.0, 0.8, 1.0, 0.01], [1.0, 1.0, 0.005]


def expected(model, a, steps, prec, bc, dx):
    if model == "ac":
        return O.ac(a, AC, steps, form=prec, bc=bc, dx=dx)
    if model == "ch":
        return O.ch(a, CH, steps, mu=O.MU_POLY, form=prec, bc=bc, dx=dx)
    return O.ch(a, DW, steps, mu=O.MU_DW, form=prec, bc=bc, dx=dx)


# strips of 48 and 56 columns: one node, a last strip of one column, exact
# strips, a grid narrower than the halo; rows fewer than the halo and chunks
# that end in every place of the six-row march
SHAPES = [(1, 1), (3, 5), (7, 49), (13, 56), (26, 97), (31, 113)]


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("model", ["ac", "ch", "ch_dw"])
@pytest.mark.parametrize("bc", [None, [(P, P), (N, M)], [(M, D), (P, P)], [(N, M), (D, N)]],
                         ids=["periodic", "columns", "rows", "walls"])
def test_multi_step_strips(model, prec, bc):
    """Whole passes and a last pass of every shorter length, unit and other
    grid weights, chunks of 2 to 9 rows."""
    params = {"ac": AC, "ch": CH, "ch_dw": DW}[model]
    for k, shape in enumerate(SHAPES):
        if bc is not None and min(shape) < 2:
            continue  # a mirror side needs two nodes
        dx = None if k % 2 else [0.9, 1.1]
        a = O.uniform(int(np.prod(shape)), 900 + k, 0.3, 0.7).reshape(shape)
        if prec == "f32":
            a = a.astype(np.float32)
        for steps in (8, 13 + k):
            exp = expected(model, a, steps, prec, bc, dx)
            for tz in (0, 48, 56):  # 0: the default
                for chunk in (2, 3 + k) if tz else (0,):
                    with mx.Grid(shape, precision=prec, bc=bc, dx=dx) as g:
                        if tz:
                            g.set_variant(2)
                            g.set_tile(1, tz, chunk)
                        g.upload(a)
                        g.step(model, params, steps)
                        assert np.array_equal(g.download(), exp), (shape, steps, tz, chunk)
                        assert g.get_tile()["opt"] in ((13,) if tz == 48 else (14,) if tz == 56 else (13, 14))


def test_multi_step_strips_refuse_what_they_cannot_run():
    """An axis periodic on one side only keeps the one-step kernels, and so
    does the reference's float form."""
    with mx.Grid((20, 20), bc=[(P, N), (P, P)]) as g:
        a = O.uniform(400, 7, 0.3, 0.7).reshape(20, 20)
        g.upload(a)
        g.step("ac", AC, 9)
        assert np.array_equal(g.download(), O.ac(a, AC, 9, bc=[(P, N), (P, P)]))
        assert g.get_tile()["opt"] not in (13, 14)
        g.set_variant(2)
        g.set_tile(1, 48, 4)
        with pytest.raises(mx.MmspxError):
            g.step("ac", AC, 8)
    with mx.Grid((20, 20), precision="f32ref") as g:
        g.set_variant(2)
        g.set_tile(1, 56, 4)
        g.upload(np.zeros((20, 20)))
        with pytest.raises(mx.MmspxError):
            g.step("ac", AC, 8)
