"""GPU: the 2-D multi-phase grain growth strips, bitwise against the oracle:
strip edges, every boundary, nodes with none to all of the fields present."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

mx = pytest.importorskip("mmsp_amd")

P, N, M, D = O.PERIODIC, O.NEUMANN, O.MIRROR, O.DIRICHLET
PARAMS = [0.01, 8.0, 1.0, 1.0]


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("q", [2, 4, 8])
@pytest.mark.parametrize("bc", [None, [(N, N), (M, D)], [(P, P), (N, P)], [(M, N), (P, P)]],
                         ids=["periodic", "walls", "columns", "rows"])
def test_strips(bc, q, prec):
    """Strips of 62 columns: narrower, exact, one column over; chunks of 2, 3
    and 8 rows and the default; unit and other grid weights."""
    for k, shape in enumerate([(2, 3), (9, 62), (14, 63), (21, 125)]):
        r = np.random.default_rng(3100 + k)
        ids = np.take(np.repeat(r.integers(0, q, (shape[0], (shape[1] + 7) // 8)), 8, axis=1), np.arange(shape[1]), axis=1)
        a = np.zeros(shape + (q,))
        np.put_along_axis(a, ids[..., None], 1.0, axis=-1)
        # from left to right more and more fields present, negative ones among them
        a += (r.random(a.shape) * np.linspace(0, 1, shape[1])[None, :, None] > 0.6) * r.uniform(-0.1, 0.4, a.shape)
        if prec == "f32":
            a = a.astype(np.float32)
        dx = [0.8, 1.1] if k % 2 else None
        exp = O.gg_aniso(a, PARAMS, 5, form=prec, bc=bc, dx=dx)
        for chunk in (0, 2, 3, 8):  # 0: the default
            with mx.Grid(shape, fields=q, vector=True, precision=prec, bc=bc, dx=dx) as g:
                if chunk:
                    g.set_variant(2)
                    g.set_tile(1, 64, chunk)
                    g.set_tile_options(body=2)
                g.upload(a)
                g.step("gg_aniso", PARAMS, 5)
                assert np.array_equal(g.download(), exp), (shape, chunk)
