"""The classification pass with a block a row and with a wave a row (1536 rows of a call and more): the counts
of a body are the same in a call of its own and in one with others."""
import numpy as np
import pytest

from andromeda_amd import api
from andromeda_amd import mesh as M

from test_learned import _model


@pytest.mark.gpu
def test_gpu_classify_rows(ctx):
    z = _model()
    ctx.set_quadrature_model(z["params"], float(z["confidence"]), float(z["near_ratio"]), z["far_table"])
    rng = np.random.default_rng(11)
    ms = [M.random_superellipsoid(rng, nu)[0] for nu in (2, 5, 7)] + [M.random_fibre(rng, 322)[0]]
    own = [ctx.resistance(m, precision=api.PREC_LEARNED) for m in ms]
    both = ctx.resistance_batch(ms, precision=api.PREC_LEARNED)
    assert sum(m.nelem for m in ms) >= 1536 > max(m.nelem for m in ms)
    for a, b, m in zip(own, both, ms):
        assert a.quad_points == b.quad_points and a.pairs_learned == b.pairs_learned
        assert a.pairs_fallback == b.pairs_fallback
        assert a.pairs_learned + a.pairs_fallback <= m.nelem * (m.nelem - 1)
        # the same matrices; another split of the products' sums moves a solution through FP32 products
        assert np.abs(a.FT - b.FT).max() < 2e-7 * np.abs(a.FT).max()
