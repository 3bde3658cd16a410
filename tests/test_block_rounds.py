"""The block GMRES of the fast forms over numbers of rounds around its chunks (the reflectors eight rounds at
a time, the update sweep sixteen blocks at a time) and over both block widths (six rigid-body problems,
three strain fields), with restarts, against the plain FP64 path."""
import numpy as np
import pytest

from andromeda_amd import api
from andromeda_amd import mesh as M


def _body(kind):
    rng = np.random.default_rng(3)
    return M.random_superellipsoid(rng, 4)[0] if kind == "super" else M.random_fibre(rng, 500)[0]


@pytest.mark.gpu
@pytest.mark.parametrize("problems", [api.PROBLEMS_RIGID, api.PROBLEMS_STRAIN])
@pytest.mark.parametrize("kind,restart", [("super", 7), ("super", 8), ("super", 9), ("super", 16), ("super", 17),
                                          ("super", 0), ("fibre", 0)])
def test_gpu_block_rounds(ctx, kind, restart, problems):
    m = _body(kind)
    ref = ctx.resistance(m, precision=api.PREC_FP64, problems=problems)
    r = ctx.resistance(m, precision=api.PREC_MIXED, problems=problems, restart=restart)
    # a relative residual of 1e-6 and FP32 quadrature: the fast forms' stated error of 1e-6
    assert r.status == 0
    assert np.abs(r.FT - ref.FT).max() < 1e-6 * np.abs(ref.FT).max()
    tight = ctx.resistance(m, precision=api.PREC_MIXED, problems=problems, restart=restart, eps=1e-9)
    assert np.abs(tight.FT - ref.FT).max() < 1e-6 * np.abs(ref.FT).max()


@pytest.mark.gpu
def test_gpu_block_rounds_in_batch(ctx):
    """Bodies of one batch stop in different rounds; each result is that of the body on its own (the
    product's column segments apart, which depend on how many rows are live)."""
    rng = np.random.default_rng(5)
    ms = [M.random_superellipsoid(rng, nu)[0] for nu in (3, 6, 4)] + [M.random_fibre(rng, 320)[0]]
    out = ctx.resistance_batch(ms, precision=api.PREC_MIXED)
    for m, r in zip(ms, out):
        one = ctx.resistance(m, precision=api.PREC_MIXED)
        assert r.status == one.status == 0
        # another order of the product's sums moves a solution by rounding through FP32 products
        assert np.abs(r.FT - one.FT).max() < 2e-7 * np.abs(one.FT).max()
