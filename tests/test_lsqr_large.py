"""LSQR with several right-hand sides of a matrix beyond the 256 MB cache: U is formed once and A^T U goes over
splits as long as leave one round of blocks; at fewer than eight column panels U is formed in the product, over 256
rows. Splits that end within a wave's rows and within the pieces of 64 rows in which U is staged."""
import numpy as np
import pytest

from test_lsqr_shapes import _system


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,nrhs,rows", [(5700, 5700, 3, 576), (33000, 1025, 6, 640), (36000, 896, 2, 256),
                                           (2100, 16500, 2, 1088)])
def test_gpu_lsqr_large(ctx, m, n, nrhs, rows):
    A, B = _system(m, n, nrhs)
    if m >= n:
        want = B[:n]
        b = A @ want
    else:  # the solution of least norm
        b = B
        want = A.T @ np.linalg.solve(A @ A.T, b)
    ctx.profile(True)
    try:
        X, st = ctx.lsqr_dense(A, b, eps=1e-13, precon=False)
        t = ctx.profile_read()["lsqr_gemv_t"]
    finally:
        ctx.profile(False)
    # identity plus a coupling of norm <= 0.6: a relative residual of 1e-13 leaves an error below
    # 4 * 1e-13 of the solution; two orders of margin
    assert all(s in (1, 2) for s in st["istop"])
    assert np.linalg.norm(X - want) < 4e-11 * np.linalg.norm(want)
    # a launch's bytes: A, U and V, and the partial result of every split, eight columns each
    partial = t["bytes"] / t["launches"] - 8.0 * m * n - 64.0 * (m + n)
    assert round(partial / (64.0 * n)) == -(-m // rows)
