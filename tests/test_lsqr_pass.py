"""LSQR with one right-hand side, where one pass over A serves both products: columns at the edges of a
thread's 2048-column pieces (and past the last of them, where the products are apart again), rows at the
edges of the register sets and of 255 blocks, FP64 here and FP32 in the mixed Laplace form."""
import numpy as np
import pytest

from test_lsqr_shapes import _system


@pytest.mark.gpu
@pytest.mark.parametrize("m,n", [(2, 1), (7, 9), (8, 64), (9, 1023), (255, 254), (256, 255), (2041, 129), (2049, 2047),
                                 (2049, 2049), (2100, 2050), (300, 4097), (520, 6143), (60, 6145), (31, 8191),
                                 (33, 8192), (33, 8193), (4100, 40)])
def test_gpu_lsqr_pass(ctx, m, n):
    A, b = _system(m, n, 1)
    X, st = ctx.lsqr_dense(A, b, eps=1e-13, precon=False)
    assert all(s in (0, 1, 2) for s in st["istop"])
    # identity plus a coupling of norm <= 0.6 (least-norm solution for m < n): a relative A^T r of 1e-13
    # leaves an error below 16 * 1e-13 of the solution; two orders of margin
    ref = np.linalg.lstsq(A, b, rcond=None)[0]
    assert np.linalg.norm(X - ref) < 2e-10 * np.linalg.norm(ref)


@pytest.mark.gpu
@pytest.mark.parametrize("maxit", [1, 2, 7, 8, 9, 16, 17])
def test_gpu_lsqr_pass_iterates(ctx, maxit):
    """The iterate of every iteration limit around the polls, against the recurrence in numpy."""
    m, n = 700, 333
    A, b = _system(m, n, 1)
    X, st = ctx.lsqr_dense(A, b, eps=1e-30, maxit=maxit, precon=False)
    assert st["nit"] == [maxit]
    u = b[:, 0].copy()
    beta = np.linalg.norm(u)
    u /= beta
    v = A.T @ u
    alpha = np.linalg.norm(v)
    v /= alpha
    w, x, phibar, rhobar = v.copy(), np.zeros(n), beta, alpha
    for _ in range(maxit):
        u = A @ v - alpha * u
        beta = np.linalg.norm(u)
        u /= beta
        v = A.T @ u - beta * v
        alpha = np.linalg.norm(v)
        v /= alpha
        rho = np.hypot(rhobar, beta)
        c, s = rhobar / rho, beta / rho
        theta, rhobar = s * alpha, -c * alpha
        phi, phibar = c * phibar, s * phibar
        x += phi / rho * w
        w = v - theta / rho * w
    # 17 steps of a well-conditioned recurrence in another order of sums
    assert np.linalg.norm(X[:, 0] - x) < 1e-12 * np.linalg.norm(x)
