"""Dense LSQR over the shapes where its kernels change path: sizes around the 16-row tiles, the row
splits and the 64- to 1024-column segments, one and several right-hand sides (plain and interleaved
vectors), few and many column segments (U formed inside the A^T U kernel or on its own)."""
import numpy as np
import pytest


def _system(m, n, nrhs):
    rng = np.random.default_rng(1000 * m + n)
    k = min(m, n)
    A = rng.standard_normal((m, n)) * (0.3 / np.sqrt(max(m, n)))
    A[np.arange(k), np.arange(k)] += 1.0
    return A, rng.standard_normal((m, nrhs))


@pytest.mark.gpu
@pytest.mark.parametrize("nrhs", [1, 2, 8, 9])
@pytest.mark.parametrize("m,n", [(1, 1), (3, 2), (15, 17), (16, 16), (129, 127), (255, 257), (520, 511), (1025, 1000)])
def test_gpu_lsqr_shapes(ctx, m, n, nrhs):
    A, B = _system(m, n, nrhs)
    X, st = ctx.lsqr_dense(A, B, eps=1e-13)
    # identity plus a coupling of norm <= 0.6: condition below 4 (columns scaled), so a relative
    # A^T r of 1e-13 leaves an error below 16 * 1e-13 of the solution; two orders of margin
    ref = np.linalg.lstsq(A, B, rcond=None)[0]
    assert all(s in (0, 1, 2) for s in st["istop"])
    if m >= n:
        assert np.linalg.norm(X - ref) < 2e-10 * np.linalg.norm(ref)
    else:  # not unique, and column scaling picks another solution: the residual vanishes
        assert np.linalg.norm(A @ X - B) < 2e-10 * np.linalg.norm(B)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,nrhs", [(40, 4352, 1), (33, 17000, 3), (8200, 300, 6)])
def test_gpu_lsqr_many_segments(ctx, m, n, nrhs):
    A, B = _system(m, n, nrhs)
    X, st = ctx.lsqr_dense(A, B, eps=1e-13, precon=False)
    assert all(s in (1, 2) for s in st["istop"])
    ref = np.linalg.lstsq(A, B, rcond=None)[0]  # without scaling LSQR gives the least-norm solution
    assert np.linalg.norm(X - ref) < 2e-10 * np.linalg.norm(ref)


@pytest.mark.gpu
def test_gpu_lsqr_stops(ctx):
    """A zero right-hand side, an exact start and the iteration limit, off the multiples of the polls."""
    A, B = _system(200, 150, 3)
    X, st = ctx.lsqr_dense(A, np.zeros((200, 2)))
    assert not X.any() and st["nit"] == [0, 0]
    for maxit in (1, 7, 8, 9, 13):
        X, st = ctx.lsqr_dense(A, B, eps=1e-15, maxit=maxit)
        assert st["nit"] == [maxit] * 3 and st["istop"] == [5] * 3
        x1, st1 = ctx.lsqr_dense(A, B[:, 1], eps=1e-15, maxit=maxit)
        assert st1["nit"] == [maxit]
        # the same recurrence on plain and on interleaved vectors, rounding apart
        assert np.linalg.norm(x1[:, 0] - X[:, 1]) < 1e-12 * np.linalg.norm(X[:, 1])
