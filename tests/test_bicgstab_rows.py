"""BiCGSTAB's product over rows that start anywhere in a 128-byte line, at the edges of its 16-column blocks
and 256-column segments, against the same system with every row on a line: the sums keep their order, so
the results are the same bits."""
import numpy as np
import pytest

from test_zz_no_alloc import _Dev, _system


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 31, 33, 48, 255, 257, 290, 1041])
@pytest.mark.parametrize("pad,offset,nrhs", [(0, 0, 1), (1, 1, 3), (2, 0, 9), (15, 7, 2)])
def test_gpu_bicgstab_rows(ctx, n, pad, offset, nrhs):
    A, B, X0 = _system(n, nrhs, n + pad)
    Xr, ir = ctx.bicgstab_dense(A, B, X0=X0.copy(), tol=1e-12, maxit=200)
    lda = n + pad
    Ap = np.full(offset + n * lda, np.nan)  # what lies outside the matrix never counts
    for i in range(n):
        Ap[offset + i * lda:offset + i * lda + n] = A[i]
    Ap = Ap[:offset + (n - 1) * lda + n]  # the last row ends the allocation
    dev = _Dev()
    try:
        dA, dB, dX = dev.put(Ap), dev.put(B.T), dev.put(X0.T)
        info = ctx.bicgstab_dense_noalloc(n, dA + 8 * offset, lda, nrhs, dB, dX, tol=1e-12, maxit=200)
        X = dev.get(dX, (nrhs, n)).T
    finally:
        dev.free()
    assert info["nit"] == ir["nit"] and info["status"] == ir["status"]
    assert np.array_equal(X, Xr)
    assert np.linalg.norm(A @ X - B) <= 1e-11 * np.linalg.norm(B)
