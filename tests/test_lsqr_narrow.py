"""LSQR with one right-hand side of narrow systems: the pass over A that serves both products up to 4080 rows or
from 400 columns on, a kernel for each product otherwise. On both sides of the line, against a direct solve."""
import numpy as np
import pytest

from test_lsqr_shapes import _system


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,one_pass", [(4080, 3, True), (4081, 3, False), (4081, 399, False), (4081, 400, True),
                                          (20011, 64, False), (9000, 127, False), (4097, 1, False), (12000, 401, True)])
def test_gpu_lsqr_narrow(ctx, m, n, one_pass):
    A, b = _system(m, n, 1)
    A[n:] *= np.sqrt(m / n) / 4  # rows below the identity carry as much of the system as those in it
    ctx.profile(True)
    try:
        X, st = ctx.lsqr_dense(A, b, eps=1e-13, precon=False)
        names = ctx.profile_read()
    finally:
        ctx.profile(False)
    assert ("lsqr_pass" in names) == one_pass
    assert all(s in (1, 2) for s in st["istop"])
    ref = np.linalg.lstsq(A, b, rcond=None)[0]
    # singular values from 0.9 on, condition below 1.5: a relative A^T r of 1e-13 leaves an error of the solution below
    # 1.5e-13 of the residual, the products' rounding as much of the solution; an order of margin
    assert np.linalg.norm(X - ref) < 2e-12 * (np.linalg.norm(b - A @ ref) + np.linalg.norm(ref))
