"""The one-pass product of LSQR in FP32, which the mixed Laplace form takes with one, two, three and four pieces of
2048 columns a row (register sets of eight, eight, four and four rows); against the FP64 form, whose own are of
eight, four, two and two. A sphere with a known linear function on its lower half and its flux on the upper one."""
import numpy as np
import pytest

from andromeda_amd import api
from andromeda_amd import mesh as M


def _solve(ctx, nu, precision):
    m = M.geodesic_sphere(nu, 1.0)
    a, b, c = (m.xyz[m.con[:, k]] for k in range(3))
    n = np.cross(b - a, c - a)
    n /= np.linalg.norm(n, axis=1)[:, None]
    g = np.array([0.4, -0.7, 1.1])
    m.bcid = np.where((a + b + c)[:, 2] < 0.0, 1, 2).astype(np.int32)
    m.walls = ["lower", "upper"]
    u, q = m.xyz @ g, -(n @ g)  # the flux of unit diffusivity
    known = np.zeros(m.nnodes, dtype=bool)
    known[np.unique(m.con[m.bcid == 1])] = True
    bc = np.array([[api.BC_FUNCTION, api.BC_FLUX]], dtype=np.int32)
    r = ctx.laplace_solve(m, [api.Subdomain([1, 2], [1.0, 1.0], 1.0)], bc,
                          np.where(known, u, 0.0)[None], np.where(m.bcid == 2, q, 0.0)[None], eps=1e-13, maxit=0,
                          precision=precision)[0]
    return r, u


@pytest.mark.gpu
@pytest.mark.parametrize("nu,pieces", [(11, 1), (12, 2), (16, 2), (17, 3), (19, 3), (21, 4), (23, 4)])
def test_gpu_pass_mixed(ctx, nu, pieces):
    ref, u = _solve(ctx, nu, api.PREC_FP64)
    ctx.profile(True)
    try:
        r, _ = _solve(ctx, nu, api.PREC_MIXED)
        names = ctx.profile_read()
    finally:
        ctx.profile(False)
    assert "lsqr_pass" in names and -(-r.nx // 2048) == pieces and r.istop in (1, 2)
    # the mixed form's stated distance, 1e-6 of u and 1e-5 of q on systems of up to 1519 unknowns, times the growth of
    # the condition with the mesh (2.3 up to 8192) and a margin of four
    assert np.linalg.norm(r.u - ref.u) < 1e-5 * np.linalg.norm(ref.u)
    assert np.linalg.norm(r.q - ref.q) < 1e-4 * np.linalg.norm(ref.q)
    # the collocation holds for a linear field on flat elements, up to its quadrature
    assert np.linalg.norm(r.u - u) < 1e-3 * np.linalg.norm(u)
