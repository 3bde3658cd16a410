"""Matrices on their way to the host: sizes below and above the threaded copy's limit and pieces that end
inside a matrix, each layout, against rows fetched a few at a time (which never reach that limit)."""
import numpy as np
import pytest

from andromeda_amd import mesh as M


@pytest.mark.gpu
@pytest.mark.parametrize("nu", [2, 5, 8])  # 0.1, 4.5 and 29 MB of Laplace rows
def test_gpu_copy_sizes(ctx, nu):
    m = M.geodesic_sphere(nu)
    nsp = m.nnodes + m.nelem
    H, G, _ = ctx.assemble_laplace(m)
    Hc, Gc, _ = ctx.assemble_laplace(m, layout=1)
    assert np.array_equal(H, Hc) and np.array_equal(G, Gc)
    step = max(1, (1 << 20) // (8 * (H.shape[1] + G.shape[1])))
    for r0 in range(0, nsp, step * 7):
        r1 = min(nsp, r0 + step)
        h, g, _ = ctx.assemble_laplace_rows(m, r0, r1)
        assert np.array_equal(H[r0:r1], h) and np.array_equal(G[r0:r1], g)
