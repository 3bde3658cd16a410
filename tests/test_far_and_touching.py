"""Integrals at the ends of the distances' range: a source on a quadrature point of another element has an infinite
1 / r there, elements so far apart that the square of their distance overflows have none."""
import numpy as np
import pytest

from andromeda_amd import mesh as M


def _pair(shift):
    tri = np.array([[1.0, 0.0, 0.0], [0.0, 1.0, 0.0], [0.0, 0.0, 0.0]])
    con = np.array([[0, 1, 2], [3, 4, 5]], dtype=np.int32)
    return M.Mesh(np.vstack([tri, tri + shift]), con, np.array([1, 1], dtype=np.int32), "pair")


@pytest.mark.gpu
@pytest.mark.parametrize("itri", [1, 2, 5])
def test_gpu_touching(ctx, itri):
    """Two elements in one place, nodes of their own: the centre of one is a point of the other's rule where
    the rule has its centroid (7 and 25 points, not 126)."""
    G = ctx.assemble_laplace(_pair(0.0), itri=itri)[1]
    row = G[6:]  # the two centres
    assert np.isfinite(np.diag(row)).all() and (np.diag(row) > 0).all()
    if itri < 5:
        assert np.isposinf(row[0, 1]) and np.isposinf(row[1, 0])
    else:
        assert row[0, 1] > 0 and np.isfinite(row[0, 1])


@pytest.mark.gpu
def test_gpu_far_apart(ctx):
    H, G, _ = ctx.assemble_laplace(_pair(np.array([0.0, 0.0, 1e160])))
    for a in (G[:3, 1], G[3:6, 0], G[6, 1], G[7, 0], H[:3, 3:].ravel(), H[3:6, :3].ravel()):
        assert (np.asarray(a) == 0).all()


@pytest.mark.gpu
def test_gpu_quads_far_apart(ctx):
    quad = np.array([[0.0, 0.0, 0.0], [1.0, 0.0, 0.0], [1.0, 1.0, 0.0], [0.0, 1.0, 0.0]])
    m = M.Mesh(np.vstack([quad, quad + np.array([0.0, 0.0, 1e160])]), np.arange(8, dtype=np.int32).reshape(2, 4),
               np.array([1, 1], dtype=np.int32), "quads")
    H, G, _ = ctx.assemble_laplace(m)
    for a in (G[:4, 1], G[4:8, 0], G[8, 1], G[9, 0], H[:4, 4:].ravel(), H[4:8, :4].ravel()):
        assert (np.asarray(a) == 0).all()
