"""Domain values and surface pressure where their work is dealt out differently: one point (every chunk
of 64 elements a workgroup of its own), a few, and enough points for one workgroup each; element counts
off the multiples of 64 and 256; a low and the full triangle rule."""
import numpy as np
import pytest

from andromeda_amd import mesh as M


def _data(nu):
    m = M.random_superellipsoid(np.random.default_rng(nu), nu)[0]
    rng = np.random.default_rng(10 + nu)
    return m, rng.normal(size=(m.nnodes, 3)), rng.normal(size=(m.nelem, 3)), rng


# FP64 sums of some 1e5 terms on both sides: 1e-13 of the largest value, three orders of margin as in
# the oracle tests of these entry points
@pytest.mark.gpu
@pytest.mark.parametrize("nu,npts,itri", [(1, 1, 5), (3, 1, 5), (3, 5, 1), (4, 600, 2), (5, 37, 5), (8, 3, 3)])
def test_gpu_domain_splits(ctx, orc, nu, npts, itri):
    m, u, q, rng = _data(nu)
    pts = rng.uniform(-0.15, 0.15, size=(npts, 3))
    vel, p, err = ctx.stokes_domain_values(m, pts, u, q, diff=1.7, itri=itri)
    vo, po, eo = orc.stokes_domain_values(m, pts, u, q, diff=1.7, itri=itri)
    assert np.abs(vel - vo).max() < 1e-10 * np.abs(vo).max()
    assert np.abs(p - po).max() < 1e-10 * np.abs(po).max()
    assert np.abs(err - eo).max() < 1e-10


@pytest.mark.gpu
@pytest.mark.parametrize("nu,itri", [(1, 5), (3, 2), (6, 5), (8, 1)])
def test_gpu_surface_splits(ctx, orc, nu, itri):
    m, u, q, _ = _data(nu)
    p = ctx.stokes_surface_pressure(m, u, q, diff=0.8, itri=itri)
    po = orc.stokes_surface_pressure(m, u, q, diff=0.8, itri=itri)
    assert np.abs(p - po).max() < 1e-10 * np.abs(po).max()
