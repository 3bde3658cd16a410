"""Integral rows over element counts around the turns of a row's workgroup (64 to 256 elements), colours
that straddle the turns, meshes mixed of quadrilaterals and triangles, elements long enough for more
than two sub-cells, and meshes whose node rows do not fit LDS; against the oracle."""
import numpy as np
import pytest

from andromeda_amd import mesh as M


def _mesh(kind):
    if kind.startswith("geo"):
        return M.geodesic_sphere(int(kind[3:]), 1.1)
    if kind.startswith("fibre"):
        return M.fibre(1.0, 0.2, 2.5, int(kind[5:]))
    m = M.cubed_sphere(int(kind[4:]), 0.8)
    m.xyz = m.xyz * np.array([1.0, 1.7, 4.0])  # long elements: several sub-cells per direction
    return M.split_some_quads(m) if kind.startswith("mixd") else m


def _close(a, b):
    # sums of up to 1e5 FP64 terms in another order: 1e-13 of the largest entry, with margin; the same
    # bound as the other assembly tests
    return np.abs(a - b).max() < 1e-10 * np.abs(b).max()


@pytest.mark.gpu
@pytest.mark.parametrize("kind,itri,iquad", [("geo1", 5, 4), ("geo2", 1, 4), ("geo3", 5, 4), ("fibre250", 3, 4),
                                             ("fibre270", 5, 4), ("quad1", 5, 4), ("quad3", 5, 1), ("mixd3", 2, 5),
                                             ("mixd6", 5, 4)])
def test_gpu_row_turns(ctx, orc, kind, itri, iquad):
    m = _mesh(kind)
    H, G, _ = ctx.assemble_laplace(m, itri=itri, iquad=iquad)
    Ho, Go, _ = orc.assemble_laplace(m, itri=itri, iquad=iquad)
    assert _close(H, Ho) and _close(G, Go)
    T, Gs, pT, pG, _ = ctx.assemble_stokes(m, itri=itri, iquad=iquad)
    To, Gso, pTo, pGo, _ = orc.assemble_stokes(m, itri=itri, pressure=True, iquad=iquad)
    for a, b in zip(T + Gs + pT + pG, To + Gso + pTo + pGo):
        assert np.abs(a - b).max() < 1e-10 * max(np.abs(To[0]).max(), np.abs(b).max())


@pytest.mark.gpu
def test_gpu_rows_outside_lds(ctx, orc):
    m = M.geodesic_sphere(15)  # 2252 nodes: nine node rows of 18 KB
    nn = m.nnodes
    for r0, r1 in ((7, 9), (nn - 1, nn + 1)):
        T, G, pT, pG, _ = ctx.assemble_stokes_rows(m, r0, r1)
        To, Go, pTo, pGo, _ = orc.assemble_stokes(m, rows=np.arange(r0, r1), pressure=True)
        for a, b in zip(T + G + pT + pG, To + Go + pTo + pGo):
            assert np.abs(a - b).max() < 1e-10 * np.abs(To[0]).max()
    m = M.geodesic_sphere(41)  # 16812 nodes: a node row of 134 KB
    nn = m.nnodes
    n, area, _ = orc.geometry(m)
    for r in (3, nn + 5):
        H, G, _ = ctx.assemble_laplace_rows(m, r, r + 1)
        s = m.xyz[r] if r < nn else m.xyz[m.con[r - nn]].mean(axis=0)
        full = np.zeros(nn)
        for e in range(m.nelem):
            if (r < nn and r in m.con[e]) or e == r - nn:
                continue  # singular pairs: G only
            out = orc.tri_lap_int(*m.xyz[m.con[e]], s, n[e], area[e])
            assert abs(G[0, e] - out[0]) < 1e-12 * abs(out[0])
            full[m.con[e]] += out[1:]
        free = -full.sum()
        if r < nn:
            full[r] += free
        else:
            full[m.con[r - nn]] += free / 3.0
        assert _close(H[0], full)
