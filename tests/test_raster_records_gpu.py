"""Raster Jacobian, its CW form and the data gradient where their tiles can go
wrong: voxel counts around 64, column counts that are no power of two and above
64, source counts around the gradient's eight waves, grids a few points wide
(differences of one side, or none), against the oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from toastpp_amd import meshgen

pytestmark = pytest.mark.gpu

TMI = pytest.importorskip("toastpp_amd")
from toastpp_amd.jacobian import jacobian_cw  # noqa: E402


@pytest.mark.parametrize("dim,grid,nq,nm", [(2, (9, 9), 1, 1), (2, (10, 11), 5, 2), (2, (3, 40), 33, 34),
                                            (3, (8, 8, 8), 3, 9), (3, (7, 9, 5), 17, 8), (3, (3, 12, 12), 40, 33)])
def test_raster_tiles(dim, grid, nq, nm):
    x, el = meshgen.disk(25.0, 7) if dim == 2 else meshgen.cylinder(25.0, 50.0, 4, 4)
    x, el = np.ascontiguousarray(x, float), np.ascontiguousarray(el, np.int32)
    om, gm = O.Mesh(nodes=x, elems=el), TMI.Mesh(data=(x, el))
    orr, gr = O.Raster(om, list(grid)), TMI.Raster(gm, np.array(grid))
    rng = np.random.default_rng(nq)
    links = [sorted(rng.choice(nm, rng.integers(1, nm + 1), replace=False).tolist()) for _ in range(nq)]
    gm.SetQM(np.ones((nq, dim)), np.ones((nm, dim)), links=links)
    lp = np.concatenate([[0], np.cumsum([len(v) for v in links])]).astype(np.int32)
    li = np.concatenate(links).astype(np.int32)
    n, nqm, s = len(x), int(lp[-1]), gr.SLen()
    assert s == orr.slen
    f = rng.standard_normal((n, nq)) + 1j * rng.standard_normal((n, nq))
    a = rng.standard_normal((n, max(nq, nm))) + 1j * rng.standard_normal((n, max(nq, nm)))
    proj = 1.0 + rng.random(nqm) + 1j * rng.standard_normal(nqm)
    # the same products and differences on both sides, a few tens of
    # roundings of 1.1e-16 each: 1e-13 of the largest entry
    J = gm.Jacobian(gr, f, a[:, :nm], proj)
    ref = O.jacobian_grid(orr, f.T, a[:, :nm].T, lp, li, proj, logscale=True)
    assert np.abs(J - ref).max() <= 1e-13 * np.abs(ref).max()
    p = proj.real
    Jm, Jk = jacobian_cw(gm, gr, f.real, a[:, :nm].real, p, scale="log", kappa=True)
    Om, Ok = O.jacobian_grid_cw(orr, f.real.T, a[:, :nm].real.T, lp, li, p, logscale=True)
    assert np.abs(Jm - Om).max() <= 1e-13 * np.abs(Om).max()
    assert np.abs(Jk - Ok).max() <= 1e-13 * np.abs(Ok).max()
    g0 = rng.standard_normal(2 * s)
    gg, go = gr.DataGradient(f, a[:, :nq], g0), O.data_gradient(orr, f.T, a[:, :nq].T, g0)
    assert np.abs(gg - go).max() <= 1e-13 * max(np.abs(go - g0).max(), np.abs(g0).max())
