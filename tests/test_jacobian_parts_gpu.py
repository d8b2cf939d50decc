"""Nodal Jacobian where the operands of all nodes exceed what a mesh keeps
(1 GiB, 262,144 nodes up to 16 neighbours), so that they are made for a part of
the nodes at a time, the last one short; where they find no memory at all (the
per-node kernel); and on rows of more than 16 neighbours at the edges of the
rule that chooses between the kernels.  Against the oracle's element loops."""
import numpy as np
import pytest
from scipy.spatial import Delaunay

from oracle import oracle as O
from toastpp_amd import meshgen

pytestmark = pytest.mark.gpu

TMI = pytest.importorskip("toastpp_amd")
from toastpp_amd import _lib as L  # noqa: E402
from toastpp_amd.jacobian import jacobian  # noqa: E402


def _neighbours(n, el):
    i, j = np.divmod(np.unique(np.concatenate([el[:, a].astype(np.int64) * n + el[:, b] for a in range(4)
                                               for b in range(4)])), n)
    return np.bincount(i, minlength=n)


def _check(x, el, nq, nm, links, calls=2):
    x, el = np.ascontiguousarray(x, float), np.ascontiguousarray(el, np.int32)
    n, rng = len(x), np.random.default_rng(nq)
    lp = np.concatenate([[0], np.cumsum([len(v) for v in links])]).astype(np.int32)
    li = np.concatenate(links).astype(np.int32)
    nqm = int(lp[-1])
    gm = TMI.Mesh(data=(x, el))
    gm.SetQM(np.ones((nq, 3)), np.ones((nm, 3)), links=links)
    f = rng.standard_normal((n, nq)) + 1j * rng.standard_normal((n, nq))
    g = rng.standard_normal((n, nm)) + 1j * rng.standard_normal((n, nm))
    proj = rng.standard_normal(nqm) + 1j * rng.standard_normal(nqm)
    ref = O.jacobian_nodal(O.Mesh(nodes=x, elems=el), f.T, g.T, lp, li, proj, logscale=True)
    for _ in range(calls):
        J = jacobian(gm, None, f, g, proj, scale="log")
        # sums of a few hundred products in FP64 (test_jacobian_tiles_gpu.py)
        for c in (slice(0, n), slice(n, 2 * n)):
            big = np.maximum(np.abs(ref[:nqm, c]), np.abs(ref[nqm:, c])).max(1)
            assert np.all(np.abs(J[:nqm, c] - ref[:nqm, c]).max(1) <= 1e-12 * big)
            assert np.all(np.abs(J[nqm:, c] - ref[nqm:, c]).max(1) <= 1e-12 * big)


def test_parts_up_to_16_neighbours():
    x, el = meshgen.ellipsoid(80.0, 65.0, 90.0, 65)
    d = _neighbours(len(x), el)
    assert len(x) > 262144 and d.max() <= 16
    _check(x, el, 2, 2, [[0, 1], [1]])


def test_operands_without_memory():
    x, el = meshgen.cylinder(25.0, 50.0, 5, 6)
    L.call("tmi_test_alloc_limit", float(len(x) * 4096 - 1))
    try:
        _check(x, el, 5, 4, [[q % 4] for q in range(5)])
    finally:
        L.call("tmi_test_alloc_limit", 0.0)
    _check(x, el, 5, 4, [[q % 4] for q in range(5)])


def _cloud(points, most):
    """triangulated random points, without the elements of nodes of more than
    `most` neighbours"""
    x = np.random.default_rng(3).random((points, 3)) * 50.0
    el = Delaunay(x).simplices
    p = x[el]
    v = np.linalg.det(p[:, 1:] - p[:, :1])
    el = np.where((v < 0)[:, None], el[:, [1, 0, 2, 3]], el)[np.abs(v) > 1e-3]
    el = el[~(_neighbours(points, el) > most)[el].any(1)]
    used = np.unique(el)
    return x[used], np.searchsorted(used, el)


# one tile (192 pairs and fewer), four (768 links and fewer), more
@pytest.mark.parametrize("nq,nm,per", [(12, 16, 16), (16, 12, 1), (13, 14, 14), (16, 16, 3), (32, 32, 24), (32, 32, 23),
                                       (17, 17, 17), (48, 16, 12)])
def test_rows_of_more_than_16_neighbours(nq, nm, per):
    x, el = _cloud(1500, 30)
    d = _neighbours(len(x), el)
    assert 24 <= d.max() <= 32 and d.mean() >= 15
    _check(x, el, nq, nm, [sorted((q + j) % nm for j in range(per)) for q in range(nq)], 1)


def test_tiles_without_links():
    x, el = meshgen.cylinder(25.0, 50.0, 5, 6)
    _check(x, el, 32, 32, [[q] for q in range(32)])
