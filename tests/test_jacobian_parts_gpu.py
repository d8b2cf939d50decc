"""Nodal Jacobian where the operands of all nodes exceed what a mesh keeps
(1 GiB: 262,144 nodes up to 16 neighbours, 65,536 up to 32), so that they are
made for a part of the nodes at a time, the last one short; and where they find
no memory at all (the per-node kernel).  Against the oracle's element loops."""
import numpy as np
import pytest

from oracle import oracle as O
from toastpp_amd import meshgen

pytestmark = pytest.mark.gpu

TMI = pytest.importorskip("toastpp_amd")
from toastpp_amd import _lib as L  # noqa: E402
from toastpp_amd.jacobian import jacobian  # noqa: E402


def _lattice(k):
    """k x k x k lattice points, each cube in five tetrahedra, mirrored from
    cube to cube: rows of 19 and 7 nodes inside"""
    c = np.stack(np.meshgrid(*[np.arange(k - 1)] * 3, indexing="ij"), -1).reshape(-1, 3)
    odd = c.sum(1) % 2
    five = np.array([[0, 3, 5, 6], [1, 0, 3, 5], [2, 3, 0, 6], [4, 0, 5, 6], [7, 3, 5, 6]])   # corners x + 2 y + 4 z
    corner = np.stack([five & 1, five >> 1 & 1, five >> 2], -1)[None]
    corner = np.repeat(corner, len(c), 0)
    corner[odd == 1, :, :, 0] ^= 1   # mirrored in x
    at = c[:, None, None, :] + corner
    el = ((at[..., 0] * k + at[..., 1]) * k + at[..., 2]).reshape(-1, 4)
    x = np.stack(np.meshgrid(*[np.arange(k)] * 3, indexing="ij"), -1).reshape(-1, 3).astype(float)
    p = x[el]
    v = np.linalg.det(p[:, 1:] - p[:, :1])
    assert np.all(np.abs(v) > 0.5)
    return x, np.where((v < 0)[:, None], el[:, [1, 0, 2, 3]], el)


def _neighbours(n, el):
    i, j = np.divmod(np.unique(np.concatenate([el[:, a].astype(np.int64) * n + el[:, b] for a in range(4)
                                               for b in range(4)])), n)
    return np.bincount(i, minlength=n)


def _check(x, el, nq, nm, links):
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
    for _ in range(2):
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


def test_parts_up_to_32_neighbours():
    x, el = _lattice(41)
    d = _neighbours(len(x), el)
    assert len(x) > 65536 and 16 < d.max() <= 32 and d.mean() >= 12
    _check(x, el, 16, 16, [[q % 3] for q in range(16)])


def test_operands_without_memory():
    x, el = meshgen.cylinder(25.0, 50.0, 5, 6)
    L.call("tmi_test_alloc_limit", float(len(x) * 4096 - 1))
    try:
        _check(x, el, 5, 4, [[q % 4] for q in range(5)])
    finally:
        L.call("tmi_test_alloc_limit", 0.0)
    _check(x, el, 5, 4, [[q % 4] for q in range(5)])
