"""Copies of the operators for resident solves: one per number of workgroups,
bounded on a handle that solves blocks of many sizes, and back with the same
results after they were given back."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

T = pytest.importorskip("toastpp_amd")
from toastpp_amd import _lib as L  # noqa: E402
from toastpp_amd import meshgen as G  # noqa: E402


def test_copies_are_bounded():
    nodes, el = G.ellipsoid(80.0, 65.0, 90.0, 62)   # 250,047 nodes: about 95 MB of copies a block size
    mesh = T.Mesh(data=(nodes, el))
    Q = G._ellipsoid_ring_points(80.0, 65.0, 90.0, [-45.0, -15.0, 15.0, 45.0], 1, 0.0)
    mesh.SetQM(Q, Q[:1])
    f = T.FwdSolver(mesh, "COCG", 1e-10)
    f.SetPrecon("DIAG")
    f.Allocate()
    omega = 100.0 * 2 * np.pi * 1e-6
    f.Reset(T.Solution(*G.params(nodes, 7)), omega)
    B = np.ascontiguousarray(mesh.Qvec(width=2.0).toarray())

    def fields(nq, mf):
        b = np.ascontiguousarray(B[:, :nq])
        dB, dX = L.DeviceArray.from_host(b), L.DeviceArray(b.shape, b.dtype)
        if mf:
            f.CalcFieldsFreqsDevice(nq, dB.ptr, dX.ptr, np.full(nq, omega))
        else:
            f.CalcFieldsDevice(nq, dB.ptr, dX.ptr)
        assert f.LastResident() == (True, 0)
        return dX.to_host(), f.OperatorBytes()

    assert f.OperatorBytes() == 0
    seen, most = [], 0.0
    for nq, mf in ((1, False), (2, False), (1, True), (2, True), (1, False), (2, True)):
        X, held = fields(nq, mf)
        seen.append((nq, mf, X))
        most = max(most, held)
    assert 150e6 < most <= 256 * 2 ** 20
    assert np.array_equal(seen[0][2], seen[4][2])   # given back and made again
    assert np.array_equal(seen[3][2], seen[5][2])
