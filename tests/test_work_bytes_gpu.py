"""WorkBytes bounds what a solve's workspace holds afterwards, on the resident
and on the launch-sequence route and where the first gives up; a server whose
budget holds only the launch sequence's workspace admits the request on it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

T = pytest.importorskip("toastpp_amd")
from toastpp_amd import _lib as L  # noqa: E402
from toastpp_amd import meshgen as G  # noqa: E402
from toastpp_amd.serve import Server  # noqa: E402


@pytest.fixture(scope="module")
def cyl():
    nodes, el = G.cylinder(25.0, 50.0, 12, 13)   # 6,566 nodes
    mesh = T.Mesh(data=(nodes, el))
    Q = np.vstack([G.ring(32, 25.0, z) for z in (-12.5, 12.5)])
    mesh.SetQM(Q, Q[:1])
    return mesh, T.Solution(*G.params(nodes, 7)), np.ascontiguousarray(mesh.Qvec(width=2.0).toarray())


def _solver(cyl, solver, mode, sequence=False):
    f = T.FwdSolver(cyl[0], solver, 1e-10, complex=solver != "CG")
    f.SetMode(mode)
    f.SetPrecon("DIAG")
    if sequence:
        f.SetGraphs(True)
    f.Allocate()
    f.Reset(cyl[1], 100.0 * 2 * np.pi * 1e-6 if f.complex else 0.0)
    return f


def _serve(srv, f, cyl, nq):
    B = np.ascontiguousarray(cyl[2] if f.complex else cyl[2].real)
    dB, dX = L.DeviceArray.from_host(B), L.DeviceArray.from_host(np.zeros_like(B))
    st, _, status = srv.wait(srv.submit(f, nq, dB.ptr, dX.ptr, 64))
    assert status == L.TMI_OK and all(s[3] for s in st)
    return srv.counts()[2], dX.to_host()[:, :nq]   # bytes held between requests


@pytest.mark.parametrize("solver,mode", [("BICGSTAB", "fp64"), ("COCG", "fp64"), ("CG", "fp64"), ("BICGSTAB", "fp64_block"),
                                         ("BICGSTAB", "mixed"), ("COCG", "mixed"), ("CG", "mixed")])
@pytest.mark.parametrize("nq", [1, 10, 33])
def test_held_bytes_within_bound(cyl, solver, mode, nq):
    for test in (0, 1, 2):
        f = _solver(cyl, solver, mode)
        L.call("tmi_test_resident", f._h, test)
        bound = f.WorkBytes(nq)
        srv = Server(slots=1, hbm_budget_gib=4.0)
        held, _ = _serve(srv, f, cyl, nq)
        srv.close()
        assert 0 < held <= bound, (test, held, bound)
        assert f.LastResident()[1] == (test != 0)


def test_budget_of_the_launch_sequence(cyl):
    f, seq = _solver(cyl, "BICGSTAB", "fp64"), _solver(cyl, "BICGSTAB", "fp64", True)
    small, big = seq.WorkBytes(33), f.WorkBytes(33)
    assert small < 0.5 * big
    srv = Server(slots=1, hbm_budget_gib=1.01 * small / 2.0 ** 30)
    held, X = _serve(srv, f, cyl, 33)
    assert held <= 1.01 * small
    srv.close()
    srv = Server(slots=1, hbm_budget_gib=0.9 * small / 2.0 ** 30)
    with pytest.raises(L.TmiError):
        _serve(srv, f, cyl, 33)
    srv.close()
    srv = Server(slots=1, hbm_budget_gib=4.0)
    _, Xs = _serve(srv, seq, cyl, 33)
    srv.close()
    assert np.array_equal(X, Xs)
