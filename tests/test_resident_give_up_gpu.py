"""Resident launches that the device refuses, or that end their bounded waits
early (the abort word is set from the start, so every workgroup exits
normally): the launch sequence solves the block, from whatever the launch left
in the fields, and the handle stays with it until the next Allocate."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

T = pytest.importorskip("toastpp_amd")
from toastpp_amd import _lib as L  # noqa: E402
from toastpp_amd import meshgen as G  # noqa: E402

TOL = 1e-10
REFUSED, ABORTED = 1, 2


@pytest.fixture(scope="module", params=["disk217", "ell9k"])
def case(request):
    # one workgroup per column (nothing waits); teams of 4 to 256 ranks
    if request.param == "disk217":
        (nodes, el), Q = G.disk(25.0, 8), G.ring(64, 25.0)
    else:
        nodes, el = G.ellipsoid(80.0, 65.0, 90.0, 20)
        Q = G._ellipsoid_ring_points(80.0, 65.0, 90.0, [-45.0, -15.0, 15.0, 45.0], 16, 0.0)
    mesh = T.Mesh(data=(nodes, el))
    mesh.SetQM(Q, Q[:1])
    return mesh, T.Solution(*G.params(nodes, 7)), np.ascontiguousarray(mesh.Qvec(width=2.0).toarray())


def _solver(case, solver, mode):
    f = T.FwdSolver(case[0], solver, TOL, complex=solver != "CG")
    f.SetMode(mode)
    f.SetPrecon("DIAG")
    f.Allocate()
    _reset(f, case)
    return f


def _reset(f, case):
    f.Reset(case[1], 100.0 * 2 * np.pi * 1e-6 if f.complex else 0.0)


def _fields(f, case, nq):
    B = case[2][:, :nq]
    B = np.ascontiguousarray(B if f.complex else B.real)
    dB, dX = L.DeviceArray.from_host(B), L.DeviceArray(B.shape, B.dtype)
    st = f.CalcFieldsDevice(nq, dB.ptr, dX.ptr)
    assert all(s[3] for s in st)
    return dX.to_host()


@pytest.mark.parametrize("what", [REFUSED, ABORTED])
@pytest.mark.parametrize("solver,mode,nq", [("COCG", "mixed", 1), ("COCG", "mixed", 57), ("BICGSTAB", "mixed", 24),
                                            ("CG", "mixed", 5), ("COCG", "fp64_block", 16), ("BICGSTAB", "fp64", 3)])
def test_launch_sequence_takes_over(case, what, solver, mode, nq):
    seq = _solver(case, solver, mode)
    seq.SetGraphs(True)
    ref = _fields(seq, case, nq)
    assert seq.LastResident() == (False, 0)
    f = _solver(case, solver, mode)
    L.call("tmi_test_resident", f._h, what)
    X = _fields(f, case, nq)
    assert f.LastResident() == (False, 1)
    if what == REFUSED:
        assert np.array_equal(X, ref)   # nothing was launched
    else:   # the same residual from another start (the bound of test_resident_gpu.py)
        assert (np.linalg.norm(X - ref, axis=0) / np.linalg.norm(ref, axis=0)).max() <= 20 * TOL
    # remembered: no further launch
    L.call("tmi_test_resident", f._h, 0)
    assert np.array_equal(_fields(f, case, nq), ref)
    assert f.LastResident() == (False, 1)
    f.Allocate()
    _reset(f, case)
    _fields(f, case, nq)
    assert f.LastResident() == (True, 0)
