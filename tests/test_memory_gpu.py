"""Solves where device memory runs out: the failed call reports it, and the
next one, with memory again, allocates what the first could not."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

T = pytest.importorskip("toastpp_amd")
from toastpp_amd import _lib as L  # noqa: E402
from toastpp_amd import meshgen as G  # noqa: E402


@pytest.fixture
def limit():
    yield lambda b: L.call("tmi_test_alloc_limit", float(b))
    L.call("tmi_test_alloc_limit", 0.0)


def _prepared(solver, sequence):
    nodes, el = G.disk(25.0, 22)   # 1,519 nodes
    mesh = T.Mesh(data=(nodes, el))
    mesh.SetQM(G.ring(16, 25.0), G.ring(1, 25.0))
    f = T.FwdSolver(mesh, solver, 1e-10)
    f.SetPrecon("DIAG")
    if sequence:
        f.SetGraphs(True)
    f.Allocate()
    f.Reset(T.Solution(*G.params(nodes, 7)), 100.0 * 2 * np.pi * 1e-6)
    return mesh, f, np.ascontiguousarray(mesh.Qvec(width=2.0).toarray())


def _fields(f, B):
    dB, dX = L.DeviceArray.from_host(B), L.DeviceArray(B.shape, B.dtype)
    f.CalcFieldsDevice(B.shape[1], dB.ptr, dX.ptr)
    return dX.to_host()


@pytest.mark.parametrize("solver", ["COCG", "BICGSTAB", "GMRES"])
def test_solve_after_out_of_memory(limit, solver):
    mesh, f, B = _prepared(solver, True)
    ref = _fields(_prepared(solver, True)[1], B)
    dB, dX = L.DeviceArray.from_host(B), L.DeviceArray(B.shape, B.dtype)
    # the solver's own vectors of all columns do not fit, smaller buffers do
    limit(1519 * 16 * 8 - 1)
    for _ in range(2):
        with pytest.raises(L.TmiError) as e:
            f.CalcFieldsDevice(16, dB.ptr, dX.ptr)
        assert e.value.code == L.TMI_ERR_OOM
    limit(0)
    assert np.array_equal(_fields(f, B), ref)


@pytest.mark.parametrize("limit_bytes", [20000, 1519 * 16 * 8 - 1])
def test_resident_solve_without_memory(limit, limit_bytes):
    """Where the resident layout (20 KB: less than it takes) or the vectors of
    all columns find no memory, the launch sequence solves one right-hand side
    after the other."""
    mesh, f, B = _prepared("BICGSTAB", False)
    f.SetMode("fp64")
    f.SetTile(1)
    ref = _fields(f, B)   # the launch sequence has its workspace from here on
    f.SetTile(0)
    dB, dX = L.DeviceArray.from_host(B), L.DeviceArray(B.shape, B.dtype)
    limit(limit_bytes)
    f.CalcFieldsDevice(16, dB.ptr, dX.ptr)
    assert f.LastResident() == (False, 0) and np.array_equal(dX.to_host(), ref)
    limit(0)
    f.CalcFieldsDevice(16, dB.ptr, dX.ptr)
    assert f.LastResident() == (True, 0)
