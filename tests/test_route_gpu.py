"""Which solves run resident: those of a handle on which no detail of the
launch sequence has been named, and for which the autotuner did not find that
one faster."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

T = pytest.importorskip("toastpp_amd")
from toastpp_amd import _lib as L  # noqa: E402
from toastpp_amd import meshgen as G  # noqa: E402


@pytest.fixture(scope="module")
def disk():
    nodes, el = G.disk(25.0, 22)
    mesh = T.Mesh(data=(nodes, el))
    mesh.SetQM(G.ring(64, 25.0), G.ring(1, 25.0))
    return mesh, T.Solution(*G.params(nodes, 7)), np.ascontiguousarray(mesh.Qvec(width=2.0).toarray())


def _solver(disk):
    mesh, sol, B = disk
    f = T.FwdSolver(mesh, "COCG", 1e-10)
    f.SetPrecon("DIAG")
    f.Allocate()
    f.Reset(sol, 100.0 * 2 * np.pi * 1e-6)
    return f


def _resident(f, disk, nq):
    B = np.ascontiguousarray(disk[2][:, :nq])
    dB, dX = L.DeviceArray.from_host(B), L.DeviceArray(B.shape, B.dtype)
    f.CalcFieldsDevice(nq, dB.ptr, dX.ptr)
    f.CalcFieldsDevice(nq, dB.ptr, dX.ptr)
    return f.LastCounts()[0] == 1   # one launch


def test_tile_zero_takes_back_only_the_tile(disk):
    f = _solver(disk)
    assert _resident(f, disk, 8)
    f.SetTile(8)
    assert not _resident(f, disk, 8)
    f.SetTile(0)
    assert _resident(f, disk, 8)
    for name in (lambda f: f.SetGraphs(True), lambda f: f.SetSpmmVariant("rowblock"), lambda f: f.SetCompaction(2),
                 lambda f: f.SetRowsPerWave(4)):
        f = _solver(disk)
        name(f)
        assert not _resident(f, disk, 8)
        f.SetTile(16)
        f.SetTile(0)
        assert not _resident(f, disk, 8)


def test_autotune_decides_for_its_own_columns(disk):
    mesh, sol, B = disk
    f = _solver(disk)
    dB, dX = L.DeviceArray.from_host(B), L.DeviceArray(B.shape, B.dtype)
    f.Autotune(64, dB.ptr, dX.ptr)
    one = _resident(f, disk, 64)
    for nq in (1, 12, 33):
        assert _resident(f, disk, nq)
    f.SetTile(0)
    assert _resident(f, disk, 64) == one
    f.Autotune(64, dB.ptr, dX.ptr)   # decides anew
    f.SetLinSolver("COCG", 1e-10)
    assert _resident(f, disk, 64)
    # a named detail stays whatever the autotuner finds
    f.SetGraphs(True)
    f.Autotune(12, dB.ptr, dX.ptr, ld=64)
    assert not _resident(f, disk, 12)
