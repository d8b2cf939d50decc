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


def test_long_blocks_take_the_launch_sequence():
    """COCG in FP32 above 16 columns: the shorter operator runs resident, the
    longer one by the launch sequence, which is faster there."""
    for (nodes, el), nq, resident in ((G.disk(25.0, 40), 33, True), (G.cylinder(25.0, 50.0, 20, 24), 16, True),
                                      (G.cylinder(25.0, 50.0, 20, 24), 33, False)):
        mesh = T.Mesh(data=(nodes, el))
        Q = G.ring(nq, 25.0) if nodes.shape[1] == 2 else G.ring(nq, 25.0, 5.0)
        mesh.SetQM(Q, Q[:1])
        f = _solver((mesh, T.Solution(*G.params(nodes, 7)), None))
        B = np.ascontiguousarray(mesh.Qvec(width=2.0).toarray())
        dB, dX = L.DeviceArray.from_host(B), L.DeviceArray(B.shape, B.dtype)
        f.CalcFieldsDevice(nq, dB.ptr, dX.ptr)
        assert f.LastResident() == (resident, 0)


@pytest.mark.parametrize("solver,mode,nq", [("BICGSTAB", "fp64_block", 4), ("BICGSTAB", "fp64", 3), ("COCG", "fp64_block", 7),
                                            ("COCG", "mixed", 8), ("BICGSTAB", "mixed", 8), ("COCG", "mixed", 3)])
def test_few_teams_on_many_rows(solver, mode, nq):
    """67,951 nodes, where a thread of a team with one column would hold more
    rows than it should: the columns share teams.  Against the launch sequence;
    strongly absorbing tissue, so that the fields follow the residual (20 x
    1e-10 as for the small meshes)."""
    nodes, el = G.disk(25.0, 150)
    mesh = T.Mesh(data=(nodes, el))
    mesh.SetQM(G.ring(8, 25.0), G.ring(1, 25.0))
    mua, mus, ref = G.params(nodes, 7)
    B = np.ascontiguousarray(mesh.Qvec(width=2.0).toarray()[:, :nq])
    X = []
    for sequence in (False, True):
        f = T.FwdSolver(mesh, solver, 1e-10)
        f.SetMode(mode)
        f.SetPrecon("DIAG")
        if sequence:
            f.SetGraphs(True)
        f.Allocate()
        f.Reset(T.Solution(100.0 * mua, mus, ref), 100.0 * 2 * np.pi * 1e-6)
        dB, dX = L.DeviceArray.from_host(B), L.DeviceArray(B.shape, B.dtype)
        assert all(s[3] for s in f.CalcFieldsDevice(nq, dB.ptr, dX.ptr))
        assert f.LastResident() == (not sequence, 0)
        X.append(dX.to_host())
    assert (np.linalg.norm(X[0] - X[1], axis=0) / np.linalg.norm(X[1], axis=0)).max() <= 20e-10


@pytest.mark.parametrize("kind,nq", [("disk", 1), ("disk", 17), ("disk", 64), ("ellipsoid", 6), ("ellipsoid", 33),
                                     ("ellipsoid", 57)])
def test_small_blocks_run_resident(kind, nq):
    """The blocks of test_resident_gpu.py run resident there, but for those
    whose three FP64 vectors a thread cannot hold (33 and more complex columns
    of 9,261 rows with BiCGSTAB), which it solves by the launch sequence twice."""
    if kind == "disk":
        (nodes, el), Q = G.disk(25.0, 22), G.ring(nq, 25.0)
    else:
        nodes, el = G.ellipsoid(80.0, 65.0, 90.0, 20)
        Q = G._ellipsoid_ring_points(80.0, 65.0, 90.0, [-45.0, -15.0, 15.0, 45.0], 16, 0.0)[np.arange(nq) * 64 // nq]
    mesh = T.Mesh(data=(nodes, el))
    mesh.SetQM(Q, Q[:1])
    B = np.ascontiguousarray(mesh.Qvec(width=2.0).toarray())
    for solver, mode in (("CG", "mixed"), ("CG", "fp64_block"), ("COCG", "mixed"), ("COCG", "fp64"),
                         ("BICGSTAB", "mixed"), ("BICGSTAB", "fp64_block")):
        f = T.FwdSolver(mesh, solver, 1e-10, complex=solver != "CG")
        f.SetMode(mode)
        f.SetPrecon("DIAG")
        f.Allocate()
        f.Reset(T.Solution(*G.params(nodes, 7)), 100.0 * 2 * np.pi * 1e-6 if f.complex else 0.0)
        b = np.ascontiguousarray(B if f.complex else B.real)
        dB, dX = L.DeviceArray.from_host(b), L.DeviceArray(b.shape, b.dtype)
        f.CalcFieldsDevice(nq, dB.ptr, dX.ptr)
        held = not (kind == "ellipsoid" and nq >= 33 and (solver, mode) == ("BICGSTAB", "fp64_block"))
        assert f.LastResident() == (held, 0), (solver, mode)
