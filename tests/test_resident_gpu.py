"""Resident solves (one cooperative kernel per block) against the launch
sequence and the oracle: real and complex, PCG / COCG / BiCGSTAB, mixed and
FP64, column counts that fill, overfill and undercut a team, systems on one
workgroup and on teams of every width, several frequencies, a zero right-hand
side and the iteration cap.  Both paths stop at the same residual, so their
fields differ by at most cond-free multiples of the tolerance: 20 x 1e-10 on
these meshes (the oracle check of the launch sequence uses 1e-8)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

T = pytest.importorskip("toastpp_amd")
from toastpp_amd import _lib as L  # noqa: E402
from toastpp_amd import meshgen as G  # noqa: E402

TOL = 1e-10


def _setup(kind):
    if kind == "disk217":        # one workgroup per column
        nodes, el = G.disk(25.0, 8)
    elif kind == "disk1519":     # just past the one-workgroup systems
        nodes, el = G.disk(25.0, 22)
    elif kind == "cyl3k":
        nodes, el = G.cylinder(25.0, 50.0, 8, 13)
    else:                        # ellipsoid, 9261 nodes
        nodes, el = G.ellipsoid(80.0, 65.0, 90.0, 20)
    dim = nodes.shape[1]
    Q = G.ring(64, 25.0) if dim == 2 else np.vstack([G.ring(32, 25.0, z) for z in (-12.5, 12.5)])
    if kind == "ell9k":
        Q = G._ellipsoid_ring_points(80.0, 65.0, 90.0, [-45.0, -15.0, 15.0, 45.0], 16, 0.0)
    mesh = T.Mesh(data=(nodes, el))
    mesh.SetQM(Q, Q[:1])
    return mesh, T.Solution(*G.params(nodes, 7)), np.ascontiguousarray(mesh.Qvec(width=2.0).toarray())


@pytest.fixture(scope="module")
def setups():
    cache = {}

    def get(kind):
        if kind not in cache:
            cache[kind] = _setup(kind)
        return cache[kind]
    return get


def _solve(mesh, sol, B, solver, mode, precon, sequence, omegas=None, maxit=0):
    cplx = solver != "CG"
    f = T.FwdSolver(mesh, solver, TOL, complex=cplx)
    f.SetMode(mode)
    f.SetPrecon(precon)
    f.SetLinSolverMaxit(maxit)
    if sequence:
        f.SetGraphs(True)
    f.Allocate()
    f.Reset(sol, 100.0 * 2 * np.pi * 1e-6 if cplx else 0.0)
    Bc = np.ascontiguousarray(B if cplx else B.real)
    dB = L.DeviceArray.from_host(Bc)
    dX = L.DeviceArray(Bc.shape, Bc.dtype)
    if omegas is None:
        st = f.CalcFieldsDevice(Bc.shape[1], dB.ptr, dX.ptr)
    else:
        st = f.CalcFieldsFreqsDevice(Bc.shape[1], dB.ptr, dX.ptr, omegas)
    return dX.to_host(), st, f.LastCounts()


def _compare(a, b):  # largest relative L2 difference of a column
    return (np.linalg.norm(a - b, axis=0) / np.linalg.norm(b, axis=0)).max()


@pytest.mark.parametrize("kind,nq", [("disk217", 1), ("disk217", 5), ("disk217", 64), ("disk1519", 3), ("disk1519", 17),
                                     ("disk1519", 64), ("cyl3k", 1), ("cyl3k", 2), ("cyl3k", 40), ("ell9k", 6),
                                     ("ell9k", 33), ("ell9k", 57)])
@pytest.mark.parametrize("solver,mode,precon", [("CG", "mixed", "DIAG"), ("CG", "fp64_block", "NONE"),
                                                ("COCG", "mixed", "DIAG"), ("COCG", "fp64", "DIAG"),
                                                ("BICGSTAB", "mixed", "DIAG"), ("BICGSTAB", "mixed", "NONE"),
                                                ("BICGSTAB", "fp64_block", "DIAG")])
def test_resident_matches_launch_sequence(setups, kind, nq, solver, mode, precon):
    mesh, sol, B = setups(kind)
    cols = np.arange(nq) * 64 // nq
    X, st, counts = _solve(mesh, sol, B[:, cols], solver, mode, precon, False)
    Xs, sts, _ = _solve(mesh, sol, B[:, cols], solver, mode, precon, True)
    # one kernel and the operator gathers; again in FP64 for a column that
    # the FP32 iteration leaves above the tolerance (on either path)
    if B.shape[0] * nq * 16 <= 4e6:
        assert counts[1] == 0 and counts[0] <= 6
    assert all(s[3] for s in st) and all(s[3] for s in sts)
    assert _compare(X, Xs) <= 20 * TOL
    X2, st2, _ = _solve(mesh, sol, B[:, cols], solver, mode, precon, False)
    assert np.array_equal(X, X2) and st == st2   # fixed-order sums


@pytest.mark.parametrize("kind,nq,mode", [("disk217", 9, "mixed"), ("cyl3k", 24, "mixed"), ("cyl3k", 10, "fp64_block")])
def test_resident_frequencies(setups, kind, nq, mode):
    mesh, sol, B = setups(kind)
    cols = np.arange(nq) * 64 // nq
    om = np.array([0.0, 50.0, 100.0, 200.0])[np.arange(nq) % 4] * 2 * np.pi * 1e-6
    X, st, counts = _solve(mesh, sol, B[:, cols], "COCG", mode, "DIAG", False, omegas=om)
    Xs, _, _ = _solve(mesh, sol, B[:, cols], "COCG", mode, "DIAG", True, omegas=om)
    assert counts[1] == 0 and all(s[3] for s in st)
    assert _compare(X, Xs) <= 20 * TOL


def test_resident_zero_column_and_cap(setups):
    mesh, sol, B = setups("cyl3k")
    Bz = B[:, [0, 20, 40]].copy()
    Bz[:, 1] = 0.0
    for solver in ("COCG", "BICGSTAB", "CG"):
        X, st, _ = _solve(mesh, sol, Bz, solver, "mixed", "DIAG", False)
        assert np.all(X[:, 1] == 0) and st[1][0] == 0 and st[1][3]
        assert st[0][3] and st[2][3]
        # an iteration cap in the FP64 mode: the true residual is reported, as by the launch sequence
        X, st, _ = _solve(mesh, sol, B[:, :4], solver, "fp64_block", "DIAG", False, maxit=16)
        Xs, sts, _ = _solve(mesh, sol, B[:, :4], solver, "fp64_block", "DIAG", True, maxit=16)
        for a, b in zip(st, sts):
            assert a[0] == b[0] == 16 and not a[3]
            assert abs(a[2] - b[2]) <= 1e-13   # rounding of b - A x, relative to ||b||
        assert _compare(X, Xs) <= 1e-9   # the same iterates up to the order of the sums


def test_resident_bicgstab_idle_columns(setups):
    """A column that has met its recursive test waits for the next residual
    replacement and may run on after it.  What the other columns of its team
    do meanwhile must not matter: beside columns that need twice its
    iterations it takes the same iterates, bit for bit, as beside others that
    stop when it does (sources in a strongly absorbing half of the mesh, which
    meet the FP32 test after about 20 iterations and fail the FP64 one)."""
    mesh, _, _ = setups("ell9k")
    nodes, _ = G.ellipsoid(80.0, 65.0, 90.0, 20)
    mua, mus, ref = G.params(nodes, 7)
    x = nodes[:, 0]
    sol = T.Solution(np.where(x > 0, 1e4 * mua, mua), mus, ref)
    fast, slow = np.where(x > 24.0)[0], np.where(x < -24.0)[0]

    def rhs(centres):
        d2 = ((nodes[:, None, :] - nodes[None, centres, :]) ** 2).sum(2)
        return np.ascontiguousarray(np.exp(-d2 / 8.0).astype(complex))
    f = rhs(fast[np.arange(64) * len(fast) // 64])
    mixed = rhs(slow[np.arange(64) * len(slow) // 64])
    mixed[:, ::2] = f[:, ::2]
    Xf, stf, _ = _solve(mesh, sol, f, "BICGSTAB", "mixed", "DIAG", False)
    Xm, stm, counts = _solve(mesh, sol, mixed, "BICGSTAB", "mixed", "DIAG", False)
    assert counts[0] <= 6 and counts[1] == 0   # resident
    assert max(s[0] for s in stf) + 8 < max(s[0] for s in stm[1::2])
    assert [s[0] for s in stf[::2]] == [s[0] for s in stm[::2]]
    assert np.array_equal(Xf[:, ::2], Xm[:, ::2])
