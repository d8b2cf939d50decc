"""Performance cases: the work a program has this framework do.

Every case calls the public entry points (toastpp_amd.FwdSolver, Mesh, Raster
and the *_device functions of the C-ABI) on generated meshes of the package's
own workloads (toastpp_amd.meshgen): ring-meshed disks (Tri3), extruded
cylinders and mapped ellipsoids (Tet4), 0-200 MHz, Gaussian boundary sources
and detectors, blob maps of mua and mus.  prepare() makes what such a program
holds before the call (mesh, QM description, assembled solver, device
buffers), run() one pass, exact() the same result in FP64 by plain torch.
"""
import ctypes as C
import functools
import math

import numpy as np
import torch

import toastpp_amd as T
from toastpp_amd import _lib as L
from toastpp_amd import meshgen as G

DEV = "cuda"

# ranges of the drawn cases: disk rings, cylinder rings, ellipsoid divisions
DISK = (16, 80)
CYL = (10, 30)
ELL = (18, 52)


def listed():
    return [
        # forward model of a 2D slice, continuous wave: the smallest call, a few
        # thousand unknowns, where launches and latency count
        dict(name="fields_disk3k_cw_16", kind="fields", mesh="disk", k=32, layers=0, freq=0.0, nq=16, solver="CG",
             mode="mixed"),
        # a dense 2D slice at 100 MHz as a serving request asks for it
        dict(name="fields_disk19k_100MHz_24", kind="fields", mesh="disk", k=80, layers=0, freq=100.0, nq=24,
             solver="COCG", mode="mixed"),
        # the reference's own method on a laboratory phantom, 32 sources in two rings
        dict(name="fields_cyl31k_bicgstab_32", kind="fields", mesh="cylinder", k=20, layers=24, freq=100.0, nq=32,
             solver="BICGSTAB", mode="mixed"),
        # a whole head-sized forward problem: 250k nodes, 64 sources (the largest solve)
        dict(name="fields_ell250k_cocg_64", kind="fields", mesh="ellipsoid", k=62, layers=0, freq=100.0, nq=64,
             solver="COCG", mode="mixed"),
        # all arithmetic in FP64, where a user wants no single precision at all
        dict(name="fields_cyl31k_fp64block_16", kind="fields", mesh="cylinder", k=20, layers=24, freq=100.0, nq=16,
             solver="COCG", mode="fp64_block"),
        # the plain FP64 path of the reference, one right-hand side at a time
        dict(name="fields_cyl31k_fp64_2", kind="fields", mesh="cylinder", k=20, layers=24, freq=100.0, nq=2,
             solver="BICGSTAB", mode="fp64"),
        # multi-frequency measurement: 12 sources at 0, 50, 100 and 200 MHz in one block
        dict(name="freqs_ell80k_48", kind="freqs", mesh="ellipsoid", k=42, layers=0, freq=200.0, nq=48,
             solver="COCG", mode="mixed"),
        # one evaluation of the forward data for new optical parameters, as every
        # step of a reconstruction's line search makes it: assembly, fields, projections
        dict(name="forward_cyl31k_8", kind="forward", mesh="cylinder", k=20, layers=24, freq=100.0, nq=8, nm=8,
             solver="COCG", mode="mixed"),
        # nodal Jacobian of a reconstruction step, 32 x 32 source-detector pairs
        dict(name="jac_nodal_cyl103k_32x32", kind="jac_nodal", mesh="cylinder", k=30, layers=36, nq=32, nm=32,
             links=1.0),
        # the same on the voxel basis of the image
        dict(name="jac_raster64_cyl103k_32x32", kind="jac_raster", mesh="cylinder", k=30, layers=36, nq=32, nm=32,
             links=1.0, grid=64),
        # gradient of the data misfit on the voxel basis (gradient-based reconstruction)
        dict(name="gradient_raster48_cyl31k_32", kind="gradient", mesh="cylinder", k=20, layers=24, nq=32, nm=32,
             links=1.0, grid=48),
        # a 2D Jacobian end to end from optical parameters, host arrays in and out
        dict(name="optical_disk3k_16x16", kind="optical", mesh="disk", k=32, layers=0, freq=100.0, nq=16, nm=16),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["fields", "fields", "fields", "freqs", "forward", "jac_nodal", "jac_nodal", "jac_raster",
                       "gradient", "optical"])
    mesh = rng.choice(["disk", "cylinder", "ellipsoid"])
    if kind == "optical":
        mesh = "disk"
    if kind == "forward" and mesh == "ellipsoid":
        mesh = "cylinder"
    k = {"disk": _logint(rng, *DISK), "cylinder": _logint(rng, *CYL), "ellipsoid": _logint(rng, *ELL)}[mesh]
    c = dict(kind=kind, mesh=mesh, k=k, layers=max(4, k + rng.randint(-4, 6)) if mesh == "cylinder" else 0)
    if kind in ("fields", "freqs", "forward", "optical"):
        c["freq"] = float(rng.choice([50, 100, 150, 200]))
    if kind == "fields":
        c["mode"] = rng.choice(["mixed", "mixed", "mixed", "fp64_block", "fp64"])
        c["solver"] = rng.choice(["COCG", "COCG", "BICGSTAB", "CG"])
        if c["solver"] == "CG":
            c["freq"] = 0.0
        c["nq"] = _logint(rng, 1, {"fp64": 3, "fp64_block": 32, "mixed": 64}[c["mode"]])
    elif kind == "freqs":
        c.update(solver="COCG", mode="mixed", nq=_logint(rng, 4, 64))
    elif kind == "forward":
        c.update(solver=rng.choice(["COCG", "BICGSTAB"]), mode="mixed", nq=_logint(rng, 2, 32), nm=_logint(rng, 2, 32))
    elif kind == "optical":
        c["k"] = _logint(rng, 16, 40)
        c.update(nq=_logint(rng, 2, 16), nm=_logint(rng, 2, 16))
    else:
        c.update(nq=_logint(rng, 2, 32), nm=_logint(rng, 2, 32), links=rng.choice([1.0, 0.5]))
        if mesh == "ellipsoid" and kind == "jac_nodal":
            c["k"] = min(k, 42)
        if kind != "jac_nodal":
            c["grid"] = _logint(rng, 12, 60)
    return c


# ------------------------------------------------------------------ inputs
@functools.lru_cache(maxsize=6)
def _geometry(mesh, k, layers):
    if mesh == "disk":
        return G.disk(25.0, k)
    if mesh == "cylinder":
        return G.cylinder(25.0, 50.0, k, layers)
    return G.ellipsoid(80.0, 65.0, 90.0, k)


def _ring_points(mesh, count, turn):
    """count points on the surface, on one ring (disk), two (cylinder) or four (ellipsoid), from the angle turn on"""
    z = {"disk": [None], "cylinder": [-12.5, 12.5], "ellipsoid": [-45.0, -15.0, 15.0, 45.0]}[mesh]
    a, b = (80.0, 65.0) if mesh == "ellipsoid" else (25.0, 25.0)
    out = []
    for i in range(count):
        zz = z[i % len(z)]
        per = (count + len(z) - 1) // len(z)
        th = 2 * math.pi * (i // len(z)) / per + turn
        s = math.sqrt(1 - (zz / 90.0) ** 2) if mesh == "ellipsoid" else 1.0
        p = [a * s * math.cos(th), b * s * math.sin(th)]
        out.append(p if zz is None else p + [zz])
    return np.array(out)


class _Inputs:
    """what the seed decides: optical maps, source and detector positions"""

    def __init__(self, case, seed):
        self.nodes, self.el = _geometry(case["mesh"], case["k"], case["layers"])
        self.n, self.dim = self.nodes.shape
        self.mua, self.mus, self.ref = G.params(self.nodes, seed)
        if case["kind"] in ("forward", "optical"):
            # measured data: tissue that lets a signal through (mua 0.01, mus 1 of the 3D regression suite)
            self.mua, self.mus = 0.4 * self.mua, 0.5 * self.mus
        rng = np.random.default_rng(seed + 1000)
        turn = rng.uniform(0.0, 1.0)
        nq, nm = case["nq"], case.get("nm", 1)
        self.Q = _ring_points(case["mesh"], nq, turn=2 * math.pi * turn / nq)
        # the first detector 10 mm along the surface from the first source
        arc = 10.0 / (80.0 if case["mesh"] == "ellipsoid" else 25.0)
        self.M = _ring_points(case["mesh"], nm, turn=2 * math.pi * turn / nq + arc)
        share = max(1, int(round(nm * case.get("links", 1.0))))
        self.links = [sorted((q + j) % nm for j in range(share)) for q in range(nq)]
        self.pairs = [(q, m) for q in range(nq) for m in self.links[q]]
        self.decay = complex(rng.uniform(0.15, 0.3), rng.uniform(0.005, 0.02))
        self.omega = case.get("freq", 0.0) * 2 * math.pi * 1e-6
        self.omegas = np.array([0.0, 50.0, 100.0, 200.0])[np.arange(nq) % 4] * 2 * math.pi * 1e-6


def _green(points, x, decay):
    """fields of point sources in a homogeneous medium at x: (len(x), len(points))"""
    d = torch.cdist(x, points)
    return torch.exp(-decay * d.to(torch.complex128)) / (d + 2.0)


def _fields(inp):
    """direct and adjoint fields [n][nq], [n][nm] and the linear projections of the linked pairs"""
    x = torch.from_numpy(inp.nodes).to(DEV)
    Q, M = torch.from_numpy(inp.Q).to(DEV), torch.from_numpy(inp.M).to(DEV)
    q, m = (torch.tensor([p[i] for p in inp.pairs], device=DEV) for i in (0, 1))
    proj = _green(Q, M, inp.decay)[m, q] * 0.1
    return _green(Q, x, inp.decay).contiguous(), _green(M, x, inp.decay).contiguous(), proj.contiguous()


def _mesh(inp):
    mesh = T.Mesh(data=(inp.nodes, inp.el))
    mesh.SetQM(inp.Q, inp.M, links=inp.links)
    return mesh


def _solver(case, inp, mesh):
    # fields as such to 1e-10, data (orders of magnitude below the fields' peak) to 1e-12
    f = T.FwdSolver(mesh, case["solver"], 1e-12 if case["kind"] == "forward" else 1e-10, complex=case["solver"] != "CG")
    f.SetMode(case["mode"])
    f.SetPrecon("DIAG")
    f.Allocate()
    f.Reset(T.Solution(inp.mua, inp.mus, inp.ref), inp.omega)
    return f


def prepare(case, seed):
    kind = case["kind"]
    inp = _Inputs(case, seed)
    mesh = _mesh(inp)
    s = dict(kind=kind, nq=case["nq"], nm=case.get("nm", 0), mesh=mesh)
    if kind in ("fields", "freqs", "forward"):
        cplx = case["solver"] != "CG"
        q = mesh.Qvec(width=2.0).toarray()
        s["rhs"] = torch.from_numpy(np.ascontiguousarray(q if cplx else q.real)).to(DEV)
        s["phi"] = torch.zeros_like(s["rhs"])
        s["solver"] = _solver(case, inp, mesh)
        if kind == "freqs":
            s["omegas"] = inp.omegas
        if kind == "forward":
            s.update(mua=inp.mua, mus=inp.mus, ref=inp.ref, omega=inp.omega,
                     mvec=mesh.Mvec(width=2.0, ref=inp.ref).T.tocsr())
    elif kind == "optical":
        s.update(mua=inp.mua, mus=inp.mus, ref=inp.ref, freq=case["freq"], qvec=mesh.Qvec(width=2.0),
                 mvec=mesh.Mvec(width=2.0, ref=inp.ref))
    else:
        s["dphi"], s["aphi"], s["proj"] = _fields(inp)
        nsol = inp.n
        if kind != "jac_nodal":
            s["raster"] = T.Raster(mesh, np.full(inp.dim, case["grid"]))
            nsol = s["raster"].SLen()
        if kind == "gradient":
            s["zero"] = torch.zeros(2 * nsol, dtype=torch.float64, device=DEV)
            s["out"] = torch.zeros_like(s["zero"])
            # one adjoint field per source
            s["aphi"] = s["aphi"][:, torch.arange(case["nq"], device=DEV) % case["nm"]].contiguous()
        else:
            s["out"] = torch.empty((2 * len(inp.pairs), 2 * nsol), dtype=torch.float64, device=DEV)
    torch.cuda.synchronize()
    return s


# -------------------------------------------------------------------- runs
def _p(t):
    return C.c_void_p(t.data_ptr())


def run(s):
    kind, nq, nm = s["kind"], s["nq"], s["nm"]
    if kind == "fields":
        s["solver"].CalcFieldsDevice(nq, s["rhs"].data_ptr(), s["phi"].data_ptr())
        return s["phi"]
    if kind == "freqs":
        s["solver"].CalcFieldsFreqsDevice(nq, s["rhs"].data_ptr(), s["phi"].data_ptr(), s["omegas"])
        return s["phi"]
    if kind == "forward":
        f = s["solver"]
        f.Reset(T.Solution(s["mua"], s["mus"], s["ref"]), s["omega"])
        f.CalcFieldsDevice(nq, s["rhs"].data_ptr(), s["phi"].data_ptr())
        return s["phi"], f.ProjectAllDevice(s["mvec"], s["phi"].data_ptr(), nq, scale="lin")
    if kind == "optical":
        return s["mesh"].JacobianOptical(None, s["qvec"], s["mvec"], s["mua"], s["mus"], s["ref"], s["freq"])
    if kind == "gradient":
        L.call("tmi_memcpy_d2d", _p(s["out"]), _p(s["zero"]), s["zero"].numel() * 8)
        L.call("tmi_raster_data_gradient_device", s["raster"].handle_ptr(), nq, _p(s["dphi"]), nq, _p(s["aphi"]), nq,
               _p(s["out"]))
        return s["out"]
    if kind == "jac_nodal":
        L.call("tmi_jacobian_nodal_device", s["mesh"].handle_ptr(), nq, nm, _p(s["dphi"]), nq, _p(s["aphi"]), nm,
               _p(s["proj"]), L.DATA_LOG, _p(s["out"]))
        return s["out"]
    L.call("tmi_jacobian_raster_device", s["raster"].handle_ptr(), nq, nm, _p(s["dphi"]), nq, _p(s["aphi"]), nm,
           _p(s["proj"]), L.DATA_LOG, _p(s["out"]))
    return s["out"]


# -------------------------------------------------------------------- work
def _sizes(case):
    """nodes, elements and nonzeros of the system matrix"""
    k = case["k"]
    if case["mesh"] == "disk":
        n, e = 1 + 3 * k * (k + 1), 6 * k * k
        return n, e, 7 * n
    if case["mesh"] == "cylinder":
        n, e = (1 + 3 * k * (k + 1)) * (case["layers"] + 1), 18 * k * k * case["layers"]
    else:
        n, e = (k + 1) ** 3, 6 * k ** 3
    return n, e, 15 * n


def work(case):
    n, e, nnz = _sizes(case)
    dim = 2 if case["mesh"] == "disk" else 3
    nq, nm, kind = case["nq"], case.get("nm", 0), case["kind"]
    es = 8 if case.get("solver") == "CG" else 16
    links = nq * max(1, int(round(nm * case.get("links", 1.0))))
    if kind in ("fields", "freqs"):   # matrix, right-hand sides in, fields out
        return dict(bytes=nnz * (es + 4) + 2 * n * nq * es, flops=2.0 * nnz * nq * (1 if es == 8 else 4))
    if kind == "forward":             # coefficients and mesh in, the rest as above
        return dict(bytes=3 * n * 8 + e * (dim + 1) * 4 + nnz * (es + 4) + 2 * n * nq * es,
                    flops=8.0 * nnz * nq + 100.0 * e)
    if kind == "optical":             # fields of both sides, Jacobian
        return dict(bytes=nnz * 20 + 2 * n * (nq + nm) * 16 + 4 * nq * nm * n * 8,
                    flops=8.0 * nnz * (nq + nm) + 16.0 * nq * nm * nnz / n * n)
    if kind == "jac_nodal":           # fields in, J out; f^T A_i g and f^T B_i g per node and link
        return dict(bytes=n * (nq + nm) * 16 + 4 * links * n * 8,
                    flops=16.0 * links * nnz + 8.0 * min(nq, nm) * nnz * nnz / n)
    inside = {"disk": math.pi / 4, "cylinder": math.pi / 4, "ellipsoid": math.pi / 6}[case["mesh"]]
    vox = inside * case["grid"] ** dim
    if kind == "gradient":            # fields in, two images out
        return dict(bytes=n * 2 * nq * 16 + 3 * 2 * vox * 8, flops=vox * nq * 8.0 * (1 + 4 * dim))
    return dict(bytes=n * (nq + nm) * 16 + 4 * links * vox * 8, flops=vox * links * 8.0 * (1 + dim))


def tolerance(case):
    kind = case["kind"]
    if kind in ("fields", "freqs", "forward"):
        # relative residual 1e-10: two correct solves are up to 3e-10 off the exact fields (measured)
        return dict(rel=5e-9, max=1e-6)
    if kind == "optical":
        # rows divided by the projections, which hold fewer digits than the fields solved to 1e-12
        return dict(rel=1e-6, max=1e-3)
    # FP64 sums in another order
    return dict(rel=1e-12, max=1e-9)


# ------------------------------------------------------------------- exact
def _tables(dim):
    """integrals of products of two and three shape functions over a unit simplex of that dimension"""
    nn = dim + 1
    f3 = np.zeros((nn, nn, nn))
    f2 = np.zeros((nn, nn))
    fact = math.factorial
    for i in range(nn):
        for j in range(nn):
            a = np.bincount([i, j], minlength=nn)
            f2[i, j] = fact(dim) * np.prod([fact(v) for v in a]) / fact(dim + 2)
            for k in range(nn):
                a = np.bincount([i, j, k], minlength=nn)
                f3[i, j, k] = fact(dim) * np.prod([fact(v) for v in a]) / fact(dim + 3)
    return torch.from_numpy(f2).to(DEV), torch.from_numpy(f3).to(DEV)


class _Fem:
    """element geometry and matrices of linear simplices in FP64 torch"""

    def __init__(self, inp):
        self.n, self.dim, self.nn = inp.n, inp.dim, inp.dim + 1
        self.x, self.el = torch.from_numpy(inp.nodes).to(DEV), torch.from_numpy(inp.el.astype(np.int64)).to(DEV)
        X = self.x[self.el]
        J = X[:, 1:] - X[:, :1]
        self.size = torch.linalg.det(J) / math.factorial(self.dim)
        Ji = torch.linalg.inv(J)
        self.grad = torch.cat([-Ji.sum(2, keepdim=True), Ji], 2).transpose(1, 2)   # [e][node][axis]
        self.f2, self.f3 = _tables(self.dim)
        # boundary sides: those of one element only
        sides = torch.cat([self.el[:, [j for j in range(self.nn) if j != i]] for i in range(self.nn)])
        key = torch.zeros(len(sides), dtype=torch.int64, device=DEV)
        for c in sides.sort(1).values.unbind(1):
            key = key * self.n + c
        _, inv, cnt = key.unique(return_inverse=True, return_counts=True)
        self.sides = sides[cnt[inv] == 1]
        S = self.x[self.sides]
        if self.dim == 2:
            self.area = (S[:, 1] - S[:, 0]).norm(dim=1)
        else:
            self.area = torch.linalg.cross(S[:, 1] - S[:, 0], S[:, 2] - S[:, 0]).norm(dim=1) / 2
        self.b2, self.b3 = _tables(self.dim - 1)

    def _sum(self, parts):
        """ELL form (columns, values) of the sum of element matrices [(elements, matrices)]"""
        i = torch.cat([e[:, :, None].expand(-1, -1, e.shape[1]).reshape(-1) for e, _ in parts])
        j = torch.cat([e[:, None, :].expand(-1, e.shape[1], -1).reshape(-1) for e, _ in parts])
        v = torch.cat([m.reshape(-1) for _, m in parts])
        key, inv = (i * self.n + j).unique(return_inverse=True)
        val = torch.zeros(len(key), dtype=v.dtype, device=DEV).index_add_(0, inv, v)
        row = key // self.n
        cnt = torch.bincount(row, minlength=self.n)
        at = torch.arange(len(key), device=DEV) - (cnt.cumsum(0) - cnt)[row]
        col = torch.zeros((self.n, int(cnt.max())), dtype=torch.int64, device=DEV)
        out = torch.zeros(col.shape, dtype=v.dtype, device=DEV)
        col[row, at], out[row, at] = key % self.n, val
        return col, out

    def system(self, inp):
        """(columns, real part, imaginary part at omega 1) of the diffusion system in ELL form"""
        c0 = 0.3
        ref = torch.from_numpy(inp.ref).to(DEV)
        mua, mus = torch.from_numpy(inp.mua).to(DEV), torch.from_numpy(inp.mus).to(DEV)
        cmua, kap = mua * c0 / ref, c0 / (3 * ref * (mua + mus))
        c2a = torch.from_numpy(_c2a(inp.ref)).to(DEV)
        V = self.size[:, None, None]
        mass = self.f2 * V
        ff = torch.einsum("ijk,ek->eij", self.f3, cmua[self.el]) * V
        dd = torch.einsum("eia,eja->eij", self.grad, self.grad) * V * kap[self.el].mean(1)[:, None, None]
        bb = torch.einsum("ijk,ek->eij", self.b3, c2a[self.sides]) * self.area[:, None, None]
        col, val = self._sum([(self.el, torch.complex(ff + dd, mass)),
                              (self.sides, torch.complex(bb, torch.zeros_like(bb)))])
        return col, val.real.contiguous(), val.imag.contiguous()

    def profiles(self, points, width, scale=None):
        """Gaussian boundary profiles [n][points] (real)"""
        g = torch.zeros((self.n, len(points)), dtype=torch.float64, device=DEV)
        on = self.sides.reshape(-1).unique()
        d = torch.cdist(self.x[on], torch.from_numpy(points).to(DEV))
        g[on] = torch.exp(-d * d / (2 * width * width)) / (math.sqrt(2 * math.pi) * width) ** (self.dim - 1)
        col, val = self._sum([(self.sides, self.b2 * self.area[:, None, None])])
        out = sum(val[:, s, None] * g[col[:, s]] for s in range(col.shape[1]))
        return out if scale is None else out * torch.from_numpy(scale).to(DEV)[:, None]


def _c2a(ref):
    costh = np.abs(np.cos(np.arcsin(1.0 / ref)))
    r0 = (ref - 1) ** 2 / (ref + 1) ** 2
    a = (2 / (1 - r0) - 1 + costh ** 3) / (1 - costh ** 2)
    return 0.3 / (2 * ref * a)


def _solve(col, re, im, omega, B, tol=2e-15):
    """(re + i omega im) X = B by diagonally preconditioned conjugate (orthogonal) gradients in FP64,
    restarted from the true residual; omega one number or one per column"""
    w = torch.as_tensor(omega, dtype=torch.float64, device=DEV)
    cplx = B.is_complex()

    def times(X):
        a, b = torch.zeros_like(X), torch.zeros_like(X)
        for s in range(col.shape[1]):
            g = X[col[:, s]]
            a += re[:, s, None] * g
            if cplx:
                b += im[:, s, None] * g
        return a + 1j * w * b if cplx else a

    own = col == torch.arange(len(col), device=DEV)[:, None]
    own &= re != 0
    d = (re * own).sum(1)[:, None] + ((1j * w * (im * own).sum(1)[:, None]) if cplx else 0.0)
    X = torch.zeros_like(B)
    bn = B.abs().square().sum(0).sqrt()
    for _ in range(4):
        R = B - times(X)
        if float((R.abs().square().sum(0).sqrt() / bn).max()) < tol:
            break
        Z = R / d
        P = Z.clone()
        rz = (R * Z).sum(0)
        for it in range(600):
            Y = times(P)
            al = rz / (P * Y).sum(0)
            al = torch.where(torch.isfinite(al.abs()), al, torch.zeros_like(al))
            X += al * P
            R -= al * Y
            if it % 10 == 9 and float((R.abs().square().sum(0).sqrt() / bn).max()) < 0.1 * tol:
                break
            Z = R / d
            new = (R * Z).sum(0)
            be = new / rz
            P = Z + torch.where(torch.isfinite(be.abs()), be, torch.zeros_like(be)) * P
            rz = new
    return X


def _jac_rows(inp, pmua, pkap, proj):
    """log Jacobian rows from the PMDFs [pairs][solution]"""
    a, b = -pmua / proj[:, None], -pkap / proj[:, None]
    return torch.cat([torch.cat([a.real, b.real], 1), torch.cat([a.imag, b.imag], 1)])


def _exact_nodal(fem, inp, dphi, aphi, proj):
    nq = dphi.shape[1]
    out = torch.empty((2 * len(inp.pairs), 2 * inp.n), dtype=torch.float64, device=DEV)
    V, at, np_ = fem.size, 0, len(inp.pairs)
    gf = torch.einsum("eia,eiq->eaq", fem.grad.to(torch.complex128), dphi[fem.el])
    ga = torch.einsum("eia,eim->eam", fem.grad.to(torch.complex128), aphi[fem.el])
    for q in range(nq):
        ms = inp.links[q]
        for m0 in range(0, len(ms), 8):
            m = torch.tensor(ms[m0:m0 + 8], device=DEV)
            f, g = dphi[fem.el, q], aphi[:, m][fem.el]                     # [e][nn], [e][nn][m]
            w = torch.einsum("ijk,ej->eik", fem.f3.to(torch.complex128), f) * V[:, None, None]
            mu = torch.einsum("eik,ekm->eim", w, g)
            ka = (torch.einsum("ea,eam->em", gf[:, :, q], ga[:, :, m]) * (V / fem.nn)[:, None])[:, None].expand_as(mu)
            pm = torch.zeros((inp.n, len(m)), dtype=torch.complex128, device=DEV)
            pk = torch.zeros_like(pm)
            pm.index_add_(0, fem.el.reshape(-1), mu.reshape(-1, len(m)))
            pk.index_add_(0, fem.el.reshape(-1), ka.reshape(-1, len(m)))
            p = proj[at:at + len(m)]
            a, b = (-pm / p).T, (-pk / p).T
            out[at:at + len(m), :inp.n], out[at:at + len(m), inp.n:] = a.real, b.real
            out[np_ + at:np_ + at + len(m), :inp.n], out[np_ + at:np_ + at + len(m), inp.n:] = a.imag, b.imag
            at += len(m)
    return out


def _grid_fields(fem, inp, grid, F):
    """columns F [n][c] on the regular grid over the bounding box: values, gradients [3][voxel][c] at
    the grid points inside the mesh, and the voxel size"""
    dim, nn = fem.dim, fem.nn
    lo, hi = fem.x.min(0).values, fem.x.max(0).values
    h = (hi - lo) / (grid - 1)
    X = fem.x[fem.el]
    e0 = ((X.min(1).values - 1e-6 - lo) / h).ceil().long().clamp(min=0)
    e1 = ((X.max(1).values + 1e-6 - lo) / h).floor().long().clamp(max=grid - 1)
    span = [int(v) + 1 for v in (e1 - e0).max(0).values]
    stride = torch.tensor([grid ** d for d in range(dim)], device=DEV)
    owner = torch.full((grid ** dim,), len(fem.el), dtype=torch.int64, device=DEV)
    ids = torch.arange(len(fem.el), device=DEV)
    for o in np.ndindex(*span):
        at = e0 + torch.tensor(o, device=DEV)
        p = at * h + lo
        lam = torch.einsum("eia,ea->ei", fem.grad[:, 1:], p - X[:, 0])
        ok = (at <= e1).all(1) & (lam >= -1e-8).all(1) & (lam.sum(1) <= 1 + 1e-8)
        owner.scatter_reduce_(0, (at * stride).sum(1)[ok], ids[ok], "amin")
    inside = owner < len(fem.el)
    g = inside.nonzero()[:, 0]
    pos = torch.stack([(g // int(s)) % grid for s in stride], 1)
    e = owner[g]
    lam = torch.einsum("eia,ea->ei", fem.grad[e][:, 1:], (pos * h + lo) - X[e, 0])
    lam = torch.cat([1 - lam.sum(1, keepdim=True), lam], 1)
    vals = torch.zeros((grid ** dim, F.shape[1]), dtype=F.dtype, device=DEV)
    vals[g] = sum(lam[:, j, None] * F[fem.el[e, j]] for j in range(nn))
    grads = []
    for d in range(dim):
        ih = grid / (hi[d] - lo[d])
        s = int(stride[d])
        bl = (pos[:, d] > 0) & inside[(g - s).clamp(min=0)]
        bh = (pos[:, d] < grid - 1) & inside[(g + s).clamp(max=grid ** dim - 1)]
        vc, vl, vh = vals[g], vals[(g - s).clamp(min=0)], vals[(g + s).clamp(max=grid ** dim - 1)]
        zero = torch.zeros_like(vc)
        grads.append(torch.where((bl & bh)[:, None], (vh - vl) * (0.5 * ih),
                                 torch.where(bl[:, None], (vc - vl) * ih,
                                             torch.where(bh[:, None], (vh - vc) * ih, zero))))
    return vals[g], grads, float(torch.prod(h))


def exact(case, seed):
    kind = case["kind"]
    inp = _Inputs(case, seed)
    fem = _Fem(inp)
    if kind in ("fields", "freqs", "forward", "optical"):
        col, re, im = fem.system(inp)
        B = fem.profiles(inp.Q, 2.0)
        if case.get("solver") == "CG":
            return _solve(col, re, im, 0.0, B)
        B = B.to(torch.complex128)
        if kind != "optical":
            X = _solve(col, re, im, inp.omegas if kind == "freqs" else inp.omega, B)
            if kind != "forward":
                return X
        Mv = fem.profiles(inp.M, 2.0, _c2a(inp.ref)).to(torch.complex128)
        if kind == "optical":
            X = _solve(col, re, im, inp.omega, torch.cat([B, Mv], 1))
            X, A = X[:, :case["nq"]].contiguous(), X[:, case["nq"]:].contiguous()
        P = Mv.T @ X
        proj = torch.stack([P[m, q] for q, m in inp.pairs])
        if kind == "forward":
            return X, proj
        return _exact_nodal(fem, inp, X, A, proj)
    dphi, aphi, proj = _fields(inp)
    if kind == "jac_nodal":
        return _exact_nodal(fem, inp, dphi, aphi, proj)
    nq = case["nq"]
    if kind == "gradient":
        aphi = aphi[:, torch.arange(nq, device=DEV) % case["nm"]]
    v, gr, size = _grid_fields(fem, inp, case["grid"], torch.cat([dphi, aphi], 1))
    if kind == "gradient":
        mu = (v[:, :nq] * v[:, nq:]).real.sum(1)
        ka = sum((x[:, :nq] * x[:, nq:]).real.sum(1) for x in gr)
        return -torch.cat([mu, ka])
    S, np_ = len(v), len(inp.pairs)
    out = torch.empty((2 * np_, 2 * S), dtype=torch.float64, device=DEV)
    for k, (q, m) in enumerate(inp.pairs):
        a = -size * v[:, q] * v[:, nq + m] / proj[k]
        b = -size * sum(x[:, q] * x[:, nq + m] for x in gr) / proj[k]
        out[k, :S], out[k, S:], out[np_ + k, :S], out[np_ + k, S:] = a.real, b.real, a.imag, b.imag
    return out
