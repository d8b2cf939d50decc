// Host side of the resident solve (krylov_resident.hpp): when it is taken,
// how the columns are split over teams, and the launch itself.
#include <algorithm>
#include <climits>
#include <cmath>

#include "krylov_resident.hpp"
#include "solver.hpp"

namespace tmi {

// When and how a solve runs resident.  Against the launch sequence (us per
// iteration; COCG/PCG/BiCGSTAB on disks and cylinders):
//   n 3,169 real x 16: 7.5 / 31       n 31,525 c64 x 2 (BiCGSTAB): 24 / 97
//   n 19,441 c32 x 24: 26 / 38        n 31,525 c64 x 16: 27 / 59
//   n 31,525 c32 x 8: 24 / 39         n 103,267 c32 x 8: 42 / 54
//   n 31,525 c32 x 32 (BiCGSTAB): 75 / 75    n 250,047 c32 x 4: 49 / 58
// so it is taken for blocks of up to RES_MAX_BYTES.  Above 16 columns the
// launch sequence's complex FP32 tiles run on the matrix cores; with COCG it is
// then the faster one for long operators (n 31,525 x 33: 79 / 71, n 50,653 x 17:
// 65 / 55, n 39,304 x 24: 52 / 52, n 19,683 x 52: 47 / 39 but 12 % faster in all):
// beyond RES_MAX_MACS entries times columns, rounded up to whole teams.
static constexpr size_t RES_MAX_BYTES = 8500000;
static constexpr long RES_MAX_MACS = 20000000;
// Teams: one column per team keeps the reductions small and the ranks few
// (n 19,441 x 24: 8 ranks 26 us, 32 ranks 28; n 31,525 c64 x 16: 16 ranks 27,
// 32 ranks 34) but every team reads the matrix: beyond RES_MAX_ENTRIES
// entries per iteration (n 103,267 x 8: 4 teams 53 us, 1 team 42) the columns
// share as few teams as hold them.  So they do where a thread of a team with
// one column would hold too many rows, as most of their operator then comes
// from memory between uses (us: one column a team / few teams / launch sequence):
//   more than 4 rows, complex (with COCG, if the XCDs fetch more than
//   RES_XCD_ENTRIES entries an iteration, a team of up to 32 ranks on one XCD):
//     c32 COCG      n 132,651 x 4: 47 / 36 / 45    n 67,951 x 8: 36 / 28 / 41
//                   n 19,441 x 24 (1.1 M entries): 25 / 28 / 37
//     c32 BiCGSTAB  n 132,651 x 4: 97 / 64 / 69    n 19,441 x 24: 54 / 42 / 55
//     c64 COCG      n 132,651 x 4: 77 / 44 / 54    n 67,951 x 7: 58 / 34 / 47
//   more than 2 rows, c64 BiCGSTAB, four teams at most (each on several XCDs
//   in any case) or twice RES_XCD_ENTRIES:
//     n 103,267 x 4: 100 / 63 / 75    n 250,047 x 2: 112 / 75 / 104
//     n 50,653 x 8: 81 / 60 / 70      n 31,525 x 16 (3.6 M entries): 67 / 68 / 113
// Tiny systems run on single workgroups without any exchange (n 817 x 4: 7.0
// us, 4 ranks 9.4; n 3,169 x 16: 11.2).
static constexpr long RES_MAX_ENTRIES = 8000000;
static constexpr long RES_XCD_ENTRIES = 2000000;
static constexpr int RES_ONE_WG = 1500;

bool Solver::resident_block(int nq, int md) const
{
    if (named || tuning || res_given_up || lsolver == TMI_LSOLVER_GMRES || nq < 1 || nq > 64) return false;
    if (tuned_sequence[md] >> (nq - 1) & 1) return false;
    return (size_t)mesh->n * nq * vbytes(md == TMI_MODE_MIXED_BLOCK ? vk32() : vk64()) <= RES_MAX_BYTES;
}

Solver::ResPlan Solver::resident_plan(int nq, int md)
{
    ResPlan none;
    if (!resident_block(nq, md)) return none;
    const bool mixed = md == TMI_MODE_MIXED_BLOCK, bicg = !pcg();
    const VKind vk = mixed ? vk32() : vk64();
    const size_t sz = vbytes(vk);
    const bool wide = vk == VK_C64;
    int pow = 1;
    while (pow < nq) pow *= 2;
    if (vk == VK_C32 && !bicg && nq > 16 && mesh->nnz * (long)pow > RES_MAX_MACS) return none;
    int T = mesh->n <= RES_ONE_WG ? RES_WG : pow;
    if (T > 1 && T < RES_WG) {
        const int per = (mesh->n + RES_WG / T * RES_NT - 1) / (RES_WG / T * RES_NT);   // rows a thread, one column a team
        const long xcd = std::min(T, 8) * (long)mesh->nnz;
        bool few = (long)T * mesh->nnz > RES_MAX_ENTRIES;
        if (cplx && per > 4) few |= bicg || xcd > RES_XCD_ENTRIES;
        if (wide && bicg && per > 2) few |= T <= 4 || xcd > 2 * RES_XCD_ENTRIES;
        // (BiCGSTAB, n 31,525 c32 x 17 to 32: two teams 75-76 us, four 73-75, the
        // launch sequence 74-75)
        if (few) T = std::max(1, pow / (wide || (bicg && pow > RES_KC) ? 8 : RES_KC));
    }
    for (;; T /= 2) {
        if (T < 1) return none;
        const int nr = RES_WG / T;
        int kc = 1;
        while (kc * T < nq) kc *= 2;
        const int cl = wide ? std::min(kc, 2) : (kc >= 4 ? 4 : 1), lpr = kc / cl;
        if (kc > RES_KC || lpr > RES_LANES) return none;
        const int rows = (mesh->n + nr - 1) / nr, need = (rows * lpr + RES_NT - 1) / RES_NT;
        int E = 1;
        while (E < need) E *= 2;
        // instantiations (krylov_resident_*.hip)
        const int emax = cl == 1 ? (wide && bicg ? 4 : 8) : (bicg ? 2 : 4);
        if (E > emax) continue;   // fewer, longer teams
        const ResLayout *l = nullptr;
        try {
            l = mesh->res_layout(order_kind, nr, st);
        } catch (const Error &err) {
            if (err.code != TMI_ERR_OOM) throw;
            return none;   // the launch sequence needs none
        }
        if (!l || l->nu == INT_MAX) continue;
        if ((((size_t)l->nu * kc * sz + 15) & ~(size_t)15) + res_lds_fixed(kc) > RES_LDS) continue;
        ResPlan p;
        p.nr = nr;
        p.kc = kc;
        p.cl = cl;
        p.E = E;
        return p;
    }
}

static constexpr size_t RES_CTL_BYTES = sizeof(ResColOut) * 64 + sizeof(double) * 64 + 8;

// Vectors of the columns rounded up to whole teams (a power of two at most),
// words and results
size_t Solver::resident_bytes(int nq, int md) const
{
    if (!resident_block(nq, md)) return 0;
    const bool mixed = md == TMI_MODE_MIXED_BLOCK;
    const size_t sin = vbytes(mixed ? vk32() : vk64()), inner = pcg() ? 1 : mixed ? 2 : 3;
    size_t cols = 1;
    while (cols < (size_t)nq) cols *= 2;
    return mesh->n * cols * (inner * sin + vbytes(vk64())) + (RES_PART_WORDS + RES_TOT_WORDS) * sizeof(res_u64) +
           RES_CTL_BYTES;
}

Solver::Slices Solver::sliced(OpKind k, const ResLayout &l, int nr)
{
    int lg = 0;
    while ((1 << lg) < nr) lg++;
    SliceOp &o = slice_op[k][lg];
    const bool f32 = k == OPK_32 || k == OPK_P32 || k == OPK_MF32;
    const void *src = k == OPK_32 ? (const void *)sval32.p : k == OPK_64 ? (const void *)sval64.p
                    : k == OPK_P32 ? (const void *)pval32.p : k == OPK_P64 ? (const void *)pval64.p
                    : k == OPK_MF32 ? (const void *)mfval32.p : (const void *)mfval64.p;
    const size_t es = (f32 ? 4 : 8) * (cplx ? 2 : 1);
    o.used = slice_clock;
    if (!o.valid) {
        if (!o.v || o.v->bytes() != (size_t)l.nent * es) {
            o.v.reset();
            o.v = std::make_shared<DBuf<char>>((size_t)l.nent * es);
        }
        launch_slice_vals((int)es, l.nent, l.slot.p, src, o.v->p, st);
        TMI_HIP(hipStreamSynchronize(st));   // other streams read it next
        o.valid = true;
    }
    return o.v;
}

size_t Solver::slice_bytes() const
{
    size_t b = 0;
    for (auto &k : slice_op)
        for (const SliceOp &o : k) b += o.v ? o.v->bytes() : 0;
    return b;
}

void Solver::trim_slices()
{
    for (size_t held = slice_bytes(); held > SLICE_BYTES;) {
        SliceOp *old = nullptr;
        for (auto &k : slice_op)
            for (SliceOp &o : k)
                if (o.v && o.used != slice_clock && (!old || o.used < old->used)) old = &o;
        if (!old) return;
        held -= old->v->bytes();
        old->v.reset();   // freed with the last solve that holds it
        old->valid = false;
    }
}

// As below, and -1 when there is no memory for it (the launch sequence works in
// narrower tiles, or has its own already)
int Solver::solve_resident(Exec &e, const ResPlan &plan, int nq, const void *d_b, void *d_x, int ld,
                           tmi_colstat *stats, int md, const double *h_omega)
{
    try {
        return launch_resident(e, plan, nq, d_b, d_x, ld, stats, md, h_omega);
    } catch (const Error &err) {
        if (err.code != TMI_ERR_OOM) throw;
        e.release_resident();
        return -1;
    }
}

// Columns 0 .. nq-1 in one cooperative launch.  Returns the number of columns
// above the tolerance, or -1 when the launch was refused or gave up: its
// memory is then free again, the fields hold initial guesses or solutions, a
// valid start for the launch sequence, and the handle keeps to that one (a
// give-up costs the 4 s of its bounded waits).
int Solver::launch_resident(Exec &e, const ResPlan &plan, int nq, const void *d_b, void *d_x, int ld,
                            tmi_colstat *stats, int md, const double *h_omega)
{
    hipStream_t st = e.st;
    const int n = mesh->n;
    const bool mixed = md == TMI_MODE_MIXED_BLOCK, mf = h_omega != nullptr;
    const bool cg = pcg(), bil = lsolver == TMI_LSOLVER_COCG, diag = precon == TMI_PRECON_DIAG;
    const VKind vk = mixed ? vk32() : vk64();
    const size_t sin = vbytes(vk), s64 = vbytes(vk64());
    const int cap = (mixed && mixed_maxit > 0) ? mixed_maxit : (maxit > 0 ? maxit : n + 1);
    const ResLayout &l = *mesh->res_layout(order_kind, plan.nr, this->st);   // built by the plan
    ResArgs a{};
    a.n = n;
    a.K = nq;
    a.kc = plan.kc;
    a.nr = plan.nr;
    a.maxit = cap;
    a.ru = mixed ? reliable_every : (1 << 30);
    a.mixed = mixed ? 1 : 0;
    a.nu = l.nu;
    a.tol2 = tol * tol;
    // the recursive residual aims a little below the target so that the
    // verifying FP64 residual usually passes at the first check
    a.itol2 = mixed ? 0.25 * a.tol2 : a.tol2;
    a.srow = l.srow.p;
    a.node = l.node.p;
    a.sofs = l.sofs.p;
    a.rslice = l.rslice.p;
    a.hofs = l.hofs.p;
    a.halo = l.halo.p;
    a.lcol = l.lcol.p;
    a.gcol = l.gcol.p;
    Slices op, op64;   // held until the launch has ended
    {
        std::lock_guard<std::mutex> lk(prep_mu);
        slice_clock++;
        const bool right = diag && !cg;   // BiCGSTAB iterates with K D^-1
        op = sliced(mf ? (mixed ? OPK_MF32 : OPK_MF64)
                         : right ? (mixed ? OPK_P32 : OPK_P64) : (mixed ? OPK_32 : OPK_64), l, plan.nr);
        op64 = sliced(mf ? OPK_MF64 : OPK_64, l, plan.nr);
        trim_slices();
    }
    a.op = op->p;
    a.op64 = (const double *)op64->p;
    if (diag) {
        if (mf) a.idiag = mixed ? (const void *)mfdiag32.p : (const void *)mfdiag64.p;
        else a.idiag = mixed ? (const void *)idiag32.p : (const void *)idiag64.p;
    }
    a.b = d_b;
    a.x = d_x;
    a.ld = ld;
    Exec::Resident &r = e.res;
    const int teams = (nq + plan.kc - 1) / plan.kc;
    const size_t elems = (size_t)n * teams * plan.kc;
    if (r.pub_p.n < elems * sin) r.pub_p.alloc(elems * sin);
    if (!cg && r.pub_s.n < elems * sin) r.pub_s.alloc(elems * sin);
    if (!cg && !mixed && r.rd0.n < elems * sin) r.rd0.alloc(elems * sin);
    if (r.x64.n < elems * s64) r.x64.alloc(elems * s64);
    if (!r.words.p) {
        r.words.alloc(RES_PART_WORDS + RES_TOT_WORDS);
        r.epoch = 0xffffffffu;   // cleared below before the first use
    }
    if (!r.ctl.p) r.ctl.alloc(RES_CTL_BYTES);
    if (!r.h_ctl) TMI_HIP(hipHostMalloc((void **)&r.h_ctl, r.ctl.n));
    double *d_om = (double *)(r.ctl.p + sizeof(ResColOut) * 64);
    double *h_om = (double *)(r.h_ctl + sizeof(ResColOut) * 64);
    a.out = (ResColOut *)r.ctl.p;
    a.abort_flag = (int *)(d_om + 64);
    a.pub_p = r.pub_p.p;
    a.pub_s = r.pub_s.p;
    a.rd0 = r.rd0.p;
    a.x64 = r.x64.p;
    a.part = r.words.p;
    a.tot = r.words.p + RES_PART_WORDS;
    const size_t lds = (((size_t)l.nu * plan.kc * sin + 15) & ~(size_t)15) + res_lds_fixed(plan.kc);
    // reductions of one launch, at most: eight per iteration (replacements
    // included) and those of the replacements between iterations
    const unsigned need = (unsigned)std::min<long>(8l * cap + 8192, 0x7fffffffl);
    if (r.epoch > 0xffffffffu - need) {
        TMI_HIP(hipMemsetAsync(r.words.p, 0, r.words.bytes(), st));
        r.epoch = 0;
    }
    a.epoch = r.epoch;
    r.epoch += need;
    // omegas and the cleared abort word in one upload
    for (int c = 0; c < 64; c++) h_om[c] = mf && c < nq ? h_omega[c] : 0.0;
    *(int *)(h_om + 64) = test_resident == 2 ? 1 : 0;
    TMI_HIP(hipMemcpyAsync(d_om, h_om, sizeof(double) * 64 + 8, hipMemcpyHostToDevice, st));
    a.omega = mf ? d_om : nullptr;
    const bool ok = test_resident != 1 && (cg ? launch_resident_cg(vk, plan.cl, plan.E, bil, mf, a, lds, st)
                                              : launch_resident_bicg(vk, plan.cl, plan.E, a, lds, st));
    if (ok) {
        TMI_HIP(hipMemcpyAsync(r.h_ctl, r.ctl.p, r.ctl.n, hipMemcpyDeviceToHost, st));
        TMI_HIP(hipStreamSynchronize(st));
        e.n_sync++;
    }
    if (!ok || *(int *)(h_om + 64)) {
        res_given_up++;
        e.release_resident();
        return -1;
    }
    const ResColOut *out = (const ResColOut *)r.h_ctl;
    int notconv = 0;
    for (int c = 0; c < nq; c++) {
        const double b2 = out[c].bnorm2, r2 = out[c].res2;
        const bool conv = b2 == 0.0 || r2 <= a.tol2 * b2;
        if (!conv) notconv++;
        stats[c].iters = out[c].iters;
        stats[c].sweeps = out[c].sweeps;
        stats[c].relres = b2 > 0.0 ? std::sqrt(r2 / b2) : 0.0;
        stats[c].converged = conv ? 1 : 0;
        e.last_iters += out[c].iters;
    }
    return notconv;
}

}  // namespace tmi
