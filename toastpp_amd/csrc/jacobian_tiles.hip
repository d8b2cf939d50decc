// Nodal-basis Jacobian on the FP64 matrix cores: GenerateJacobian_mesh
// (jacobian.cc:441-497) and its CW form (:727-790) for meshes whose rows hold
// at most 32 neighbours, where jacobian_tiles_pay (jacobian_kernels.hip) finds
// it the faster kernel.
//
// Per node i and link (q, m) the PMDFs are f_q^T A_i g_m and f_q^T B_i g_m
// over the neighbours of i (jacobian_kernels.hip states A_i and B_i).  A
// workgroup takes one kind (A or B), 16 sources x 16 detectors and a run of
// consecutive nodes; each of its computing waves takes every eighth node:
//   H = A_i G   (neighbours x detectors, G the adjoint fields)
//   P = F H     (sources x detectors,    F the direct fields)
// with v_mfma_f64_16x16x4.  Lane l of an operand holds row or column l % 16 at
// k = l / 16, register t of a result row l / 16 + 4t of column l % 16: register
// t of H is the k-step t operand of P, so that the chain stays in registers;
// F and G are read from the node-major fields in the operand's own layout (16
// lanes per 256-byte run), A_i and B_i from a plan of the mesh in the same.
//
// What bounds it is J's writes.  J has 4 nq nm rows of n doubles, whose starts
// have any 8-byte alignment when n is odd, and a 128-byte line written in parts
// costs several times a whole one: 3.4 GB of J (103,640 nodes, 32 x 32 links)
// written in pieces of 16 nodes take 1.8 ms at any place, 1.04 ms as 64-byte
// halves of lines, 0.65 ms as lines.  So the results go to a ring of two lines
// per row in LDS, at the row's own place within its lines, and every 16 nodes
// four waves that do nothing else write the one line per row that is complete;
// only the two ends of a run are written in parts.  Writers of their own,
// because a wait for loads also waits for the stores that a wave issued
// before them: with every wave storing its share the kernel took 4.0 ms.
//
// Measured (103,267 nodes, 32 x 32 links): 1.67 ms against 2.99 ms of the
// per-node kernel; without its stores 1.16 ms, of which the matrix
// instructions are 0.52 ms.  31,525 nodes with 2 x 2 links: 0.100 against
// 0.276 ms.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>

#include "fe_integrals.hpp"
#include "jacobian.hpp"

namespace tmi {

typedef double jt_v4 __attribute__((ext_vector_type(4)));
typedef double jt_v2 __attribute__((ext_vector_type(2)));

// a barrier for what is in LDS: global loads and stores stay in flight
__device__ inline void jt_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

constexpr size_t JT_OPS_BYTES = (size_t)1 << 30;
constexpr int JT_WAVES = 8, JT_NT = 64 * (JT_WAVES + 4);   // computing waves (and four writers), threads
constexpr int JT_LINE = 16;                                // doubles of a 128-byte line: nodes per step

struct JtArgs {
    int n, lo, hi, nq, nm, nqm, ldd, lda, tq, tm, nkind, kind0, len, logscale;   // nodes lo .. hi-1
    const int *rowptr, *colidx;
    const double *ops;                   // of node lo onwards: k_jac_ops
    const double2 *dphi, *aphi;
    const int *lk;                       // [nq][nm] link or -1
    const double *proj;
    double *J, *Jkap;                    // CW: the mua and the kappa block
};

// A_i and B_i of the nodes lo .. hi-1 as k_jac_tiles' operands: per node, kind,
// k-step s and tile j a run of 64 doubles, lane l's being entry (4s + l / 16,
// 16j + l % 16).  A wave per node; lane (element, a, b) takes four elements at
// a time and adds them to the matrices in LDS one after the other.
template <int DIM, int JT>
__global__ void __launch_bounds__(256) k_jac_ops(int lo, int hi, const int *__restrict__ rowptr,
                                                 const int *__restrict__ colidx, const int *__restrict__ n2e_ptr,
                                                 const int *__restrict__ n2e, const int *__restrict__ el,
                                                 const double *__restrict__ geo, double *__restrict__ ops)
{
    constexpr int NN = DIM + 1, GS = DIM == 3 ? GEO3 : GEO2, LD = 16 * JT, SZ = LD * LD;
    __shared__ double mat[4][2][SZ];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), i = lo + blockIdx.x * 4 + wave;
    if (i >= hi) return;
    const int l = threadIdx.x & 63, lr = l & 15, lq = l >> 4, ia = lr / NN, ib = lr % NN;
    double *am = mat[wave][0], *bm = mat[wave][1];
    for (int t = l; t < 2 * SZ; t += 64) am[t] = 0.0;
    const int rb = rowptr[i], re = rowptr[i + 1], e1 = n2e_ptr[i + 1];
    auto place = [&](int v) {
        int a = rb, b = re - 1;
        while (a < b) {
            const int mid = (a + b) >> 1;
            if (colidx[mid] < v) a = mid + 1;
            else b = mid;
        }
        return a - rb;
    };
    for (int p = n2e_ptr[i]; p < e1; p += 4) {
        const bool on = p + lq < e1 && lr < NN * NN;
        double a = 0.0, b = 0.0;
        int at = 0;
        if (on) {
            const int e = n2e[p + lq];
            const int *nd = el + (long)NN * e;
            const double *g = geo + (long)GS * e;
            int li = 0;
            for (int k = 1; k < NN; k++) li = nd[k] == i ? k : li;
            a = DIM == 3 ? tet_intfff(g, li, ia, ib) : tri_intfff(g, li, ia, ib);
            b = DIM == 3 ? tet_intfdd(g, ia, ib) : tri_intfdd(g, ia, ib);
            at = place(nd[ia]) * LD + place(nd[ib]);
        }
        for (int e = 0; e < 4; e++) {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            if (on && lq == e) {
                am[at] += a;
                bm[at] += b;
            }
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    double *o = ops + (size_t)(i - lo) * 2 * SZ + l;
    for (int k = 0; k < 2; k++)
        for (int s = 0; s < 4 * JT; s++)
            for (int j = 0; j < JT; j++)
                o[k * SZ + (s * JT + j) * 64] = mat[wave][k][(4 * s + lq) * LD + 16 * j + lr];
}

// KS: steps of four neighbours (2: up to 8, 4: up to 16, 8: up to 32)
template <bool CW, int KS>
__global__ void __launch_bounds__(JT_NT, 3) k_jac_tiles(JtArgs A)
{
    constexpr int JT = (KS + 3) / 4, SZ = 256 * JT * JT;   // tiles of neighbours, entries of an operand
    constexpr int PARTS = CW ? 1 : 2, ROWS = 256 * PARTS;
    extern __shared__ double lds[];
    double *ring = lds;                               // [ROWS][2 JT_LINE], row = (part, source, detector)
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l = tid & 63, lr = l & 15, lq = l >> 4;
    // the workgroups of one run of nodes read the same fields: they go to one XCD
    const int b = blockIdx.x, x = b & 7, tot = gridDim.x;
    int g = x * (tot >> 3) + min(x, tot & 7) + (b >> 3);
    const int kind = A.kind0 + g % A.nkind;
    g /= A.nkind;
    const int m0 = 16 * (g % A.tm);
    g /= A.tm;
    const int q0 = 16 * (g % A.tq), i0 = A.lo + g / A.tq * A.len, i1 = min(A.hi, i0 + A.len), cnt = i1 - i0;
    const size_t ld = CW ? (size_t)A.n : 2 * (size_t)A.n;
    double *const Jk = (CW ? (kind ? A.Jkap : A.J) : A.J + (size_t)kind * A.n) + i0;
    auto link = [&](int q, int m) { return q < A.nq && m < A.nm ? A.lk[(size_t)q * A.nm + m] : -1; };
    bool any = false;
#pragma unroll
    for (int t = 0; t < 4; t++) any |= link(q0 + lq + 4 * t, m0 + lr) >= 0;
    if (!__any(any)) return;                          // no link in this tile (every wave holds the same pairs)

    if (wave >= JT_WAVES) {
        // a writer: two doubles of a line of each of its rows a step
        constexpr int LPR = JT_LINE / 2, RS = (JT_NT - 64 * JT_WAVES) / LPR, SW = ROWS / RS;
        const int w = tid - 64 * JT_WAVES, r0 = w / LPR, pr = 2 * (w % LPR);
        int row[SW];
#pragma unroll
        for (int s = 0; s < SW; s++) {
            const int r = s * RS + r0, k = link(q0 + ((r & 255) >> 4), m0 + (r & 15));
            row[s] = k < 0 ? -1 : k + (r >> 8) * A.nqm;
        }
        for (int c0 = 0; c0 < cnt; c0 += JT_LINE) {
            const int end = min(cnt, c0 + JT_LINE);
            jt_barrier();                             // the ring holds this step's nodes
            for (int c = c0; c <= (end < cnt ? c0 : c0 + JT_LINE); c += JT_LINE) {
                jt_v2 v[SW];
#pragma unroll
                for (int s = 0; s < SW; s++) {
                    const int r = s * RS + r0;
                    v[s] = *(const jt_v2 *)(ring + r * (2 * JT_LINE) + (((c & JT_LINE) + pr) ^ ((r & 15) << 1)));
                }
                if (c == c0) jt_barrier();         // the ring may take the next step's
#pragma unroll
                for (int s = 0; s < SW; s++) {
                    if (row[s] < 0) continue;
                    double *p = Jk + (size_t)row[s] * ld;
                    const int o = c + pr - (int)(((size_t)p >> 3) & (JT_LINE - 1));   // node of the run at v[s].x
                    p += o;
                    if (o >= 0 && o + 1 < end) {
                        __builtin_nontemporal_store(v[s], (jt_v2 *)p);
                    } else {
                        if (o >= 0 && o < end) p[0] = v[s].x;
                        if (o + 1 >= 0 && o + 1 < end) p[1] = v[s].y;
                    }
                }
            }
        }
        return;
    }

    // this lane's four pairs (q0 + lq + 4t, m0 + lr): scale -1/proj and the
    // rows' places within their lines
    double2 sc[4];
    unsigned shift = 0;
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const int k = link(q0 + lq + 4 * t, m0 + lr);
        sc[t] = make_double2(-1.0, 0.0);
        if (k < 0) continue;
        if (A.logscale) {
            if (CW) {
                sc[t].x = -(1.0 / A.proj[k]);
            } else {
                const double2 p = ((const double2 *)A.proj)[k];
                const double den = p.x * p.x + p.y * p.y;
                sc[t] = make_double2(-(p.x / den), p.y / den);
            }
        }
#pragma unroll
        for (int c = 0; c < PARTS; c++)
            shift |= (unsigned)(((size_t)(Jk + ((size_t)k + (size_t)c * A.nqm) * ld) >> 3) & (JT_LINE - 1))
                     << (4 * (2 * t + c));
    }
    // past the last source or detector a lane repeats it (its pairs are not
    // written); past the last neighbour too (A_i is zero there)
    const int qc = min(q0 + lr, A.nq - 1), mc = min(m0 + lr, A.nm - 1);

    // what the wave holds of its node: the operands A_i, G, F and H.  The
    // neighbours of the nodes after it are read ahead, a lane holding one
    // (lane / NL), and a word of every line of the second next node's fields
    // and A_i: under J's writes a line from beyond the L2 takes longer than a
    // step, one from the L2 does not
    constexpr int NL = 4 / JT;
    int col[KS], d, d1, d2, d3, c1, c2, c3;
    float seen_f = 0.0f, seen_a = 0.0f;
    double2 f[KS], gv[KS];
    double am[KS][JT];
    jt_v4 hr[JT], hi[JT];
    auto neighbours = [&](int i, int &dn) {
        const int rb = A.rowptr[i];
        dn = A.rowptr[i + 1] - rb;
        return dn ? A.colidx[rb + min(l / NL, dn - 1)] : 0;
    };
    auto touch = [&](int i, int c) {
        asm volatile("" ::"v"(seen_f), "v"(seen_a));
        const int part = l % NL;
        const double2 *pf = part < NL / 2 ? A.aphi + (size_t)c * A.lda + min(m0 + 8 * part, A.nm - 1)
                                          : A.dphi + (size_t)c * A.ldd + min(q0 + 8 * (part - NL / 2), A.nq - 1);
        seen_f = *(const float *)pf;
        seen_a = *(const float *)(A.ops + (size_t)(i - A.lo) * 2 * SZ + min(16 * l, 2 * SZ - 1));
    };
    auto take = [&]() {
        d = d1;
#pragma unroll
        for (int s = 0; s < KS; s++) col[s] = __shfl(c1, NL * (4 * s + lq));
    };
    auto load_ag = [&](int i) {
        const double *o = A.ops + ((size_t)(i - A.lo) * 2 + kind) * SZ + l;
#pragma unroll
        for (int s = 0; s < KS; s++) {
#pragma unroll
            for (int j = 0; j < JT; j++) am[s][j] = o[(s * JT + j) * 64];
            gv[s] = A.aphi[(size_t)col[s] * A.lda + mc];
        }
    };
    auto load_f = [&]() {
#pragma unroll
        for (int s = 0; s < KS; s++) f[s] = A.dphi[(size_t)col[s] * A.ldd + qc];
    };
    // H = A_i G (A_i is symmetric)
    auto product_h = [&]() {
#pragma unroll
        for (int j = 0; j < JT; j++) hr[j] = hi[j] = jt_v4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int s = 0; s < KS; s++) {
            if (KS > 4 && 4 * s >= d) break;
#pragma unroll
            for (int j = 0; j < JT; j++) {
                hr[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(am[s][j], gv[s].x, hr[j], 0, 0, 0);
                if (!CW) hi[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(am[s][j], gv[s].y, hi[j], 0, 0, 0);
            }
        }
    };
    // (nodes past the run's last repeat it; what they leave in the ring is
    // not written)
    auto node = [&](int c) { return i0 + min(c + wave, cnt - 1); };
    c1 = neighbours(node(0), d1);
    c2 = neighbours(node(JT_WAVES), d2);
    c3 = neighbours(node(2 * JT_WAVES), d3);
    take();
    load_ag(node(0));
    load_f();
    c1 = c2; d1 = d2;
    c2 = c3; d2 = d3;
    touch(node(JT_WAVES), c1);
    product_h();

    // one node's products into the ring, and what comes next
    auto step = [&](int c0) {
        const int dc = d;
        take();
        load_ag(node(c0 + JT_WAVES));
        touch(node(c0 + 2 * JT_WAVES), c2);
        c3 = neighbours(node(c0 + 3 * JT_WAVES), d3);
        c1 = c2; d1 = d2;
        // P = F H
        jt_v4 vr = {0.0, 0.0, 0.0, 0.0}, vi = vr;
#pragma unroll
        for (int s = 0; s < KS; s++) {
            if (KS > 4 && 4 * s >= dc) break;
            const double br = hr[s / 4][s % 4], bi = hi[s / 4][s % 4];
            vr = __builtin_amdgcn_mfma_f64_16x16x4f64(f[s].x, br, vr, 0, 0, 0);
            if (CW) continue;
            vi = __builtin_amdgcn_mfma_f64_16x16x4f64(f[s].x, bi, vi, 0, 0, 0);
            vr = __builtin_amdgcn_mfma_f64_16x16x4f64(-f[s].y, bi, vr, 0, 0, 0);
            vi = __builtin_amdgcn_mfma_f64_16x16x4f64(f[s].y, br, vi, 0, 0, 0);
        }
        load_f();
        c2 = c3; d2 = d3;
        // into the ring; the places of a row are permuted by the row so that
        // the 16 rows of a register do not meet in one bank
        const int u = c0 + wave, swz = lr << 1;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const double a = vr[t], c = vi[t];
            double *at = ring + (l + 64 * t) * (2 * JT_LINE);
            const int ur = ((u + (shift >> (8 * t) & (JT_LINE - 1))) & (2 * JT_LINE - 1)) ^ swz;
            if (CW) {
                at[ur] = a * sc[t].x;
            } else {
                const int ui = ((u + (shift >> (8 * t + 4) & (JT_LINE - 1))) & (2 * JT_LINE - 1)) ^ swz;
                at[ur] = a * sc[t].x - c * sc[t].y;
                at[256 * 2 * JT_LINE + ui] = a * sc[t].y + c * sc[t].x;
            }
        }
    };
    for (int c0 = 0; c0 < cnt; c0 += JT_LINE) {
        step(c0);
        product_h();
        step(c0 + JT_WAVES);
        jt_barrier();
        product_h();   // the next node's, while the writers read the ring
        jt_barrier();
    }
}

// tiles of neighbours a side, and bytes of a node's operands (4 KB up to 16
// neighbours, 16 KB up to 32)
static int jt_of(int dmax) { return dmax <= 16 ? 1 : 2; }
static size_t jt_node_bytes(int dmax) { return 2 * 256 * sizeof(double) * jt_of(dmax) * jt_of(dmax); }

bool jacobian_tiles_whole(const Mesh &m, int dmax) { return (size_t)m.n <= JT_OPS_BYTES / jt_node_bytes(dmax); }

bool launch_jacobian_tiles(Mesh &m, int nq, int nm, const double *d_dphi, int ldd, const double *d_aphi, int lda,
                           int nqm, const double *d_proj, int logscale, double *d_J, int dmax, hipStream_t st, bool cw,
                           double *d_Jkap)
{
    JtArgs a{};
    a.n = m.n; a.nq = nq; a.nm = nm; a.nqm = nqm; a.ldd = ldd; a.lda = lda;
    a.tq = (nq + 15) / 16; a.tm = (nm + 15) / 16;
    a.kind0 = cw && !d_J ? 1 : 0;
    a.nkind = cw && (!d_J || !d_Jkap) ? 1 : 2;
    a.logscale = logscale;
    a.rowptr = m.rowptr.p; a.colidx = m.colidx.p;
    a.dphi = (const double2 *)d_dphi; a.aphi = (const double2 *)d_aphi;
    a.lk = m.d_lk.p; a.proj = d_proj; a.J = d_J; a.Jkap = d_Jkap;
    const int jt = jt_of(dmax);
    // the operands of all nodes are kept with the mesh up to JT_OPS_BYTES;
    // beyond, they are made for a part of the nodes at a time, on each call
    const size_t per = jt_node_bytes(dmax);
    const int part = (int)std::min<size_t>(m.n, JT_OPS_BYTES / per);
    const bool whole = part == m.n;
    std::unique_lock<std::mutex> lock(m.jac_mu);
    if (m.jac_ops.n * sizeof(double) < part * per) {
        try {
            m.jac_ops.alloc(part * per / sizeof(double));
        } catch (const Error &err) {
            if (err.code != TMI_ERR_OOM) throw;
            return false;   // the per-node kernel needs none
        }
    }
    const size_t lds = (size_t)256 * (cw ? 1 : 2) * 2 * JT_LINE * sizeof(double);
    const long units = (long)a.tq * a.tm * a.nkind;
    for (int lo = 0; lo < m.n; lo += part) {
        const int nn = std::min(part, m.n - lo);
        if (!whole || !m.jac_ops_ok) {
#define JTO(D, T)                                                                                                     \
    hipLaunchKernelGGL((k_jac_ops<D, T>), dim3((nn + 3) / 4), dim3(256), 0, st, lo, lo + nn, m.rowptr.p, m.colidx.p, \
                       m.n2e_ptr.p, m.n2e.p, m.elist.p, m.geo.p, m.jac_ops.p);
            if (m.dim == 3) { if (jt == 1) JTO(3, 1) else JTO(3, 2) }
            else { if (jt == 1) JTO(2, 1) else JTO(2, 2) }
#undef JTO
            TMI_LAUNCH_CHECK();
            if (whole) {
                TMI_HIP(hipStreamSynchronize(st));   // other streams may read them from here on
                m.jac_ops_ok = true;
            }
        }
        // runs of equal length such that the workgroups, one per CU, fill
        // whole rounds; a run is at least a line of nodes, so that at most every
        // other line is written in parts
        const long slots = 256, most = (nn + JT_LINE - 1) / JT_LINE;
        long runs = 1;
        double best = 0.0;
        for (int w = 1; w <= 4; w++) {
            const long r = std::max(1L, std::min(most, w * slots / units)), wg = r * units;
            const double full = (double)wg / (double)((wg + slots - 1) / slots * slots);
            if (full > best + 0.02) { best = full; runs = r; }
        }
        a.lo = lo; a.hi = lo + nn; a.ops = m.jac_ops.p;
        a.len = (int)(((nn + runs - 1) / runs + JT_LINE - 1) / JT_LINE * JT_LINE);
        runs = (nn + a.len - 1) / a.len;
        const long grid = runs * units;
        TMI_CHECK(grid < (1L << 31), TMI_ERR_UNSUPPORTED, "nodal Jacobian: %ld workgroups", grid);
#define JTL(C, T) hipLaunchKernelGGL((k_jac_tiles<C, T>), dim3((unsigned)grid), dim3(JT_NT), lds, st, a);
        if (jt == 2) { if (cw) JTL(true, 8) else JTL(false, 8) }
        else if (dmax > 8) { if (cw) JTL(true, 4) else JTL(false, 4) }
        else { if (cw) JTL(true, 2) else JTL(false, 2) }
#undef JTL
        TMI_LAUNCH_CHECK();
    }
    // the parts' operands are shared: the next call's stream may be another
    if (!whole) TMI_HIP(hipStreamSynchronize(st));
    return true;
}

}  // namespace tmi
