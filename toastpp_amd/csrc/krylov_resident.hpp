// Resident Krylov solve: the whole iteration of a block of right-hand sides
// in one cooperative kernel, for systems whose Krylov vectors fit the
// registers and the LDS of the chip.
//
// A launch sequence pays, per iteration, five dependent kernels (25-30 us at
// a few thousand to 30k nodes, where the data of an iteration moves in 2-5
// us), and streams every Krylov vector through memory.  Here one 512-thread
// workgroup per CU owns a fixed set of rows for the whole solve: x, r and the
// SpMM result of its elements stay in registers, the direction p in LDS;
// only the vector the next SpMM gathers is published to memory, and the
// inner products travel through stamped words.
//
// Teams: the workgroups form T teams of nr = 256/T ranks; team t owns kc
// consecutive columns, rank r of a team a contiguous range of rows (ResLayout,
// built on the GPU once per mesh order and nr).  Workgroup b runs on XCD
// b % 8 and takes the logical id (b % 8) 32 + b / 8, so a team of up to 32
// ranks shares one XCD and a wider one whole XCDs.  Teams never exchange
// anything: each runs until its own columns are done.
//
// SpMM: a rank's rows and the rows they couple to (its halo) are staged in
// LDS: own rows are written there by their owner, halo rows loaded from the
// published vector, so each neighbour row crosses the memory system once per
// rank and SpMM instead of once per nonzero (gathers per nonzero run at about
// 9 TB/s over the whole chip however they are laid out; a rank of 123 rows of
// a tetrahedral mesh has 1845 nonzeros and about 280 halo rows, one of 977
// rows 14.7k and 750).  The matrix is stored in slices of 8 rows (rows of a
// rank sorted by length, slice entries interleaved by row, padded with zeros
// to a multiple of 4) with 16-bit local columns; a lane takes CL consecutive
// columns of a row, so an entry is loaded once for them.
//
// Memory model: every word one workgroup writes and another reads (published
// vectors, partial sums) is accessed by relaxed agent-scope atomics only,
// which bypass the non-coherent L1 and are coherent between the XCDs (as fast
// as plain loads in a gather test, where an agent acquire fence cost 28 us);
// the placement above affects speed, not results.  Order: a wave waits for
// its published stores (vmcnt 0) before the workgroup barrier after which the
// workgroup's stamped words are written, and a reader consumes the vector
// only after it has seen the stamps of every rank.  A double travels as two
// 8-byte words, each holding half of it and the 32-bit stamp of its
// reduction, so a word is valid by itself once its stamp matches.  Slots
// alternate between two parities: a rank can write a slot again only after
// the reduction in between, which needs every rank's words, i.e. every rank
// has read the earlier ones.
//
// Every wait is bounded (RES_TIMEOUT ticks of the 100 MHz counter and a
// shared abort word): a rank that gives up sets the abort word, the others
// see it in their polls, and the kernel ends.  Columns of teams that had
// finished are then written, rows of the others hold their initial guesses
// (or, where only some ranks saw the abort at the very end, solutions): a
// start for the launch sequence, which the host then runs.
//
// The arithmetic per element and the per-column recurrences (fin_column) are
// the launch sequence's; sums over rows are grouped by thread, wave, rank in
// a fixed order, so results are reproducible run to run.
#pragma once
#include "krylov_device.hpp"

namespace tmi {

constexpr int RES_NT = 512;           // threads per workgroup, one workgroup per CU
constexpr int RES_WAVES = RES_NT / 64;
constexpr int RES_KC = 16;            // columns per team, at most (a power of two)
constexpr int RES_SLOTS = 4;          // sums per column of one reduction, at most
constexpr int RES_WG = 256;           // workgroups (one per CU of the chip)
constexpr size_t RES_LDS = 160 * 1024;
constexpr unsigned long long RES_TIMEOUT = 400000000ull;   // 4 s of the 100 MHz counter

typedef unsigned long long res_u64;

// Stamped words of a team: per parity one line of RES_LINE words for every
// rank ([output][2]), then one for every group of RES_GROUP ranks; padded so
// that the teams' lines do not share a memory channel.
constexpr int RES_OUT = RES_SLOTS * RES_KC;      // outputs of a reduction, at most
constexpr int RES_LINE = 2 * RES_OUT;
constexpr int RES_GROUP = 16;
constexpr size_t RES_PAD = 544;
__host__ __device__ constexpr size_t res_part_stride(int nr) { return (size_t)RES_LINE * nr + RES_PAD; }
__host__ __device__ constexpr size_t res_tot_stride(int nr) { return (size_t)RES_LINE * (nr / RES_GROUP) + RES_PAD; }
// most over all nr > 1 (rank lines), nr > RES_GROUP (group lines)
constexpr size_t RES_PART_WORDS = 2 * (RES_WG / 2) * res_part_stride(2);
constexpr size_t RES_TOT_WORDS = 2 * (RES_WG / (2 * RES_GROUP)) * res_tot_stride(2 * RES_GROUP);

struct ResColOut {
    double res2, bnorm2;
    int iters, sweeps;
};

struct ResArgs {
    int n, K, kc, nr;                // rows, columns, columns per team, ranks per team
    int maxit, ru;                   // iteration cap; inner iterations between residual replacements
    int mixed;
    int nu;                          // rows of the LDS stage (longest own + halo of a rank)
    double tol2, itol2;
    const int *srow, *node;          // per position: row of the solver's order, mesh node
    const int *sofs;                 // slice bounds (entries)
    const int *rslice;               // first slice of each rank
    const int *hofs, *halo;          // halo rows (positions) of each rank
    const unsigned short *lcol;      // per entry: LDS row
    const int *gcol;                 // per entry: position
    const void *op;                  // inner operator in slice order (BiCGSTAB: K D^-1)
    const double *op64;              // operator of the FP64 residual in slice order
    const void *idiag;               // inverse diagonal, or null; multi-frequency: the diagonal at omega = 1
    const double *omega;             // per column, or null
    const void *b;                   // caller's right-hand sides [n][ld]
    void *x;                         // caller's fields: initial guess in, solution out
    long ld;
    int q0;                          // first column of the block in b and x: 0 (as a constant it costs other
                                     // registers and 4 % of the c64 COCG solve, n 31,525 x 16)
    void *pub_p, *pub_s;             // published vectors [T][n][kc]
    void *x64;                       // FP64 solution [T][n][kc], published
    void *rd0;                       // shadow residual of the FP64 BiCGSTAB [T][n][kc], private to its owner
    res_u64 *part, *tot;             // stamped words
    unsigned epoch;
    int *abort_flag;
    ResColOut *out;                  // per column
};

// ---------------------------------------------------------- published data
__device__ inline float ld_pub(const float *p)
{
    return __builtin_bit_cast(float, __hip_atomic_load((const unsigned *)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}
__device__ inline double ld_pub(const double *p)
{
    return __builtin_bit_cast(double, __hip_atomic_load((const res_u64 *)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}
__device__ inline float2 ld_pub(const float2 *p)
{
    return __builtin_bit_cast(float2, __hip_atomic_load((const res_u64 *)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}
__device__ inline double2 ld_pub(const double2 *p)
{
    return make_double2(ld_pub((const double *)p), ld_pub((const double *)p + 1));
}
__device__ inline void st_pub(float *p, float v)
{
    __hip_atomic_store((unsigned *)p, __builtin_bit_cast(unsigned, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void st_pub(double *p, double v)
{
    __hip_atomic_store((res_u64 *)p, __builtin_bit_cast(res_u64, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void st_pub(float2 *p, float2 v)
{
    __hip_atomic_store((res_u64 *)p, __builtin_bit_cast(res_u64, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void st_pub(double2 *p, double2 v)
{
    st_pub((double *)p, v.x);
    st_pub((double *)p + 1, v.y);
}

// ------------------------------------------------------------ reductions
struct ResTeam {
    int nr, rank, kc, lkc, lpr;      // ranks, this rank, columns, their log2, lanes per row (at most RES_LANES)
    res_u64 *part, *tot;             // this team's words
    size_t pstride, tstride;         // words of one parity
    unsigned stamp;                  // stamp of the last reduction
    int *abort_flag;
    // LDS
    double *red;                     // [slot][CL][RES_LANES][wave]
    double *xch;                     // [RES_GROUP][output]
    double *sum;                     // [slot][column]
    double *S, *O;                   // inner / outer scalars [column][S_NSLOT]
    int *I, *OI;                     // inner / outer flags [column][I_NSLOT + 1]
    int *dead;
};
// bytes of LDS beside the stage
inline __host__ __device__ size_t res_lds_fixed(int kc)
{
    return (size_t)kc * (8 * (RES_SLOTS + 2 * S_NSLOT) + 4 * 2 * (I_NSLOT + 1)) +
           8 * (RES_SLOTS * 4 * 4 * RES_WAVES + RES_GROUP * RES_SLOTS * kc) + 16;
}

__device__ inline void put_word(res_u64 *w, double v, unsigned stamp)
{
    const res_u64 b = __builtin_bit_cast(res_u64, v);
    __hip_atomic_store(w, ((res_u64)stamp << 32) | (b >> 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(w + 1, ((res_u64)stamp << 32) | (b & 0xffffffffull), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// wait for the double of this stamp; 0 and sh.dead set when the wait ends
// without it (timeout, or another rank's abort)
__device__ inline double take_word(const res_u64 *w, unsigned stamp, int *abort_flag, int &dead)
{
    res_u64 a, b, t0 = 0;
    for (unsigned spin = 0;; spin++) {
        a = __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        b = __hip_atomic_load(w + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if ((unsigned)(a >> 32) == stamp && (unsigned)(b >> 32) == stamp) break;
        if ((spin & 255u) == 255u) {
            const res_u64 now = __builtin_amdgcn_s_memrealtime();
            if (t0 == 0) t0 = now;
            if (now - t0 > RES_TIMEOUT)
                __hip_atomic_store(abort_flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (__hip_atomic_load(abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
                dead = 1;
                return 0.0;
            }
        }
    }
    return __builtin_bit_cast(double, (a << 32) | (b & 0xffffffffull));
}

// own published stores complete (every wave, before the workgroup barrier
// that precedes the stamps)
__device__ inline void pub_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// v + (v of the lane ROR lanes on, within rows of 16 lanes)
template <int ROR>
__device__ inline double ror_add(double v)
{
    const long long b = __builtin_bit_cast(long long, v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xffffffffll), 0x120 + ROR, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x120 + ROR, 0xf, 0xf, true);
    return v + __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned)lo);
}
// v of the lower plus v of the upper half of the wave (H = 32), or of the
// even plus the odd rows of 16 lanes (H = 16)
template <int H>
__device__ inline double half_add(double v)
{
    const res_u64 b = __builtin_bit_cast(res_u64, v);
    const unsigned lo = (unsigned)b, hi = (unsigned)(b >> 32);
    if constexpr (H == 32) {
        const auto l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
        const auto h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
        return __builtin_bit_cast(double, ((res_u64)h[0] << 32) | l[0]) + __builtin_bit_cast(double, ((res_u64)h[1] << 32) | l[1]);
    } else {
        const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
        const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
        return __builtin_bit_cast(double, ((res_u64)h[0] << 32) | l[0]) + __builtin_bit_cast(double, ((res_u64)h[1] << 32) | l[1]);
    }
}
// sum over the lanes of the wave that share lane % RES_LANES
constexpr int RES_LANES = 4;
__device__ inline double wave_sum4(double v) { return half_add<32>(half_add<16>(ror_add<4>(ror_add<8>(v)))); }

// Sum NS per-thread values of the thread's CL columns over the team into
// t.sum[slot][column]; also a barrier of the team (the published stores of
// every rank are visible after it).  NS = 0: only the barrier.  false: the
// solve was aborted.
template <int NS, int CL>
__device__ __forceinline__ bool team_sum(ResTeam &t, const double (*d)[CL])
{
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const unsigned stamp = ++t.stamp;
    const int par = stamp & 1;
    const int nout = NS > 0 ? NS * t.kc : 1;
    res_u64 *part = t.part + par * t.pstride;
    res_u64 *tot = t.tot + par * t.tstride;
    pub_done();
    if constexpr (NS > 0) {
#pragma unroll
        for (int s = 0; s < NS; s++)
#pragma unroll
            for (int j = 0; j < CL; j++) {
                const double v = wave_sum4(d[s][j]);
                if (lane < RES_LANES) t.red[((s * CL + j) * RES_LANES + lane) * RES_WAVES + wave] = v;
            }
    }
    __syncthreads();
    if (tid < nout) {
        double mine = 0.0;
        if constexpr (NS > 0) {
            // output (slot, column lr CL + j): lanes lr, lr + lpr, .. of every wave
            const int s = tid >> t.lkc, c = tid & (t.kc - 1), lr = c / CL, j = c - lr * CL;
            for (int l = lr; l < RES_LANES; l += t.lpr) {
                const double *q = t.red + ((s * CL + j) * RES_LANES + l) * RES_WAVES;
#pragma unroll
                for (int w = 0; w < RES_WAVES; w++) mine += q[w];
            }
        }
        if (t.nr > 1) put_word(part + t.rank * RES_LINE + 2 * tid, mine, stamp);
        else if (NS > 0) t.sum[tid] = mine;
    }
    int dead = 0;
    if (t.nr > 1) {
        // Up to RES_GROUP ranks: every workgroup reads every rank's line.
        // More: the first rank of each group of RES_GROUP sums the lines of
        // its group and publishes one, and every workgroup reads those.
        // Measured per reduction of 1 / 12 / 24 outputs: one hop 1.3 / 1.5 /
        // 1.7 us at 16 ranks but 1.9 / 2.1 / 2.2 at 32 and 4.9 / 7.0 / 9.3 at
        // 256 (the polls of all workgroups meet in the same lines), two hops
        // 1.9 / 2.3 / 2.3 at 32 and 2.3 / 2.8 / 2.8 at 256.
        const bool tree = t.nr > RES_GROUP;
        const int ng = t.nr / RES_GROUP, g = t.rank / RES_GROUP;
        if (tree && t.rank % RES_GROUP == 0) {
            const res_u64 *src = part + (size_t)g * RES_GROUP * RES_LINE;
            for (int k = tid; k < nout * RES_GROUP; k += RES_NT) {
                const int r = k / nout, o = k - r * nout;
                t.xch[k] = take_word(src + r * RES_LINE + 2 * o, stamp, t.abort_flag, dead);
            }
            // a rank whose wait ended early publishes nothing
            const bool lost = __syncthreads_or(dead) != 0;
            if (tid < nout && !lost) {
                double v = 0.0;
                for (int r = 0; r < RES_GROUP; r++) v += t.xch[r * nout + tid];
                put_word(tot + g * RES_LINE + 2 * tid, v, stamp);
            }
            __syncthreads();
        }
        const int nl = tree ? ng : t.nr;
        const res_u64 *src = tree ? tot : part;
        for (int k = tid; k < nout * nl; k += RES_NT) {
            const int r = k / nout, o = k - r * nout;
            const double v = take_word(src + r * RES_LINE + 2 * o, stamp, t.abort_flag, dead);
            if constexpr (NS > 0) t.xch[k] = v;
        }
        if constexpr (NS > 0) {
            __syncthreads();
            if (tid < nout) {
                double v = 0.0;
                for (int r = 0; r < nl; r++) v += t.xch[r * nout + tid];
                t.sum[tid] = v;
            }
        }
    }
    if (dead) *t.dead = 1;
    __syncthreads();
    return *t.dead == 0;
}

// the scalar recurrence of every column (threads 0 .. kc-1) from slots
// s0, s1, s2 of the last reduction (-1: not used)
__device__ inline void res_fin(int fk, const ResTeam &t, double *S, int *I, int s0, int s1, int s2, int maxit,
                               double tol2)
{
    const int c = threadIdx.x;
    if (c < t.kc) {
        I += c * (I_NSLOT + 1);
        I[I_NSLOT] = t.OI[c * (I_NSLOT + 1) + I_ACTIVE];
        fin_column(fk, s0 >= 0 ? t.sum[s0 * t.kc + c] : 0.0, s1 >= 0 ? t.sum[s1 * t.kc + c] : 0.0,
                   s2 >= 0 ? t.sum[s2 * t.kc + c] : 0.0, S + c * S_NSLOT, I, maxit, tol2);
    }
}

enum ResMethod { RES_CG = 0, RES_COCG = 1, RES_BICG = 2 };

template <class V> struct WideOf { using type = double; };
template <> struct WideOf<float2> { using type = double2; };
template <> struct WideOf<double2> { using type = double2; };

// v times a real or complex scalar in the vector's own precision
template <class V, class S>
__device__ inline V res_scale(V v, S s)
{
    if constexpr (std::is_same<V, S>::value) return v * s;
    else {
        v.x *= s;
        v.y *= s;
        return v;
    }
}
template <class V, class S>
__device__ inline V res_scale(V v, S a, S b)
{
    V o;
    o.x = v.x * a - v.y * b;
    o.y = v.x * b + v.y * a;
    return o;
}

// E rows (groups) of CL columns per thread; M the Krylov method; MF: each
// column at its own frequency (COCG)
template <class V, int CL, int E, int M, bool MF>
__global__ void __launch_bounds__(RES_NT) k_resident(ResArgs a)
{
    using V64 = typename WideOf<V>::type;
    using S = typename ScalarOf<V>::type;
    using S64 = typename ScalarOf<V64>::type;
    extern __shared__ char dyn[];
    V *stage = (V *)dyn;   // [own rows, then halo rows][kc]
    const int tid = threadIdx.x, kc = a.kc;
    const int logical = (blockIdx.x % 8) * (RES_WG / 8) + blockIdx.x / 8;
    const int team = logical / a.nr, rank = logical % a.nr;
    const int c0 = team * kc;
    if (c0 >= a.K) return;                // an unused team
    const int ncol = min(kc, a.K - c0);   // columns in use; the others stay inactive
    const int lpr = kc / CL, rps = RES_NT / lpr;
    int c = (tid % lpr) * CL;             // this thread's columns c .. c+CL-1
    const int r0 = (int)((long)a.n * rank / a.nr), nrow = (int)((long)a.n * (rank + 1) / a.nr) - r0;
    int i0 = tid / lpr;                   // its rows i0 + e rps of the rank
    const size_t pstride = res_part_stride(a.nr);
    ResTeam tm;
    tm.nr = a.nr; tm.rank = rank; tm.kc = kc; tm.lkc = 31 - __builtin_clz(kc); tm.lpr = lpr;
    tm.part = a.part + (size_t)team * 2 * pstride;
    tm.tstride = res_tot_stride(a.nr);
    tm.tot = a.tot + (size_t)team * 2 * tm.tstride;
    tm.pstride = pstride;
    tm.stamp = a.epoch;
    tm.abort_flag = a.abort_flag;
    {
        double *q = (double *)(dyn + (((size_t)a.nu * kc * sizeof(V) + 15) & ~(size_t)15));
        tm.red = q; q += RES_SLOTS * CL * RES_LANES * RES_WAVES;
        tm.xch = q; q += RES_GROUP * RES_SLOTS * kc;
        tm.sum = q; q += RES_SLOTS * kc;
        tm.S = q; q += kc * S_NSLOT;
        tm.O = q; q += kc * S_NSLOT;
        tm.I = (int *)q;
        tm.OI = tm.I + kc * (I_NSLOT + 1);
        tm.dead = tm.OI + kc * (I_NSLOT + 1);
    }
    const size_t tbase = (size_t)a.n * c0 + (size_t)r0 * kc;   // the rank's rows in the published vectors
    V *P = (V *)a.pub_p + tbase, *Q = (V *)a.pub_s + tbase, *rd0 = (V *)a.rd0 + tbase;
    const V *Pt = (const V *)a.pub_p + (size_t)a.n * c0, *Qt = (const V *)a.pub_s + (size_t)a.n * c0;
    V64 *X = (V64 *)a.x64 + tbase;
    const V64 *Xt = (const V64 *)a.x64 + (size_t)a.n * c0;
    const V *op = (const V *)a.op, *idiag = (const V *)a.idiag;
    const V64 *op64 = (const V64 *)a.op64;
    const int h0 = a.hofs[rank], nh = a.hofs[rank + 1] - h0;
    const double *omg = MF ? a.omega + c0 : nullptr;
    if (tid == 0) *tm.dead = 0;
    for (int s = tid; s < kc * S_NSLOT; s += RES_NT) { tm.S[s] = 0.0; tm.O[s] = 0.0; }
    for (int s = tid; s < kc * (I_NSLOT + 1); s += RES_NT) {
        tm.I[s] = 0;
        tm.OI[s] = s % (I_NSLOT + 1) == I_ACTIVE && s / (I_NSLOT + 1) < ncol;
    }
    // slice entries of this thread's rows
    int eofs[E], elen[E];
#pragma unroll
    for (int e = 0; e < E; e++) {
        const int i = i0 + e * rps;
        eofs[e] = elen[e] = 0;
        if (i < nrow) {
            const int sl = a.rslice[rank] + (i >> 3);
            const int b = a.sofs[sl];
            eofs[e] = b + (i & 7);
            elen[e] = (a.sofs[sl + 1] - b) >> 3;
        }
    }
    V x[E][CL], r[E][CL], y[E][CL];      // correction, residual (or s), SpMM result
    V tv[M == RES_BICG ? E : 1][CL];     // BiCGSTAB: second SpMM result
    V pv[M == RES_BICG ? E : 1][CL];     // ... and the direction (the stage holds s in between)
    unsigned sg = 0;                     // signs of the mixed BiCGSTAB's shadow residual, 4 bits per element
    double d[RES_SLOTS][CL];
#define FOR_E _Pragma("unroll") for (int e = 0; e < E; e++)
#define FOR_J _Pragma("unroll") for (int j = 0; j < CL; j++)
#define ROW(e) (i0 + (e) * rps)
#define ON(e) (ROW(e) < nrow)
#define AT(e) ((size_t)ROW(e) * kc + c)
#define CLEAR_D _Pragma("unroll") for (int s = 0; s < RES_SLOTS; s++) FOR_J d[s][j] = 0.0
// the addresses a phase derives from the thread's rows and columns are
// formed anew: kept across phases and iterations they would take the
// registers that hold the Krylov vectors
#define FRESH asm volatile("" : "+v"(i0), "+v"(c))
#define IN(slot, j) tm.I[(c + (j)) * (I_NSLOT + 1) + (slot)]
#define OUT(slot, j) tm.OI[(c + (j)) * (I_NSLOT + 1) + (slot)]
#define SC(slot, j) tm.S[(c + (j)) * S_NSLOT + (slot)]
#define OSC(slot, j) tm.O[(c + (j)) * S_NSLOT + (slot)]
    auto prec = [&](V di, V v, int j) __attribute__((always_inline)) {
        (void)j;
        return idiag ? prec_apply(di, v, omg, c + j) : v;
    };
    V dg[E];                             // (inverse) diagonal of the rows
    FOR_E dg[e] = idiag && ON(e) ? idiag[a.srow[r0 + ROW(e)]] : vzero<V>();
    auto diag = [&](int e) __attribute__((always_inline)) { return dg[e]; };
    // the shadow residual: the sign pattern of r0 (mixed mode) or r0 itself
    auto shadow = [&](int e, int j) __attribute__((always_inline)) -> V {
        if (a.mixed) {
            const unsigned nib = (sg >> (4 * (e * CL + j))) & 15u;
            if constexpr (std::is_same<V, S>::value) return (V)sh_val(nib & 3u);
            else {
                V v;
                v.x = (S)sh_val(nib & 3u);
                v.y = (S)sh_val(nib >> 2);
                return v;
            }
        }
        return rd0[AT(e) + j];
    };
    // halo rows of a published vector into the stage
    auto load_halo = [&](const V *src) __attribute__((always_inline)) {
        const int tot = nh * kc, lk = 31 - __builtin_clz(kc);   // kc: a power of two
        constexpr int U = 4;
        for (int t = tid; t < tot; t += RES_NT * U) {
            V v[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int tt = min(t + u * RES_NT, tot - 1), h = tt >> lk;
                v[u] = ld_pub(src + (size_t)a.halo[h0 + h] * kc + (tt & (kc - 1)));
            }
#pragma unroll
            for (int u = 0; u < U; u++)
                if (t + u * RES_NT < tot) stage[(size_t)nrow * kc + t + u * RES_NT] = v[u];
        }
        __syncthreads();
    };
    // A times the staged vector for the thread's rows and columns, all rows
    // in step: the entries of NB columns of every row are in flight together
    // (they come from the L2, about 300 ns away, and a CU has only 8 waves
    // here).  Each row adds its entries in ascending column order.
    // The first batch is loaded ahead: once per solve where it holds (nearly)
    // whole rows, else before the barrier that precedes the product.
    constexpr int NB = E >= 4 || (E == 2 && sizeof(V) > 8) ? 4 : E == 2 || sizeof(V) > 8 ? 8 : 16;
    V pa[E][NB];
    int pl[E][NB];
    auto prefetch = [&]() __attribute__((always_inline)) {
        FOR_E
#pragma unroll
            for (int g = 0; g < NB; g += 4) {
                const bool in = g < elen[e];
#pragma unroll
                for (int u = g; u < g + 4; u++) {
                    pa[e][u] = in ? op[eofs[e] + u * 8] : vzero<V>();
                    pl[e][u] = in ? a.lcol[eofs[e] + u * 8] : 0;
                }
            }
    };
    constexpr bool KEEP = E <= 2;
    if (KEEP) prefetch();
    auto products = [&](V (*acc)[CL]) __attribute__((always_inline)) {
        S w[CL];
        FOR_J w[j] = MF ? (S)omg[min(c + j, ncol - 1)] : (S)1;
        FOR_E FOR_J acc[e][j] = vzero<V>();
        FOR_E
#pragma unroll
            for (int u = 0; u < NB; u++) {   // zero past the row's end
                const V *sp = stage + pl[e][u] * kc + c;
                FOR_J acc[e][j] = vmac(acc[e][j], mfc<MF>(pa[e][u], w[j]), sp[j]);
            }
        for (int k = NB; k < elen[0]; k += NB) {   // rows come by falling length
            V aa[E][NB];
            int l[E][NB];
            FOR_E
#pragma unroll
                for (int g = 0; g < NB; g += 4)
                    if (k + g < elen[e]) {   // lengths are multiples of 4
#pragma unroll
                        for (int u = g; u < g + 4; u++) {
                            aa[e][u] = op[eofs[e] + (k + u) * 8];
                            l[e][u] = a.lcol[eofs[e] + (k + u) * 8];
                        }
                    }
            FOR_E
#pragma unroll
                for (int g = 0; g < NB; g += 4)
                    if (k + g < elen[e]) {
#pragma unroll
                        for (int u = g; u < g + 4; u++) {
                            const V *sp = stage + l[e][u] * kc + c;
                            FOR_J acc[e][j] = vmac(acc[e][j], mfc<MF>(aa[e][u], w[j]), sp[j]);
                        }
                    }
        }
    };
    // ---- right-hand side norms, initial guess published
    CLEAR_D;
    FOR_E if (ON(e)) {
        const size_t node = (size_t)a.node[r0 + ROW(e)] * a.ld + a.q0 + c0 + c;
        FOR_J if (c + j < ncol) {
            const V64 b = ((const V64 *)a.b)[node + j];
            d[0][j] += dotR(b, b);
            st_pub(X + AT(e) + j, ((const V64 *)a.x)[node + j]);
        }
    }
    __syncthreads();
    if (!team_sum<1, CL>(tm, d)) return;
    res_fin(FIN_OUTER_BNORM, tm, tm.O, tm.OI, 0, -1, -1, 0, 0.0);
    __syncthreads();
    constexpr int NRES = M == RES_COCG ? 4 : 3;
    enum { T_NONE, T_INIT, T_REPLACE, T_FINAL };
    int todo = T_INIT, it = 0, nupd = 0, since = 0;
    bool capped = false;
    FOR_E FOR_J {
        x[e][j] = r[e][j] = y[e][j] = vzero<V>();
        if (ON(e)) stage[AT(e) + j] = vzero<V>();
        if constexpr (M == RES_BICG) pv[e][j] = tv[e][j] = vzero<V>();
    }
    for (;;) {
        if (todo != T_NONE) {
            // the FP64 residual b - A x64 of the outer-active columns into r,
            // scaled by 1/||b||: to start the iteration (T_INIT), as the
            // reliable update (T_REPLACE), or to record the end of columns
            // still active (T_FINAL: FP64 modes, iteration cap); the latter
            // two first fold x into x64 and publish it
            const bool init = todo == T_INIT;
            FRESH;
            if (!init) {
                FOR_E if (ON(e)) FOR_J if (OUT(I_ACTIVE, j)) {
                    const double inv = 1.0 / OSC(S_SCALE, j);
                    V64 *xp = X + AT(e) + j;
                    st_pub(xp, vadd(ld_pub((const V64 *)xp), vscale(to64(x[e][j]), inv)));
                }
                if (!team_sum<0, CL>(tm, d)) return;
            }
            // sums: ||b - A x||^2, then the inner ones
            FRESH;
            CLEAR_D;
            bool any = false;
            FOR_J any |= OUT(I_ACTIVE, j) != 0;
            if (any) FOR_E if (ON(e)) {
                const size_t node = (size_t)a.node[r0 + ROW(e)] * a.ld + a.q0 + c0 + c;
                V64 s[CL];
                S64 w[CL];
                FOR_J { s[j] = vzero<V64>(); w[j] = MF ? (S64)omg[min(c + j, ncol - 1)] : (S64)1; }
                const V64 *vp = op64 + eofs[e];
                const int *gp = a.gcol + eofs[e];
                for (int k = 0; k < elen[e]; k += 4) {
                    V64 aa[4], xx[4][CL];
                    int g[4];
#pragma unroll
                    for (int u = 0; u < 4; u++) { aa[u] = vp[(k + u) * 8]; g[u] = gp[(k + u) * 8]; }
#pragma unroll
                    for (int u = 0; u < 4; u++) FOR_J xx[u][j] = ld_pub(Xt + (size_t)g[u] * kc + c + j);
#pragma unroll
                    for (int u = 0; u < 4; u++) FOR_J s[j] = vmac(s[j], mfc<MF>(aa[u], w[j]), xx[u][j]);
                }
                const V di = diag(e);
                FOR_J if (OUT(I_ACTIVE, j)) {
                    const V64 t = vsub(((const V64 *)a.b)[node + j], s[j]);
                    d[0][j] += dotR(t, t);
                    const V v = cvt<V>(vscale(t, OSC(S_SCALE, j)));
                    r[e][j] = v;
                    x[e][j] = vzero<V>();
                    if constexpr (M == RES_BICG) {
                        if (init) {
                            if (a.mixed) {
                                unsigned code;
                                if constexpr (std::is_same<V, S>::value) code = sh_code((float)v);
                                else code = sh_code((float)v.x) | (sh_code((float)v.y) << 2);
                                sg |= code << (4 * (e * CL + j));
                            } else {
                                rd0[AT(e) + j] = v;
                            }
                        }
                        d[1][j] += dotR(v, v);
                        d[2][j] += dotR(shadow(e, j), v);
                    } else if constexpr (M == RES_COCG) {
                        bil_add(v, prec(di, v, j), d[1][j], d[2][j]);
                        d[3][j] += dotR(v, v);
                    } else {
                        d[1][j] += dotR(v, v);
                        d[2][j] += dotR(v, prec(di, v, j));
                    }
                }
            }
            if (!team_sum<NRES, CL>(tm, d)) return;
            res_fin(FIN_OUTER_RES, tm, tm.O, tm.OI, 0, -1, -1, 0, a.tol2);
            if (todo == T_FINAL) break;
            if (init && tid < kc) {
                tm.I[tid * (I_NSLOT + 1) + I_ACTIVE] = tm.OI[tid * (I_NSLOT + 1) + I_ACTIVE];
                tm.I[tid * (I_NSLOT + 1) + I_FIRST] = 1;
                tm.S[tid * S_NSLOT + S_TOL2] = a.itol2;
            }
            if constexpr (M == RES_COCG)
                res_fin(init ? FIN_COCG_INIT : FIN_COCG_RELIABLE, tm, tm.S, tm.I, 1, 2, 3, a.maxit, 0.0);
            else if constexpr (M == RES_CG)
                res_fin(init ? FIN_CG_INIT : FIN_CG_RELIABLE, tm, tm.S, tm.I, init ? 2 : 1, init ? 1 : 2, -1, a.maxit,
                        0.0);
            else
                res_fin(init ? FIN_BICG_INIT : FIN_BICG_RELIABLE, tm, tm.S, tm.I, 1, 2, -1, a.maxit, 0.0);
            if (!init) nupd++;
            since = 0;
            todo = T_NONE;
        }
        const int oany = tid < kc && tm.OI[min(tid, kc - 1) * (I_NSLOT + 1) + I_ACTIVE];
        const int iany = tid < kc && tm.I[min(tid, kc - 1) * (I_NSLOT + 1) + I_ACTIVE];
        if (!__syncthreads_or(oany)) break;
        if (!__syncthreads_or(iany)) {
            // every recursive residual met the tolerance: the FP64 modes stop
            // here (as the reference does), the mixed mode verifies in FP64
            // (once more at the iteration cap, as the launch sequence does)
            todo = !a.mixed || capped ? T_FINAL : T_REPLACE;
            capped = it >= a.maxit;
            continue;
        }
        if (it >= a.maxit) {
            todo = T_FINAL;
            continue;
        }
        it++;
        const bool due = ++since >= a.ru;
        // ---- direction: into the stage and published
        FRESH;
        {
            bool act[CL], first[CL];
            S br[CL], bi[CL], om[CL];
            FOR_J {
                act[j] = IN(I_ACTIVE, j) != 0;
                first[j] = IN(I_FIRST, j) != 0;
                br[j] = (S)SC(S_BETA, j);
                bi[j] = M == RES_COCG ? (S)SC(S_BETA_I, j) : (S)0;
                om[j] = M == RES_BICG ? (S)SC(S_OMEGA, j) : (S)0;
            }
            FOR_E if (ON(e)) {
                const V di = diag(e);
                V *sp = stage + AT(e), *pp = P + AT(e);
                FOR_J {
                    V p;
                    if constexpr (M == RES_COCG) {
                        const V z = prec(di, r[e][j], j);
                        p = first[j] ? z : vadd(res_scale(sp[j], br[j], bi[j]), z);
                    } else if constexpr (M == RES_CG) {
                        const V z = prec(di, r[e][j], j);
                        p = first[j] ? z : vadd(res_scale(sp[j], br[j]), z);
                    } else {
                        p = first[j] ? r[e][j]
                                     : vadd(r[e][j], res_scale(vsub(pv[e][j], res_scale(y[e][j], om[j])), br[j]));
                    }
                    if constexpr (M == RES_BICG) {
                        // the stage holds s of the last iteration: an idle
                        // column's p goes back too, for its product below
                        if (act[j]) pv[e][j] = p;
                        else p = pv[e][j];
                        sp[j] = p;
                        if (act[j] && a.nr > 1) st_pub(pp + j, p);
                    } else if (act[j]) {
                        sp[j] = p;
                        if (a.nr > 1) st_pub(pp + j, p);
                    }
                }
            }
        }
        if (!KEEP) prefetch();
        if (!team_sum<0, CL>(tm, d)) return;
        if (a.nr > 1) load_halo(Pt);
        // ---- y = A p and its product
        FRESH;
        // (an idle column's p is unchanged, here and where it is published, so
        // its product is too: BiCGSTAB needs it if the column runs on after a
        // residual replacement)
        CLEAR_D;
        products(y);
        FOR_E if (ON(e)) {
            const V *sp = stage + AT(e);
            FOR_J {
                if constexpr (M == RES_COCG) bil_add(sp[j], y[e][j], d[0][j], d[1][j]);
                else if constexpr (M == RES_CG) d[0][j] += dotR(sp[j], y[e][j]);
                else d[0][j] += dotR(shadow(e, j), y[e][j]);
            }
        }
        if constexpr (M == RES_BICG) {
            if (!team_sum<1, CL>(tm, d)) return;
            res_fin(FIN_BICG_ALPHA, tm, tm.S, tm.I, 0, -1, -1, 0, 0.0);
            __syncthreads();
            FRESH;
            bool act[CL];
            S al[CL];
            FOR_J {
                act[j] = IN(I_ACTIVE, j) != 0;
                al[j] = (S)SC(S_ALPHA, j);
            }
            FOR_E if (ON(e)) {
                V *sp = stage + AT(e), *qp = Q + AT(e);
                FOR_J if (act[j]) {
                    const V s = vsub(r[e][j], res_scale(y[e][j], al[j]));
                    r[e][j] = s;
                    sp[j] = s;
                    if (a.nr > 1) st_pub(qp + j, s);
                }
            }
            if (!KEEP) prefetch();
            if (!team_sum<0, CL>(tm, d)) return;
            if (a.nr > 1) load_halo(Qt);
            FRESH;
            CLEAR_D;
            products(tv);
            FOR_E if (ON(e)) FOR_J {
                d[0][j] += dotR(r[e][j], tv[e][j]);
                d[1][j] += dotR(tv[e][j], tv[e][j]);
            }
            if (!team_sum<2, CL>(tm, d)) return;
            res_fin(FIN_BICG_OMEGA, tm, tm.S, tm.I, 0, 1, -1, 0, 0.0);
            __syncthreads();
            FRESH;
            CLEAR_D;
            S om[CL];
            FOR_J om[j] = (S)SC(S_OMEGA, j);
            FOR_E if (ON(e)) {
                const V di = diag(e);
                FOR_J {
                    const V s = r[e][j];
                    V upd = vadd(res_scale(pv[M == RES_BICG ? e : 0][j], al[j]), res_scale(s, om[j]));
                    if (idiag) upd = vmul(di, upd);
                    const V rn = vsub(s, res_scale(tv[M == RES_BICG ? e : 0][j], om[j]));
                    if (act[j]) {
                        x[e][j] = vadd(x[e][j], upd);
                        r[e][j] = rn;
                    }
                    d[0][j] += dotR(rn, rn);
                    d[1][j] += dotR(shadow(e, j), rn);
                }
            }
            if (!team_sum<2, CL>(tm, d)) return;
            res_fin(FIN_BICG_RHO, tm, tm.S, tm.I, 0, 1, -1, a.maxit, 0.0);
        } else {
            if (!team_sum<M == RES_COCG ? 2 : 1, CL>(tm, d)) return;
            res_fin(M == RES_COCG ? FIN_COCG_ALPHA : FIN_CG_ALPHA, tm, tm.S, tm.I, 0, M == RES_COCG ? 1 : -1, -1, 0,
                    0.0);
            __syncthreads();
            FRESH;
            CLEAR_D;
            bool act[CL];
            S ar[CL], ai[CL];
            FOR_J {
                act[j] = IN(I_ACTIVE, j) != 0;
                ar[j] = (S)SC(S_ALPHA, j);
                ai[j] = M == RES_COCG ? (S)SC(S_ALPHA_I, j) : (S)0;
            }
            FOR_E if (ON(e)) {
                const V di = diag(e);
                const V *sp = stage + AT(e);
                FOR_J {
                    V xn, rn;
                    if constexpr (M == RES_COCG) {
                        xn = vadd(x[e][j], res_scale(sp[j], ar[j], ai[j]));
                        rn = vsub(r[e][j], res_scale(y[e][j], ar[j], ai[j]));
                        bil_add(rn, prec(di, rn, j), d[0][j], d[1][j]);
                        d[2][j] += dotR(rn, rn);
                    } else {
                        xn = vadd(x[e][j], res_scale(sp[j], ar[j]));
                        rn = vsub(r[e][j], res_scale(y[e][j], ar[j]));
                        d[0][j] += dotR(rn, prec(di, rn, j));
                        d[1][j] += dotR(rn, rn);
                    }
                    if (act[j]) {
                        x[e][j] = xn;
                        r[e][j] = rn;
                    }
                }
            }
            if (!team_sum<M == RES_COCG ? 3 : 2, CL>(tm, d)) return;
            res_fin(M == RES_COCG ? FIN_COCG_BETA : FIN_CG_BETA, tm, tm.S, tm.I, 0, 1, M == RES_COCG ? 2 : -1, a.maxit,
                    0.0);
        }
        if (due && a.mixed) {
            todo = T_REPLACE;
            __syncthreads();
        }
    }
    __syncthreads();
    FRESH;
    FOR_E if (ON(e)) {
        const size_t node = (size_t)a.node[r0 + ROW(e)] * a.ld + a.q0 + c0 + c;
        FOR_J if (c + j < ncol)((V64 *)a.x)[node + j] = ld_pub((const V64 *)X + AT(e) + j);
    }
    if (rank == 0 && tid < ncol) {
        ResColOut &o = a.out[c0 + tid];
        o.res2 = tm.O[tid * S_NSLOT + S_RES2];
        o.bnorm2 = tm.O[tid * S_NSLOT + S_BNORM2];
        o.iters = tm.I[tid * (I_NSLOT + 1) + I_ITERS];
        o.sweeps = nupd;
    }
#undef FOR_E
#undef FOR_J
#undef ROW
#undef ON
#undef AT
#undef CLEAR_D
#undef IN
#undef OUT
#undef SC
#undef OSC
#undef FRESH
}

// launch (krylov_resident_*.hip) with lds bytes of dynamic LDS: false when no
// instantiation covers (cl, E) or the device cannot hold one workgroup per CU
bool launch_resident_cg(VKind vk, int cl, int E, bool cocg, bool mf, const ResArgs &a, size_t lds, hipStream_t st);
bool launch_resident_bicg(VKind vk, int cl, int E, const ResArgs &a, size_t lds, hipStream_t st);

}  // namespace tmi
