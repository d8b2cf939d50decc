// Layout of a relabelled system for the resident solve (ResLayout, mesh.hpp),
// built on the GPU: the first solve of a mesh builds the one it uses, and
// building it on the host took as long as the solve it serves (4-7 ms at
// 31,525 nodes; here 0.1 ms for 64 ranks, 0.9 ms for 16: a rank's rows are
// sorted by counting, which grows with their square).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>

#include "mesh.hpp"

namespace tmi {

constexpr int RL_NT = 512;

__device__ inline int rank_begin(int n, int r, int nr) { return (int)((long)n * r / nr); }

// One workgroup per rank: its rows (part[r0 .. r1), any order) by falling
// length, equal ones ascending; the length of each slice of 8, a multiple of 4.
__global__ void __launch_bounds__(RL_NT) k_res_rows(int n, int nr, const int *__restrict__ part,
                                                    const int *__restrict__ rowptr, const int *__restrict__ perm,
                                                    int *__restrict__ srow, int *__restrict__ node,
                                                    int *__restrict__ pos, const int *__restrict__ rslice,
                                                    int *__restrict__ slen)
{
    extern __shared__ int lds[];
    const int r = blockIdx.x, r0 = rank_begin(n, r, nr), m = rank_begin(n, r + 1, nr) - r0;
    int *row = lds, *len = lds + m, *sorted = len + m;
    for (int i = threadIdx.x; i < m; i += RL_NT) {
        const int v = part[r0 + i];
        row[i] = v;
        len[i] = rowptr[v + 1] - rowptr[v];
    }
    __syncthreads();
    for (int i = threadIdx.x; i < m; i += RL_NT) {
        const int v = row[i], l = len[i];
        int at = 0;
        for (int k = 0; k < m; k++) at += len[k] > l || (len[k] == l && row[k] < v);
        srow[r0 + at] = v;
        node[r0 + at] = perm[v];
        pos[v] = r0 + at;
        sorted[at] = l;
    }
    __syncthreads();
    for (int s = threadIdx.x; s < (m + 7) / 8; s += RL_NT) slen[rslice[r] + s] = (sorted[8 * s] + 3) / 4 * 4 * 8;
}

// The halo of a rank: one bit per position in LDS marks the columns of its
// rows outside it; the bits' running count is a column's place in the halo,
// which is ascending by position.  FILL false: only the halo's size; true:
// the halo and the slice entries.
template <bool FILL>
__global__ void __launch_bounds__(RL_NT) k_res_halo(int n, int nr, const int *__restrict__ rowptr,
                                                    const int *__restrict__ colidx, const int *__restrict__ srow,
                                                    const int *__restrict__ pos, const int *__restrict__ rslice,
                                                    const int *__restrict__ sofs, int *__restrict__ hcnt,
                                                    const int *__restrict__ hofs, int *__restrict__ halo,
                                                    unsigned short *__restrict__ lcol, int *__restrict__ gcol,
                                                    int *__restrict__ slot)
{
    extern __shared__ unsigned bits[];
    const int W = (n + 31) / 32;
    unsigned *pre = bits + W;
    __shared__ unsigned part[RL_NT];
    const int tid = threadIdx.x, r = blockIdx.x, r0 = rank_begin(n, r, nr), r1 = rank_begin(n, r + 1, nr);
    for (int w = tid; w < W; w += RL_NT) bits[w] = 0u;
    __syncthreads();
    for (int i = r0 + tid; i < r1; i += RL_NT) {
        const int v = srow[i];
        for (int k = rowptr[v]; k < rowptr[v + 1]; k++) {
            const int p = pos[colidx[k]];
            if (p < r0 || p >= r1) atomicOr(&bits[p >> 5], 1u << (p & 31));
        }
    }
    __syncthreads();
    // running count: a contiguous chunk of words per thread, then the chunks
    const int chunk = (W + RL_NT - 1) / RL_NT, b = min(W, tid * chunk), e = min(W, b + chunk);
    unsigned sum = 0;
    for (int w = b; w < e; w++) sum += __popc(bits[w]);
    part[tid] = sum;
    __syncthreads();
    for (int off = 1; off < RL_NT; off <<= 1) {
        const unsigned v = tid >= off ? part[tid - off] : 0u;
        __syncthreads();
        part[tid] += v;
        __syncthreads();
    }
    if constexpr (!FILL) {
        if (tid == 0) hcnt[r] = (int)part[RL_NT - 1];
        return;
    } else {
        unsigned run = part[tid] - sum;
        const int h0 = hofs[r];
        for (int w = b; w < e; w++) {
            pre[w] = run;
            for (unsigned m = bits[w]; m; m &= m - 1) halo[h0 + run++] = 32 * w + __ffs((int)m) - 1;
        }
        __syncthreads();
        const int rows8 = (r1 - r0 + 7) / 8 * 8;
        for (int i = tid; i < rows8; i += RL_NT) {
            const int s = rslice[r] + i / 8, len = (sofs[s + 1] - sofs[s]) / 8;
            int at = sofs[s] + i % 8, k0 = 0, kn = 0;
            if (r0 + i < r1) {
                const int v = srow[r0 + i];
                k0 = rowptr[v];
                kn = rowptr[v + 1] - k0;
            }
            for (int k = 0; k < len; k++, at += 8) {
                if (k < kn) {
                    const int p = pos[colidx[k0 + k]];
                    const unsigned h = pre[p >> 5] + __popc(bits[p >> 5] & ((1u << (p & 31)) - 1u));
                    lcol[at] = (unsigned short)(p >= r0 && p < r1 ? p - r0 : r1 - r0 + (int)h);
                    gcol[at] = p;
                    slot[at] = k0 + k;
                } else {   // padding: a zero coefficient on the rank's first row
                    lcol[at] = 0;
                    gcol[at] = r0 < n ? r0 : 0;
                    slot[at] = -1;
                }
            }
        }
    }
}

const ResLayout *Mesh::res_layout(int kind, int nr, hipStream_t st)
{
    int lg = 0;
    while ((1 << lg) < nr) lg++;
    TMI_CHECK(nr >= 1 && (1 << lg) == nr && lg < 9, TMI_ERR_INVALID_ARG, "resident layout for %d ranks", nr);
    std::lock_guard<std::mutex> lk(res_mu);
    NodeOrder &o = order[kind];
    TMI_CHECK(o.valid, TMI_ERR_STATE, "resident layout before the node order");
    if (o.res[lg]) return o.res[lg].get();
    // LDS of the builders: three ints per row of a rank; two words per 32 nodes
    const size_t lds1 = 12 * (size_t)((n + nr - 1) / nr + 1), lds2 = 8 * (size_t)((n + 31) / 32) + 4 * RL_NT;
    if (lds1 > 150 * 1024 || lds2 > 150 * 1024) return nullptr;
    std::unique_ptr<ResLayout> l(new ResLayout);
    std::vector<int> rslice(nr + 1, 0);
    for (int r = 0; r < nr; r++) {
        const int m = (int)((long)n * (r + 1) / nr) - (int)((long)n * r / nr);
        rslice[r + 1] = rslice[r] + (m + 7) / 8;
    }
    const int ns = rslice[nr];
    DBuf<int> pos(n), slen(ns), hcnt(nr);
    l->rslice.upload(rslice.data(), nr + 1, st);
    l->srow.alloc(n);
    l->node.alloc(n);
    l->sofs.alloc(ns + 1);
    l->hofs.alloc(nr + 1);
    hipLaunchKernelGGL(k_res_rows, dim3(nr), dim3(RL_NT), lds1, st, n, nr, o.part.p, o.rowptr.p, o.perm.p, l->srow.p,
                       l->node.p, pos.p, l->rslice.p, slen.p);
    TMI_LAUNCH_CHECK();
    launch_exclusive_scan(slen.p, l->sofs.p, ns, st);
    hipLaunchKernelGGL(k_res_halo<false>, dim3(nr), dim3(RL_NT), lds2, st, n, nr, o.rowptr.p, o.colidx.p, l->srow.p,
                       pos.p, l->rslice.p, l->sofs.p, hcnt.p, (const int *)nullptr, (int *)nullptr,
                       (unsigned short *)nullptr, (int *)nullptr, (int *)nullptr);
    TMI_LAUNCH_CHECK();
    launch_exclusive_scan(hcnt.p, l->hofs.p, nr, st);
    std::vector<int> hofs(nr + 1);
    l->hofs.download(hofs.data(), nr + 1, st);
    TMI_HIP(hipMemcpyAsync(&l->nent, l->sofs.p + ns, sizeof(int), hipMemcpyDeviceToHost, st));
    TMI_HIP(hipStreamSynchronize(st));
    for (int r = 0; r < nr; r++) {
        const int m = (int)((long)n * (r + 1) / nr) - (int)((long)n * r / nr);
        l->nu = std::max(l->nu, m + hofs[r + 1] - hofs[r]);
    }
    if (l->nu > 65535) l->nu = INT_MAX;   // local columns do not fit 16 bits: the layout is not used
    l->halo.alloc(std::max(1, hofs[nr]));
    l->lcol.alloc(l->nent);
    l->gcol.alloc(l->nent);
    l->slot.alloc(l->nent);
    hipLaunchKernelGGL(k_res_halo<true>, dim3(nr), dim3(RL_NT), lds2, st, n, nr, o.rowptr.p, o.colidx.p, l->srow.p,
                       pos.p, l->rslice.p, l->sofs.p, (int *)nullptr, l->hofs.p, l->halo.p, l->lcol.p, l->gcol.p,
                       l->slot.p);
    TMI_LAUNCH_CHECK();
    TMI_HIP(hipStreamSynchronize(st));   // other streams read it next
    o.res[lg] = std::move(l);
    return o.res[lg].get();
}

}  // namespace tmi
