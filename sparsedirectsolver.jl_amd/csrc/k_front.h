// Device helpers shared by the front kernels: the assembly of a dense front held in
// LDS (A through the owner-grouped assembly runs, then the children's contribution
// blocks in child_list order), in the order the CPU reference uses
// (src/reference/cholesky.jl:73-92, src/reference/ldlt.jl:176-190): every front entry
// receives its A entries first, summed in nzval order, then each child's value in turn.
#pragma once
#include "sds_common.h"

namespace sds {

__device__ inline int64_t lane_int64(int64_t v, int lane) {
    const int lo = __builtin_amdgcn_readlane((int)v, lane), hi = __builtin_amdgcn_readlane((int)(v >> 32), lane);
    return ((int64_t)hi << 32) | (uint32_t)lo;
}

// Descriptors of up to 64 children of a front from child_list[kb] on, a lane each: read at once,
// before A is added, so that their loads overlap A's instead of following one another per child.
struct Children {
    int64_t cb, rel;  // the contribution block (-1: none) and the row positions in the parent
    int m;            // order of the block
    __device__ void load(const DevSym& S, int kb, int k1, int lane) {
        if (kb >= k1) return;
        const int c = S.child_list[min(kb + lane, k1 - 1)];
        cb = S.cb_off[c];
        rel = S.relind_ptr[c];
        m = S.fnrows[c] - S.fncols[c];
    }
};

// Entry k of a front's assembly list: false unless it is the first of a run of entries with one
// destination; the destination and the run's sum in nzval order. A run is nearly always a single
// entry: its neighbours and its value are read together.
__device__ inline bool asm_run(const DevSym& S, const double* __restrict__ nz, int64_t a0, int64_t a1, int64_t k,
                               int64_t& d, double& v) {
    d = S.asm_dst[k];
    const int64_t before = S.asm_dst[max(k - 1, a0)], after = S.asm_dst[min(k + 1, a1 - 1)];
    const double x = nz[S.asm_src[k]];
    if (k > a0 && before == d) return false;
    v = 0.0;
    v += x;
    if (k + 1 < a1 && after == d)
        for (int64_t q = k + 1; q < a1 && S.asm_dst[q] == d; ++q) v += nz[S.asm_src[q]];
    return true;
}

// F (f x f, column-major, any address space) <- 0 + A + children; `full`: the children's
// whole m x m blocks (LU), else their lower triangles. Every thread of the block calls it;
// it ends with a barrier.
template <typename T>
__device__ __forceinline__ void assemble_dense(const DevSym& S, int s, const double* __restrict__ nz, const T* __restrict__ cbpool,
                               T* F, int f, int full) {
    const int tid = threadIdx.x, nt = blockDim.x;
    const int lane = tid & 63, wv = tid >> 6, nw = nt >> 6;
    const int k0 = S.child_ptr[s], k1 = S.child_ptr[s + 1];
    const int64_t a0 = S.asm_ptr[s], a1 = S.asm_ptr[s + 1];
    Children ch;
    ch.load(S, k0, k1, lane);
    for (int q = tid; q < f * f; q += nt) F[q] = T(0);
    __syncthreads();
    // one thread sums each run of entries with the same destination, in nzval order
    for (int64_t k = a0 + tid; k < a1; k += nt) {
        int64_t d;
        double v;
        if (!asm_run(S, nz, a0, a1, k, d, v)) continue;
        if (d >= 0) {
            F[d] += T(v);
        } else {
            // a mirrored entry: the U^T structure of an unsymmetric front is stored transposed
            const int64_t loc = -(d + 1);
            if (S.unsym) {
                const int64_t j = loc / f, i = loc - j * f;
                F[i * f + j] += T(v);
            } else {
                F[loc] += T(v);
            }
        }
    }
    __syncthreads();
    // each child is added by a wave per four of its columns, lanes along the rows, eight loads a lane
    // in flight (m_c <= f <= 128)
    for (int kb = k0; kb < k1; kb += 64) {
        if (kb > k0) ch.load(S, kb, k1, lane);
        for (int kc = 0; kc < min(64, k1 - kb); ++kc) {
            const int64_t co = lane_int64(ch.cb, kc), rp = lane_int64(ch.rel, kc);
            const int mc = __builtin_amdgcn_readlane(ch.m, kc);
            if (co < 0 || mc == 0) continue;
            const T* C = cbpool + co;
            const int32_t* ri = S.relind + rp;
            const int r0 = ri[min(lane, mc - 1)], r1 = ri[min(lane + 64, mc - 1)];
            for (int j0 = wv; j0 < mc; j0 += 4 * nw) {
                T v[4][2];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const T* col = C + (int64_t)min(j0 + u * nw, mc - 1) * mc;
                    v[u][0] = col[min(lane, mc - 1)];
                    if (mc > 64) v[u][1] = col[min(lane + 64, mc - 1)];
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int jj = j0 + u * nw;
                    if (jj >= mc) break;
                    T* col = F + (jj < 64 ? __builtin_amdgcn_readlane(r0, jj) : __builtin_amdgcn_readlane(r1, jj - 64)) * f;
                    if (lane < mc && (full || lane >= jj)) col[r0] += v[u][0];
                    if (mc > 64 && lane + 64 < mc && (full || lane + 64 >= jj)) col[r1] += v[u][1];
                }
            }
            __syncthreads();
        }
    }
}

}  // namespace sds
