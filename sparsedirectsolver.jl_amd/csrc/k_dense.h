// Dense front kernels' device helpers: the Cholesky of a front held in LDS and the inverse of
// its diagonal block, shared by the per-level small-front kernel and the subtree kernel.
#pragma once
#include "sds_common.h"

namespace sds {

// Cholesky pivot acceptance on the FP64 value of the pivot (src/numeric/front.jl:46-50):
// a pivot in [0, eps] is raised to eps (cuDSS pivot_epsilon), negative or NaN fails.
__device__ inline bool chol_accept(double a, double eps) { return a > eps || (eps > 0.0 && a >= 0.0); }

// panel width of the blocked dense Cholesky
constexpr int DPB = 16;

// LDS written by some lanes of a wave is read by others after this (in-order LDS per wave; the
// fence keeps the compiler from moving accesses across it and waits for the outstanding ones)
__device__ inline void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// value of v in lane `lane` (wave-uniform) with v_readlane (no LDS round trip)
__device__ inline double lane_value(double v, int lane) {
    const int lo = __builtin_amdgcn_readlane(__double2loint(v), lane);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(v), lane);
    return __hiloint2double(hi, lo);
}
__device__ inline float lane_value(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// Right-looking Cholesky of the first w columns of the dense f x f front F (LDS, column-major,
// ld f; f <= 64 RPL) by a workgroup of 256 threads, in panels of DPB columns:
//  - wave 0 factors the panel in registers (rows over the lanes, RPL rows per lane; pivots and
//    the panel's rows broadcast with lane reads): column j gets d = sqrt(max(a_jj, eps)) and the
//    rows below are multiplied by 1/d (as the CPU reference's potf2 scaling), then each later
//    panel column c gets -= L(i, j) L(c, j);
//  - all four waves give the columns right of the panel (the rest of the fully summed columns and
//    the contribution block, lower triangle) the panel's update, a wave per two columns, rows over
//    the lanes, the panel's row of the lane held in registers.
// What bounds it: in a level of few fronts the first fetch of its code and the pivots' serial chain,
// in one of thousands the workgroups a CU holds. So the panel is a rolled loop over the pivots, the
// wave index is made uniform (addresses and conditions in scalar registers), and it is always
// inlined: as a function of its own it cost its callers 268 registers and three of four workgroups.
// Two barriers per panel. Every entry receives its column updates one by one in column order, as
// a separate product and difference, exactly as in the column-by-column form. Returns 0, or the
// local column (1-based) of the first failed pivot (the columns from it on are left unfactored).
// `sh` is one int of LDS. Every thread of the block calls it; it ends with a barrier.
template <typename T, int RPL>
__device__ __forceinline__ int front_chol_lds(T* F, int f, int w, double eps, int* sh) {
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (tid == 0) *sh = 0;
    __syncthreads();
#pragma unroll 1
    for (int k0 = 0; k0 < w; k0 += DPB) {
        const int kb = min(DPB, w - k0), k1 = k0 + kb;
        if (wv == 0) {
            // p[q][c2] = row k0 + lane + 64 q of column j + c2: the columns move one register left per
            // pivot, so that one rolled loop body serves the panel (unrolled over the pivots the code,
            // fetched once per launch, cost more than the arithmetic)
            T p[RPL][DPB];
#pragma unroll
            for (int q = 0; q < RPL; ++q) {
                const int i = k0 + lane + 64 * q;
#pragma unroll
                for (int c = 0; c < DPB; ++c) p[q][c] = F[(k0 + min(c, kb - 1)) * f + min(i, f - 1)];
            }
            int st = 0;
#pragma unroll 1
            for (int c = 0; c < kb; ++c) {
                const int j = k0 + c;
                const double a = (double)lane_value(p[0][0], c);
                if (!st && !chol_accept(a, eps)) st = j + 1;
                if (st) {  // left as it stands
#pragma unroll
                    for (int q = 0; q < RPL; ++q) {
                        const int i = k0 + lane + 64 * q;
                        if (i >= j && i < f) F[j * f + i] = p[q][0];
#pragma unroll
                        for (int c2 = 1; c2 < DPB; ++c2) p[q][c2 - 1] = p[q][c2];
                    }
                    continue;
                }
                const T d = T(sqrt(fmax(a, eps)));
                const T rd = T(1) / d;
                T x[RPL];
#pragma unroll
                for (int q = 0; q < RPL; ++q) {
                    const int i = k0 + lane + 64 * q;
                    x[q] = i == j ? d : p[q][0] * rd;
                    if (i >= j && i < f) F[j * f + i] = x[q];
                }
                // (columns past the panel and entries above the diagonal: never stored)
#pragma unroll
                for (int cb = 0; cb < DPB; cb += 4) {
                    if (c + cb < kb) {
#pragma unroll
                        for (int c2 = cb == 0 ? 1 : cb; c2 < cb + 4; ++c2) {
                            const T l = lane_value(x[0], c + c2);
#pragma unroll
                            for (int q = 0; q < RPL; ++q) {
                                const T prod = x[q] * l;
                                p[q][c2 - 1] = p[q][c2] - prod;
                            }
                        }
                    }
                }
            }
            if (lane == 0 && st) *sh = st;
        }
        __syncthreads();
        const int st = __builtin_amdgcn_readfirstlane(*sh);
        if (st) return st;
        // the panel's update of the columns right of it, lower triangle: 64 rows at a time (a row a
        // lane), a wave per two columns
#pragma unroll 1
        for (int i0 = k1; i0 < f; i0 += 64) {
            const int i = i0 + lane, jend = min(f, i0 + 64);
            T pr[DPB];
#pragma unroll
            for (int c = 0; c < DPB; ++c) pr[c] = F[(k0 + min(c, kb - 1)) * f + min(i, f - 1)];
#pragma unroll 1
            for (int j = k1 + wv; j < jend; j += 8) {
                // (f hidden from the optimizer: the sixteen columns' addresses, moved out of the loop,
                // would take a register each)
                int fj = __builtin_amdgcn_readfirstlane(f);
                asm volatile("" : "+s"(fj));
                const int j2 = min(j + 4, f - 1);
                const bool u1 = i >= j && i < f, u2 = i >= j2 && i < f && j + 4 < jend;
                T v1 = F[j * f + min(i, f - 1)], v2 = F[j2 * f + min(i, f - 1)];
#pragma unroll
                for (int cb = 0; cb < DPB; cb += 4) {
                    if (cb < kb) {
                        T l1[4], l2[4];
#pragma unroll
                        for (int c = 0; c < 4; ++c) {
                            const T* Lc = F + (k0 + min(cb + c, kb - 1)) * fj;
                            l1[c] = Lc[j];
                            l2[c] = Lc[j2];
                        }
#pragma unroll
                        for (int c = 0; c < 4; ++c) {
                            const T p1 = pr[cb + c] * l1[c], p2 = pr[cb + c] * l2[c];
                            if (cb + c < kb) {
                                v1 = v1 - p1;
                                v2 = v2 - p2;
                            }
                        }
                    }
                }
                if (u1) F[j * f + i] = v1;
                if (u2) F[j2 * f + i] = v2;
            }
        }
        __syncthreads();
    }
    return 0;
}

// Inverse of the lower-triangular w x w diagonal block L11 of the factored front F (LDS, ld f),
// w <= FUSED_INV_MAX <= NB, into `out` (column-major, ld NB: column c at out + c NB, rows past w
// zero): thread c < w computes column c by forward substitution, x = L11^-1 e_c (x_m *= 1 / L_mm,
// then x_r -= L_rm x_m), the arithmetic of the per-block inverse kernel. x[r] is row m + r at step
// m: the rows move one register down per step, one rolled loop body serves them all.
template <typename T>
__device__ void diag_inverse_lds(const T* F, int f, int w, T* __restrict__ out) {
    // column c of the block is factor column super_ptr[s] + c: only the front's own w columns
    const int c = threadIdx.x;
    if (c >= w) return;
    T x[FUSED_INV_MAX];
#pragma unroll
    for (int r = 0; r < FUSED_INV_MAX; ++r) x[r] = r == c ? T(1) : T(0);
    T* o = out + (int64_t)c * NB;
#pragma unroll 1
    for (int m = 0; m < w; ++m) {
        const T* Lm = F + m * f;
        const T rinv = T(1) / Lm[m];
        const T xm = x[0] * rinv;
        o[m] = xm;
#pragma unroll
        for (int r = 1; r < FUSED_INV_MAX; ++r) x[r - 1] = fma(-Lm[min(m + r, w - 1)], xm, x[r]);
    }
    for (int r = w; r < NB; ++r) o[r] = T(0);
}

}  // namespace sds
