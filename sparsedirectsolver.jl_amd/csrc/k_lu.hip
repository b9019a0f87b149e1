// LU factorization kernels (gfx950) for structure "G": threshold partial pivoting by rows
// inside each front's fully summed block (keep the diagonal when |a_kk| >= u max_i |a_ik|
// over the whole column, else take the largest fully summed row), static perturbation,
// and the Schur update F22 <- F22 - (L21 D) U12.
//
// As the LDL^T kernels, every floating-point operation is the CPU reference's, in the
// same order, with contraction off: in FP64 the row order, D, L, U and the contribution
// blocks are bitwise those of src/reference/lu.jl.
//
// Storage of a front while it is factored: the L panel P (f x w, column-major, ld f,
// the factor buffer) holds the columns < w including the whole fully summed square; the
// rows < w of the columns >= w (U12) are stored transposed in the U panel Q (the ufactor
// buffer, same layout: Q[i * f + j] = F[i, j] for i < w <= j); F22 is the contribution
// block square. At the end P is unit lower (L) and Q holds U^T, unit diagonal.
//
// Reference counterparts: ref_lu! and _lu_front! (src/reference/lu.jl:84-214),
// _lu_choose_row (:216-231), assembly with U^T entries (:114-131), the Schur update
// (:137-145).
#pragma clang fp contract(off)
#include "k_front.h"
#include "k_panel.h"
#include "panel_plan.h"
#include "sds_common.h"
#include "sds_kernels.h"

namespace sds {

enum { LST_NZERO = 2, LST_NPERT = 3, LST_INFO = 5 };

__device__ inline double lu_jmax(double a, double b) {
    if (a != a || b != b) return a + b;
    return a > b ? a : b;
}

// a front as the LU loop sees it
template <typename T>
struct LuFront {
    T* P;      // columns < w (ld f)
    T* Q;      // rows < w of columns >= w, transposed (ld f); == nullptr: F is the dense f x f P
    int f, w;
    __device__ T& l(int i, int j) const { return P[(int64_t)j * f + i]; }  // j < w
    __device__ T& u(int i, int j) const {                                   // i < w <= j
        return Q ? Q[(int64_t)i * f + j] : P[(int64_t)j * f + i];
    }
    __device__ T& at(int i, int j) const { return j < w ? l(i, j) : u(i, j); }
};

template <int NT>
struct LuRed {
    double v[NT / 64];
    int i[NT / 64];
};

// the LU pivot loop of one front (lu.jl:163-214), all NT threads
template <typename T, int NT>
__device__ void lu_front(const LuFront<T>& Fr, int pivoting, double u, double eps, int* lp, int8_t* kind, T* dd,
                         int* st, LuRed<NT>& rb, double* sh) {
    const int f = Fr.f, w = Fr.w, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    for (int k = 0; k < w; ++k) {
        int r = k;
        if (pivoting) {
            // g = max_{i >= k} |F[i, k]| (NaN-propagating)
            double g = 0.0;
            for (int i = k + tid; i < f; i += NT) g = lu_jmax(g, fabs((double)Fr.l(i, k)));
            for (int o = 32; o > 0; o >>= 1) g = lu_jmax(g, __shfl_xor(g, o));
            if (lane == 0) rb.v[wv] = g;
            __syncthreads();
            g = rb.v[0];
            for (int q = 1; q < NT / 64; ++q) g = lu_jmax(g, rb.v[q]);
            __syncthreads();
            const double akk = fabs((double)Fr.l(k, k));
            if (!(akk >= u * g)) {
                // the largest fully summed row, the first on ties, k if none is larger
                double bv = akk;
                int bi = k;
                for (int i = k + 1 + tid; i < w; i += NT) {
                    const double a = fabs((double)Fr.l(i, k));
                    if (a > bv) {
                        bv = a;
                        bi = i;
                    }
                }
                for (int o = 32; o > 0; o >>= 1) {
                    const double ov = __shfl_xor(bv, o);
                    const int oi = __shfl_xor(bi, o);
                    if (ov > bv || (ov == bv && oi < bi)) {
                        bv = ov;
                        bi = oi;
                    }
                }
                if (lane == 0) {
                    rb.v[wv] = bv;
                    rb.i[wv] = bi;
                }
                __syncthreads();
                bv = rb.v[0];
                bi = rb.i[0];
                for (int q = 1; q < NT / 64; ++q)
                    if (rb.v[q] > bv || (rb.v[q] == bv && rb.i[q] < bi)) {
                        bv = rb.v[q];
                        bi = rb.i[q];
                    }
                r = bi;
            }
            __syncthreads();  // every read of the pivot column is done before the swap
        }
        if (r != k) {
            for (int j = tid; j < f; j += NT) {
                T& a = Fr.at(k, j);
                T& b = Fr.at(r, j);
                const T t = a;
                a = b;
                b = t;
            }
            if (tid == 0) {
                const int t = lp[k];
                lp[k] = lp[r];
                lp[r] = t;
            }
            __syncthreads();
        }
        if (tid == 0) {
            double dk = (double)Fr.l(k, k);
            int8_t kd = KIND_1X1;
            if (!(fabs(dk) >= eps) || dk == 0.0) {
                if (dk == 0.0) st[LST_NZERO]++;
                dk = (dk < 0.0 ? -1.0 : 1.0) * eps;
                kd = KIND_PERTURBED;
                st[LST_NPERT]++;
                if (dk == 0.0 && st[LST_INFO] == 0) st[LST_INFO] = k + 1;
            }
            Fr.l(k, k) = T(dk);
            dd[k] = T(dk);
            kind[k] = kd;
            sh[0] = dk;
        }
        __syncthreads();
        const T dk = T(sh[0]);
        // trailing fully summed columns (all rows below k), then U12 (the fully summed rows)
        const int R = f - k - 1, C = w - k - 1;
        for (int q = tid; q < R * C; q += NT) {
            const int j = k + 1 + q / R, i = k + 1 + q % R;
            Fr.l(i, j) = Fr.l(i, j) - Fr.l(i, k) / dk * Fr.l(k, j);
        }
        const int m = f - w;
        for (int q = tid; q < C * m; q += NT) {
            const int j = w + q / C, i = k + 1 + q % C;
            Fr.u(i, j) = Fr.u(i, j) - Fr.l(i, k) / dk * Fr.u(k, j);
        }
        __syncthreads();
        for (int i = k + 1 + tid; i < f; i += NT) Fr.l(i, k) = Fr.l(i, k) / dk;
        for (int j = k + 1 + tid; j < f; j += NT) {
            T& x = Fr.at(k, j);
            x = x / dk;
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// small fronts: the dense front in LDS

constexpr int LU_SMALL_W = 128;

template <typename T>
__global__ void __launch_bounds__(256) k_front_small_lu(DevSym S, const int32_t* __restrict__ fronts,
                                                       const double* __restrict__ nz, T* __restrict__ factor,
                                                       T* __restrict__ ufactor, T* __restrict__ cbpool,
                                                       T* __restrict__ dvec, int32_t* __restrict__ piv,
                                                       int8_t* __restrict__ pkind, int64_t* __restrict__ stats,
                                                       int pivoting, double u, double eps, int scaled,
                                                       const double* __restrict__ aux) {
    constexpr int NT = 256;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    T* F = reinterpret_cast<T*>(smem_raw);
    __shared__ LuRed<NT> rb;
    __shared__ int lp[LU_SMALL_W];
    __shared__ int8_t kind[LU_SMALL_W];
    __shared__ T dd[LU_SMALL_W];
    __shared__ int st[NF];
    __shared__ double sh[2];
    const int s = fronts[blockIdx.x];
    const int f = S.fnrows[s], w = S.fncols[s], m = f - w;
    const int c0 = S.super_ptr[s];
    const int tid = threadIdx.x;
    if (scaled && aux[0] > 0) eps = eps * aux[0];
    for (int k = tid; k < w; k += NT) {
        lp[k] = k;
        kind[k] = KIND_1X1;
        dd[k] = T(0);
    }
    if (tid < NF) st[tid] = 0;
    assemble_dense<T>(S, s, nz, cbpool, F, f, 1);
    LuFront<T> Fr{F, nullptr, f, w};
    lu_front<T, NT>(Fr, pivoting, u, eps, lp, kind, dd, st, rb, sh);
    // F22 <- F22 - (L21 D) U12, the whole block, each entry's sum in k order
    const int64_t co = S.cb_off[s];
    if (co >= 0) {
        T* C = cbpool + co;
        for (int q = tid; q < m * m; q += NT) {
            const int jj = q / m, ii = q - jj * m;
            T acc = T(0);
            for (int k = 0; k < w; ++k) acc = acc + F[k * f + w + ii] * dd[k] * F[(w + jj) * f + k];
            C[q] = F[(w + jj) * f + w + ii] - acc;
        }
    }
    T* P = factor + S.panel_off[s];
    T* Q = ufactor + S.panel_off[s];
    for (int q = tid; q < f * w; q += NT) {
        const int j = q / f, i = q - j * f;
        P[q] = i > j ? F[q] : (i == j ? T(1) : T(0));
        Q[q] = i > j ? F[i * f + j] : (i == j ? T(1) : T(0));
    }
    for (int k = tid; k < w; k += NT) {
        const int g = c0 + k;
        piv[g] = c0 + lp[k];
        pkind[g] = kind[k];
        dvec[g] = dd[k];
        dvec[S.n + g] = T(0);
    }
    if (tid < NF) stats[(int64_t)s * NF + tid] = st[tid];
}

// ---------------------------------------------------------------------------
// large fronts

// zero a chunk of columns [col0, col0 + ncols) of the front: panel columns of P and Q, or
// contribution-block columns. task: (s, col0, ncols)
template <typename T>
__global__ void __launch_bounds__(256) k_big_lu_zero(DevSym S, const Task* __restrict__ tasks, T* __restrict__ factor,
                                                    T* __restrict__ ufactor, T* __restrict__ cbpool) {
    const Task t = tasks[blockIdx.x];
    const int s = t.s, f = S.fnrows[s], w = S.fncols[s], m = f - w;
    T* P = factor + S.panel_off[s];
    T* Q = ufactor + S.panel_off[s];
    T* C = cbpool + (S.cb_off[s] >= 0 ? S.cb_off[s] : 0);
    const int j1 = min(t.a + t.b, f);
    for (int j = t.a; j < j1; ++j) {
        if (j < w) {
            for (int i = threadIdx.x; i < f; i += 256) {
                P[(int64_t)j * f + i] = T(0);
                Q[(int64_t)j * f + i] = T(0);
            }
        } else if (S.cb_off[s] >= 0) {
            for (int i = threadIdx.x; i < m; i += 256) C[(int64_t)(j - w) * m + i] = T(0);
        }
    }
}

// A into a zeroed front, the runs of the assembly entries of panel columns [col0, col0 +
// ncols) (a U^T entry at panel position (i, j) is F[j, i]). task: (s, col0, ncols)
template <typename T>
__global__ void __launch_bounds__(256) k_big_lu_scatter(DevSym S, const Task* __restrict__ tasks,
                                                       const double* __restrict__ nz, T* __restrict__ factor,
                                                       T* __restrict__ ufactor) {
    const Task t = tasks[blockIdx.x];
    const int s = t.s, f = S.fnrows[s], w = S.fncols[s];
    T* P = factor + S.panel_off[s];
    T* Q = ufactor + S.panel_off[s];
    const int c0 = S.super_ptr[s];
    const int j1 = min(t.a + t.b, w);
    for (int j = t.a; j < j1; ++j) {
        const int64_t a0 = S.acol_ptr[c0 + j], a1 = S.acol_ptr[c0 + j + 1];
        for (int64_t k = a0 + threadIdx.x; k < a1; k += 256) {
            const int64_t d = S.asm_dst[k];
            if (k > a0 && S.asm_dst[k - 1] == d) continue;
            double v = 0.0;
            for (int64_t q = k; q < a1 && S.asm_dst[q] == d; ++q) v += nz[S.asm_src[q]];
            if (d >= 0) {
                P[d] += T(v);
            } else {
                const int64_t loc = -(d + 1);
                const int pc = (int)(loc / f), pr = (int)(loc - (int64_t)pc * f);  // F[pc, pr]
                if (pr < w)
                    P[(int64_t)pr * f + pc] += T(v);
                else
                    Q[loc] += T(v);
            }
        }
    }
}

// extend-add of one child per front, the child's whole m x m block. task: (s, child, jj0, njj)
template <typename T>
__global__ void __launch_bounds__(256) k_big_lu_extend_add(DevSym S, const Task* __restrict__ tasks,
                                                          T* __restrict__ factor, T* __restrict__ ufactor,
                                                          T* __restrict__ cbpool) {
    const Task t = tasks[blockIdx.x];
    const int s = t.s, f = S.fnrows[s], w = S.fncols[s], m = f - w;
    const int c = t.a, mc = S.fnrows[c] - S.fncols[c];
    T* P = factor + S.panel_off[s];
    T* Q = ufactor + S.panel_off[s];
    T* Cs = cbpool + (S.cb_off[s] >= 0 ? S.cb_off[s] : 0);
    const T* Cc = cbpool + S.cb_off[c];
    const int32_t* ri = S.relind + S.relind_ptr[c];
    const int jend = min(t.b + t.c, mc);
    for (int jj = t.b; jj < jend; ++jj) {
        const int pc = ri[jj];
        for (int ii = threadIdx.x; ii < mc; ii += 256) {
            const int pr = ri[ii];
            T* dst = pc < w ? P + (int64_t)pc * f + pr : pr < w ? Q + (int64_t)pr * f + pc
                                                               : Cs + (int64_t)(pc - w) * m + (pr - w);
            *dst = *dst + Cc[(int64_t)jj * mc + ii];
        }
    }
}

// ---------------------------------------------------------------------------
// large fronts too tall for the panels below, one pivot per pair of launches: k_lu_pivot (one workgroup per front) takes
// the previous pivot's deferred scaling, searches column k, swaps the rows and sets d_k;
// k_lu_update (64 x 64 tiles over every front of the level) applies the rank-1 update of
// step k to the fully summed columns (all rows) and to U12 (the fully summed rows). Each
// entry goes through the same operations, in the same order, as in lu_front above; the
// scaling of column k and row k by d_k moves to the next pivot launch because the update
// tiles read them unscaled.

// the pivot of step k of every front with more than k columns. task: (s)
template <typename T>
__global__ void __launch_bounds__(1024) k_lu_pivot(DevSym S, const Task* __restrict__ tasks, int k,
                                                  T* __restrict__ factor, T* __restrict__ ufactor,
                                                  T* __restrict__ dvec, int32_t* __restrict__ piv,
                                                  int8_t* __restrict__ pkind, int64_t* __restrict__ stats,
                                                  int pivoting, double u, double eps, int scaled,
                                                  const double* __restrict__ aux) {
    constexpr int NT = 1024;
    __shared__ LuRed<NT> rb;
    const int s = tasks[blockIdx.x].s;
    const int f = S.fnrows[s], w = S.fncols[s];
    if (k >= w) return;
    const int c0 = S.super_ptr[s];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    if (scaled && aux[0] > 0) eps = eps * aux[0];
    LuFront<T> Fr{factor + S.panel_off[s], ufactor + S.panel_off[s], f, w};
    int* lp = piv + c0;
    int8_t* kind = pkind + c0;
    T* dd = dvec + c0;
    int64_t* st = stats + (int64_t)s * NF;
    if (k == 0) {
        for (int q = tid; q < w; q += NT) {
            lp[q] = q;
            kind[q] = KIND_1X1;
            dd[q] = T(0);
            dvec[S.n + c0 + q] = T(0);
        }
        if (tid < NF) st[tid] = 0;
    }
    // The usual step in one pass: column k's entries k..f-1 in registers, loaded together with
    // step k - 1's column and row (which are divided by its pivot here) and reduced once for the
    // threshold test's column maximum and the row search; the general loops below serve fronts
    // with more than CR x NT rows.
    constexpr int CR = 8;
    __shared__ double sg[NT / 64];
    int r = k;
    if (f - k <= CR * NT) {
        T x[CR], cv[CR], rv[CR];
        const T* colk = &Fr.l(0, k);
#pragma unroll
        for (int q = 0; q < CR; ++q) x[q] = colk[min(k + tid + NT * q, f - 1)];
        const double akk = fabs((double)colk[k]);
        if (k > 0) {
            const T dp = dd[k - 1];
#pragma unroll
            for (int q = 0; q < CR; ++q) {
                const int i = min(k + tid + NT * q, f - 1);
                cv[q] = Fr.l(i, k - 1);
                rv[q] = Fr.at(k - 1, i);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int q = 0; q < CR; ++q) {
                const int i = k + tid + NT * q;
                if (i < f) {
                    Fr.l(i, k - 1) = cv[q] / dp;
                    Fr.at(k - 1, i) = rv[q] / dp;
                }
            }
        }
        if (pivoting) {
            double g = 0.0, bv = akk;
            int bi = k;
#pragma unroll
            for (int q = 0; q < CR; ++q) {
                const int i = k + tid + NT * q;
                if (i < f) {
                    const double a = fabs((double)x[q]);
                    g = lu_jmax(g, a);
                    if (i > k && i < w && a > bv) {
                        bv = a;
                        bi = i;
                    }
                }
            }
            for (int o = 32; o > 0; o >>= 1) {
                g = lu_jmax(g, __shfl_xor(g, o));
                const double ov = __shfl_xor(bv, o);
                const int oi = __shfl_xor(bi, o);
                if (ov > bv || (ov == bv && oi < bi)) {
                    bv = ov;
                    bi = oi;
                }
            }
            if (lane == 0) {
                sg[wv] = g;
                rb.v[wv] = bv;
                rb.i[wv] = bi;
            }
            __syncthreads();
            g = sg[0];
            bv = rb.v[0];
            bi = rb.i[0];
            for (int q = 1; q < NT / 64; ++q) {
                g = lu_jmax(g, sg[q]);
                if (rb.v[q] > bv || (rb.v[q] == bv && rb.i[q] < bi)) {
                    bv = rb.v[q];
                    bi = rb.i[q];
                }
            }
            if (!(akk >= u * g)) r = bi;
        }
        __syncthreads();
    } else {
        if (k > 0) {
            // step k - 1's column and row, divided by its pivot
            const T dp = dd[k - 1];
            for (int i = k + tid; i < f; i += NT) Fr.l(i, k - 1) = Fr.l(i, k - 1) / dp;
            for (int j = k + tid; j < f; j += NT) {
                T& x = Fr.at(k - 1, j);
                x = x / dp;
            }
        }
        __syncthreads();
        if (pivoting) {
            double g = 0.0;
            for (int i = k + tid; i < f; i += NT) g = lu_jmax(g, fabs((double)Fr.l(i, k)));
            for (int o = 32; o > 0; o >>= 1) g = lu_jmax(g, __shfl_xor(g, o));
            if (lane == 0) rb.v[wv] = g;
            __syncthreads();
            g = rb.v[0];
            for (int q = 1; q < NT / 64; ++q) g = lu_jmax(g, rb.v[q]);
            __syncthreads();
            const double akk = fabs((double)Fr.l(k, k));
            if (!(akk >= u * g)) {
                double bv = akk;
                int bi = k;
                for (int i = k + 1 + tid; i < w; i += NT) {
                    const double a = fabs((double)Fr.l(i, k));
                    if (a > bv) {
                        bv = a;
                        bi = i;
                    }
                }
                for (int o = 32; o > 0; o >>= 1) {
                    const double ov = __shfl_xor(bv, o);
                    const int oi = __shfl_xor(bi, o);
                    if (ov > bv || (ov == bv && oi < bi)) {
                        bv = ov;
                        bi = oi;
                    }
                }
                if (lane == 0) {
                    rb.v[wv] = bv;
                    rb.i[wv] = bi;
                }
                __syncthreads();
                bv = rb.v[0];
                bi = rb.i[0];
                for (int q = 1; q < NT / 64; ++q)
                    if (rb.v[q] > bv || (rb.v[q] == bv && rb.i[q] < bi)) {
                        bv = rb.v[q];
                        bi = rb.i[q];
                    }
                r = bi;
            }
            __syncthreads();
        }
    }
    if (r != k) {
        for (int j = tid; j < f; j += NT) {
            T& a = Fr.at(k, j);
            T& b = Fr.at(r, j);
            const T t = a;
            a = b;
            b = t;
        }
        if (tid == 0) {
            const int t = lp[k];
            lp[k] = lp[r];
            lp[r] = t;
        }
        __syncthreads();
    }
    if (tid == 0) {
        double dk = (double)Fr.l(k, k);
        int8_t kd = KIND_1X1;
        if (!(fabs(dk) >= eps) || dk == 0.0) {
            if (dk == 0.0) st[LST_NZERO]++;
            dk = (dk < 0.0 ? -1.0 : 1.0) * eps;
            kd = KIND_PERTURBED;
            st[LST_NPERT]++;
            if (dk == 0.0 && st[LST_INFO] == 0) st[LST_INFO] = k + 1;
        }
        Fr.l(k, k) = T(dk);
        dd[k] = T(dk);
        kind[k] = kd;
    }
}

// the rank-1 update of step k: tile (s, I0, J0) of 64 x 64 entries, J0 < w: fully summed
// columns (rows I0.. of every row > k), J0 >= w: U12 (rows I0.. < w, stored transposed)
template <typename T>
__global__ void __launch_bounds__(256) k_lu_update(DevSym S, const Task* __restrict__ tasks, int k,
                                                   T* __restrict__ factor, T* __restrict__ ufactor,
                                                   const T* __restrict__ dvec) {
    const Task t = tasks[blockIdx.x];
    const int s = t.s, f = S.fnrows[s], w = S.fncols[s];
    if (k >= w) return;
    const int I0 = t.a, J0 = t.b;
    LuFront<T> Fr{factor + S.panel_off[s], ufactor + S.panel_off[s], f, w};
    const T dk = dvec[S.super_ptr[s] + k];
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    if (J0 < w) {
        // lanes along the rows: column-major panel
        const int i = I0 + tx;
        if (i <= k || i >= f) return;
        // the thread's sixteen columns: loads in flight together (clamped), then the stores;
        // row k is not written here
        const int jb = max(J0, k + 1) + ty, j1 = min(J0 + 64, w);
        if (jb >= j1) return;
        const T lk = Fr.l(i, k) / dk;
        T a[16], b[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const int j = min(jb + 4 * q, j1 - 1);
            a[q] = Fr.l(i, j);
            b[q] = Fr.l(k, j);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < 16; ++q)
            if (jb + 4 * q < j1) Fr.l(i, jb + 4 * q) = a[q] - lk * b[q];
    } else {
        // lanes along the columns: U12 is stored transposed; the thread's sixteen rows as above
        const int j = J0 + tx;
        if (j >= f) return;
        const int ib = max(I0, k + 1) + ty, i1 = min(I0 + 64, w);
        if (ib >= i1) return;
        const T rk = Fr.u(k, j);
        T a[16], l[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const int i = min(ib + 4 * q, i1 - 1);
            l[q] = Fr.l(i, k);
            a[q] = Fr.u(i, j);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < 16; ++q)
            if (ib + 4 * q < i1) Fr.u(ib + 4 * q, j) = a[q] - (l[q] / dk) * rk;
    }
}

// after the last pivot of a front: its deferred scaling, then U^T (the upper triangle of the
// fully summed square moves to Q) and the unit diagonals. task: (s)
template <typename T>
__global__ void __launch_bounds__(1024) k_lu_finish(DevSym S, const Task* __restrict__ tasks,
                                                   T* __restrict__ factor, T* __restrict__ ufactor,
                                                   const T* __restrict__ dvec, int32_t* __restrict__ piv) {
    constexpr int NT = 1024;
    const int s = tasks[blockIdx.x].s;
    const int f = S.fnrows[s], w = S.fncols[s], c0 = S.super_ptr[s], tid = threadIdx.x;
    T* P = factor + S.panel_off[s];
    T* Q = ufactor + S.panel_off[s];
    LuFront<T> Fr{P, Q, f, w};
    const T dp = dvec[c0 + w - 1];
    for (int i = w + tid; i < f; i += NT) Fr.l(i, w - 1) = Fr.l(i, w - 1) / dp;
    for (int j = w + tid; j < f; j += NT) {
        T& x = Fr.at(w - 1, j);
        x = x / dp;
    }
    __syncthreads();
    // U^T: eight entries per thread per pass, their loads in flight together (clamped to the
    // square), then the stores of those below the diagonal
    const int ww = w * w;
    for (int q0 = 0; q0 < ww; q0 += 8 * NT) {
        T v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int q = min(q0 + tid + u * NT, ww - 1), j = q / w, i = q - j * w;
            v[u] = P[(int64_t)i * f + j];
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int q = q0 + tid + u * NT, j = q / w, i = q - j * w;
            if (q < ww && i > j) Q[(int64_t)j * f + i] = v[u];
        }
    }
    __syncthreads();
    for (int q = tid; q < w * w; q += NT) {
        const int j = q / w, i = q - j * w;
        if (i <= j) {
            P[(int64_t)j * f + i] = i == j ? T(1) : T(0);
            Q[(int64_t)j * f + i] = i == j ? T(1) : T(0);
        }
    }
    for (int q = tid; q < w; q += NT) piv[c0 + q] = c0 + piv[c0 + q];
}

// ---------------------------------------------------------------------------
// large fronts in panels of NBP columns, three launches each: k_lu_panel (one workgroup per front)
// takes the panel's pivots with its columns in registers (thread t: the rows k0 + t + NT u, R rows,
// R NBP entries); k_lu_urows forms the panel's U rows in every column after it (a thread per
// column); k_lu_trail (64 x 64 tiles) applies the panel to the fully summed columns and to U12. Each
// entry goes through the operations of lu_front above, in the same order: L = a / d first, then
// a - L u with the unscaled row entry u, and U = u / d stored in its place in Q.
//
// A pivot of k_lu_panel costs one barrier: the column's two maxima (all rows for the threshold, the
// fully summed rows below for the row choice) by lane reductions, the scaling, the rank-1 update of
// the panel's later columns, which moves each column one register to the left. An interchange adds
// two barriers (the row of the largest entry, the two rows through LDS) and exchanges the two
// rows of the columns in memory (L, the columns after the panel, U12).

template <typename T, int R, int NBP>
struct LuPanel {
    T x[R][NBP];  // x[u][c] = entry (k0 + tid + NT u, k + c)
    int nr;       // row slots in use
    int buf;
};
template <typename T, int NBP>
struct LuPanelLds {
    __align__(16) double red[2][512 / 64][2];
    int found[512 / 64];
    __align__(16) T urow[2][NBP];
    __align__(16) T rrow[NBP];
};
struct LuPrm {
    int pivoting;
    double u, eps;
};

// pivots k, k + 1, ... of the panel while its remaining columns number more than W - 8 (of W registers
// per row)
template <typename T, int NT, int R, int NBP, int W>
__device__ __attribute__((always_inline)) inline void lu_panel_pivots(LuPanel<T, R, NBP>& X, const LuFront<T>& F, int k0,
                                                                      int& k, int kend, const LuPrm& p,
                                                                      LuPanelLds<T, NBP>& D, int* lp, int8_t* kind,
                                                                      T* dd, int64_t* st) {
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, f = F.f, w = F.w;
    const int kstop = min(kend, k0 + NBP - (W > 8 ? W - 8 : 0));
    while (k < kstop) {
        const PanelRows<NT, (int)sizeof(T)> rw(k0, f);
        const int nf = rw.count(f), nw = rw.count(w);
        const bool up = tid > k - k0;  // (the pivot's row is among the first slot's)
        double lam = 0.0, mx = 0.0;
        bool nan = false;
#pragma unroll
        for (int u = 0; u < R; ++u) {
            if (u < X.nr) {  // (only the last slot can hold rows past the front's end)
                double a = (double)X.x[u][0];
                if (u == 0) a = tid >= k - k0 ? a : 0.0;
                if (u + 1 == X.nr) a = u < nf ? a : 0.0;
                nan |= a != a;
                mx = max_abs(mx, a);
                if (NT * u < w - k0) lam = max_abs(lam, u < nw && (u > 0 || up) ? a : 0.0);
            }
        }
        lam = wave_max_last(lam);
        mx = wave_max_last(mx);
        if (__any(nan)) mx = __builtin_nan("");
        X.buf ^= 1;
        if (lane == 63) {
            D.red[X.buf][wv][0] = lam;
            D.red[X.buf][wv][1] = mx;
        }
        if (tid == k - k0) {
#pragma unroll
            for (int c = 0; c < W; ++c) D.urow[X.buf][c] = X.x[0][c];
        }
        __syncthreads();  // (waits for LDS only: the L columns' stores stay in flight)
        nan = false;
        lam = 0.0;
        mx = 0.0;
#pragma unroll
        for (int q = 0; q < NT / 64; ++q) {
            lam = max_abs(lam, D.red[X.buf][q][0]);
            const double v = D.red[X.buf][q][1];
            nan |= v != v;
            mx = max_abs(mx, v);
        }
        const double akk = fabs((double)D.urow[X.buf][0]);
        // keep the diagonal when |a_kk| >= u max |a_ik|; else the largest fully summed row, the first
        // on ties, k if none is larger
        if (uni(p.pivoting && !(!nan && akk >= p.u * mx) && lam > akk)) {
            int ri = 0x7fffffff;
#pragma unroll
            for (int u = R - 1; u >= 0; --u)
                if (u < nw && (u > 0 || up) && fabs((double)X.x[u][0]) == lam) ri = k0 + tid + NT * u;
            ri = wave_min_last(ri);
            if (lane == 63) D.found[wv] = ri;
            __syncthreads();
            int r = D.found[0];
#pragma unroll
            for (int q = 1; q < NT / 64; ++q) r = min(r, D.found[q]);
            r = uni(r);
            // rows k and r of the panel's columns through LDS (the old row k is in urow)
            const int ur = (r - k0) / NT, tr = r - k0 - ur * NT;
#pragma unroll
            for (int u = 0; u < R; ++u)
                if (u == ur && tid == tr) {
#pragma unroll
                    for (int c = 0; c < W; ++c) {
                        D.rrow[c] = X.x[u][c];
                        X.x[u][c] = D.urow[X.buf][c];
                    }
                }
            __syncthreads();
            if (tid < W) D.urow[X.buf][tid] = D.rrow[tid];
            for (int j = tid; j < w; j += NT)
                if (j < k || j >= kend) {
                    T& a = F.l(k, j);
                    T& b = F.l(r, j);
                    const T t = a;
                    a = b;
                    b = t;
                }
            for (int j = w + tid; j < f; j += NT) {
                T& a = F.u(k, j);
                T& b = F.u(r, j);
                const T t = a;
                a = b;
                b = t;
            }
            if (tid == 0) {
                const int t = lp[k];
                lp[k] = lp[r];
                lp[r] = t;
            }
            __syncthreads();
        }
        double dk = (double)D.urow[X.buf][0];
        const bool pert = !(fabs(dk) >= p.eps) || dk == 0.0;
        if (tid == 0) {
            kind[k] = pert ? KIND_PERTURBED : KIND_1X1;
            if (pert) {
                if (dk == 0.0) st[LST_NZERO]++;
                st[LST_NPERT]++;
            }
        }
        if (pert) dk = (dk < 0.0 ? -1.0 : 1.0) * p.eps;
        const T d = T(dk);
        if (tid == 0) {
            if (pert && dk == 0.0 && st[LST_INFO] == 0) st[LST_INFO] = k + 1;
            dd[k] = d;
        }
        // row k of U in the panel's later columns
        if (tid > 0 && tid < min(W, kend - k)) F.Q[(int64_t)k * f + k + tid] = D.urow[X.buf][tid] / d;
        T* col = F.P + (int64_t)k * f;
        // the scaling of three row slots at a time (independent divisions), then their updates
#pragma unroll
        for (int u0 = 0; u0 < R; u0 += 3) {
            if (u0 < X.nr) {
                T l[3] = {};
#pragma unroll
                for (int u = 0; u < 3 && u0 + u < R; ++u) l[u] = X.x[u0 + u][0] / d;
                pin<3>(l);
#pragma unroll
                for (int u = 0; u < 3 && u0 + u < R; ++u) {
                    if (u0 + u < nf && (u0 + u > 0 || up)) store_at(col, rw.off(u0 + u), l[u]);
                    shift_update<W>(X.x[u0 + u], l[u], D.urow[X.buf]);
                }
            }
        }
        ++k;
    }
}

// the panel of columns [k0, k0 + NBP) of every large front of a level that has them. task: (s)
//
// Bound: latency, one workgroup per front walks the pivots one after another. NT = 512 (two waves
// per SIMD) leaves 256 registers a thread, 192 of them for the panel: NBP R <= 96. 32 x 32 x 32
// convection-diffusion, FP64: 71 us a launch of 32 columns, 2.2 us a pivot; one pivot per launch pair
// took 13.5 us, a gradient step 72.3 ms instead of 24.6.
template <typename T, int R, int NBP>
__global__ void __launch_bounds__(512) k_lu_panel(DevSym S, const Task* __restrict__ tasks, int k0,
                                                  T* __restrict__ factor, T* __restrict__ ufactor,
                                                  T* __restrict__ dvec, int32_t* __restrict__ piv,
                                                  int8_t* __restrict__ pkind, int64_t* __restrict__ stats, LuPrm prm,
                                                  int scaled, const double* __restrict__ aux) {
    constexpr int NT = 512;
    __shared__ LuPanelLds<T, NBP> D;
    const int s = tasks[blockIdx.x].s;
    const int f = S.fnrows[s], w = S.fncols[s];
    if (k0 >= w) return;
    const int c0 = S.super_ptr[s], tid = threadIdx.x;
    if (scaled && aux[0] > 0) prm.eps = prm.eps * aux[0];
    const LuFront<T> F{factor + S.panel_off[s], ufactor + S.panel_off[s], f, w};
    int* lp = piv + c0;
    int8_t* kind = pkind + c0;
    T* dd = dvec + c0;
    int64_t* st = stats + (int64_t)s * NF;
    if (k0 == 0) {
        for (int q = tid; q < w; q += NT) {
            lp[q] = q;
            dvec[S.n + c0 + q] = T(0);
        }
        if (tid < NF) st[tid] = 0;
    }
    const int kend = min(w, k0 + NBP);
    LuPanel<T, R, NBP> X;
    X.nr = (f - k0 + NT - 1) / NT;
    X.buf = 0;
    {
        const PanelRows<NT, (int)sizeof(T)> rw(k0, f);
#pragma unroll
        for (int u = 0; u < R; ++u) {
            const uint32_t off = rw.clamped(u);
#pragma unroll
            for (int c = 0; c < NBP; ++c) X.x[u][c] = load_at(F.P + (int64_t)min(k0 + c, w - 1) * f, off);
        }
    }
    __syncthreads();
    int k = k0;
    if constexpr (NBP > 24) lu_panel_pivots<T, NT, R, NBP, 32>(X, F, k0, k, kend, prm, D, lp, kind, dd, st);
    if constexpr (NBP > 16) lu_panel_pivots<T, NT, R, NBP, 24>(X, F, k0, k, kend, prm, D, lp, kind, dd, st);
    if constexpr (NBP > 8) lu_panel_pivots<T, NT, R, NBP, 16>(X, F, k0, k, kend, prm, D, lp, kind, dd, st);
    lu_panel_pivots<T, NT, R, NBP, (NBP < 8 ? NBP : 8)>(X, F, k0, k, kend, prm, D, lp, kind, dd, st);
}

// the U rows of a panel's pivots k0 .. k0 + np - 1 in the 64 columns from J0 (after the panel): u = a -
// L u in pivot order, a thread per column with all its np entries in registers, loaded together; the
// unscaled rows go to the front's scratch (U[q f + j], read by k_lu_trail), u / d to Q. task: (s, J0,
// 0, scratch offset). Bound: latency, one wave per 64 columns: the chain of 32 pivots after one
// round of loads (eight rows at a time, each block read the rows before it back from the scratch:
// 16.8 us a launch of a 32 x 32 x 32 LU in FP64, 10.7 now).
constexpr int LU_PANEL_MAX = 32;  // most columns of a panel

template <typename T>
__global__ void __launch_bounds__(64) k_lu_urows(DevSym S, const Task* __restrict__ tasks, int k0, int cols,
                                                 const T* __restrict__ factor, T* __restrict__ ufactor,
                                                 const T* __restrict__ dvec, T* __restrict__ scratch) {
    __shared__ __align__(16) T Lc[LU_PANEL_MAX][LU_PANEL_MAX];  // Lc[q][r] = L(k0 + r, k0 + q)
    const Task t = tasks[blockIdx.x];
    const int s = t.s, f = S.fnrows[s], w = S.fncols[s];
    if (k0 >= w) return;
    const int np = min(cols, w - k0), j = t.a + threadIdx.x;
    if (t.a + 64 <= k0 + np) return;
    const T* P = factor + S.panel_off[s];
    T* Q = ufactor + S.panel_off[s];
    const T* dd = dvec + S.super_ptr[s] + k0;
    T* U = scratch + (int64_t)t.c * PANEL_SCR_UNIT;
    const bool on = j >= k0 + np && j < f;
    const int jc = min(max(j, k0 + np), f - 1);  // (np < f - k0 in a front with columns after the panel)
    // row r of the column in P (fully summed) or of U12, stored by rows, in Q; blocks of eight rows up to
    // np: rows past np in the last block repeat row np - 1 and are neither stored nor read by others
    const T* col = jc < w ? P + (int64_t)jc * f + k0 : Q + (int64_t)k0 * f + jc;
    const int64_t step = jc < w ? 1 : f;
    T a[LU_PANEL_MAX];
#pragma unroll
    for (int g = 0; g < LU_PANEL_MAX; g += 8)
        if (g < np) {
#pragma unroll
            for (int r = 0; r < 8; ++r) a[g + r] = col[min(g + r, np - 1) * step];
        }
    const int lane = threadIdx.x;
    T lv[LU_PANEL_MAX / 2];
#pragma unroll
    for (int u = 0; u < LU_PANEL_MAX / 2; ++u) {
        const int c = 2 * u + (lane >> 5), r = lane & 31;
        lv[u] = P[(int64_t)(k0 + min(c, np - 1)) * f + k0 + min(r, np - 1)];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < LU_PANEL_MAX / 2; ++u) Lc[2 * u + (lane >> 5)][lane & 31] = lv[u];
    __syncthreads();
#pragma unroll
    for (int g = 0; g < LU_PANEL_MAX; g += 8)
        if (g < np) {
#pragma unroll
            for (int r = g; r < g + 8; ++r) {
#pragma unroll
                for (int r2 = r + 1; r2 < g + 8; ++r2) a[r2] = a[r2] - Lc[r][r2] * a[r];
            }
            // the block's rows in the rows after it
#pragma unroll
            for (int h = g + 8; h < LU_PANEL_MAX; h += 8)
                if (h < np) {
#pragma unroll
                    for (int r = g; r < g + 8; ++r)
#pragma unroll
                        for (int r2 = h; r2 < h + 8; ++r2) a[r2] = a[r2] - Lc[r][r2] * a[r];
                }
#pragma unroll
            for (int r = g; r < g + 8; ++r)
                if (on && r < np) {
                    U[(int64_t)r * f + j] = a[r];
                    Q[(int64_t)(k0 + r) * f + j] = a[r] / dd[r];
                }
        }
}

// a panel's update of the entries after it: tile (s, I0, J0, scratch offset) of 64 x 64 entries, J0 < w: the
// fully summed columns (every row), J0 >= w: U12 (the fully summed rows, stored transposed), each
// entry a - L u in pivot order. Lanes along the contiguous direction, sixteen entries a thread loaded
// together; the panel's factor along the lanes in registers, the other from LDS by broadcast.
// Bound: HBM / L2 (two accesses per entry and panel): 12.6 us a launch of a 32 x 32 x 32 LU.
template <typename T>
__global__ void __launch_bounds__(256) k_lu_trail(DevSym S, const Task* __restrict__ tasks, int k0, int cols,
                                                  T* __restrict__ factor, T* __restrict__ ufactor,
                                                  const T* __restrict__ scratch) {
    __shared__ __align__(16) T Bs[LU_PANEL_MAX][TILE];
    const Task t = tasks[blockIdx.x];
    const int s = t.s, f = S.fnrows[s], w = S.fncols[s];
    if (k0 >= w) return;
    const int np = min(cols, w - k0), kend = k0 + np;
    const int I0 = t.a, J0 = t.b;
    if (I0 + TILE <= kend || J0 + TILE <= kend) return;
    T* P = factor + S.panel_off[s];
    T* Q = ufactor + S.panel_off[s];
    const T* U = scratch + (int64_t)t.c * PANEL_SCR_UNIT;
    const int tid = threadIdx.x, lane = tid & 63, cb = (tid >> 6) * 16;
    const bool u12 = J0 >= w;
    // element c of the thread: row `lane`, column cb + c (P), or column `lane`, row cb + c (Q); A: the
    // panel's factor along the lanes, B along c
    const T* A = u12 ? U + min(J0 + lane, f - 1) : P + (int64_t)k0 * f + min(I0 + lane, f - 1);
    const T* B = u12 ? P + (int64_t)k0 * f + I0 : U + J0;
    const int nb = (u12 ? w - I0 : w - J0);  // rows / columns of the tile that exist
    for (int q = tid; q < np * TILE; q += 256) {
        const int pp = q / TILE, c = q - pp * TILE;
        Bs[pp][c] = B[(int64_t)pp * f + min(c, nb - 1)];
    }
    T* X = u12 ? Q + (int64_t)I0 * f + min(J0 + lane, f - 1) : P + (int64_t)J0 * f + min(I0 + lane, f - 1);
    T x[16];
#pragma unroll
    for (int c = 0; c < 16; ++c) x[c] = X[(int64_t)min(cb + c, nb - 1) * f];
    __syncthreads();
    for (int q0 = 0; q0 < np; q0 += 8) {
        T a[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) a[q] = A[(int64_t)min(q0 + q, np - 1) * f];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            if (q0 + q >= np) break;
#pragma unroll
            for (int c = 0; c < 16; ++c) x[c] = x[c] - a[q] * Bs[q0 + q][cb + c];
        }
    }
    const int il = (u12 ? J0 : I0) + lane, ic = (u12 ? I0 : J0) + cb;
    if (il >= f || il < kend) return;
#pragma unroll
    for (int c = 0; c < 16; ++c)
        if (ic + c >= kend && cb + c < nb) X[(int64_t)(cb + c) * f] = x[c];
}

// after the last panel: unit diagonals and empty upper triangles of both panels, the global pivot
// order. task: (s, I0, J0), a 64 x 64 tile of the fully summed square with I0 <= J0
template <typename T>
__global__ void __launch_bounds__(256) k_lu_unit(DevSym S, const Task* __restrict__ tasks, T* __restrict__ factor,
                                                 T* __restrict__ ufactor, int32_t* __restrict__ piv) {
    const Task t = tasks[blockIdx.x];
    const int s = t.s, f = S.fnrows[s], w = S.fncols[s], c0 = S.super_ptr[s];
    const int i = t.a + (threadIdx.x & 63);
    T* P = factor + S.panel_off[s];
    T* Q = ufactor + S.panel_off[s];
    for (int j = t.b + (threadIdx.x >> 6); j < min(t.b + 64, w); j += 4)
        if (i <= j) {
            P[(int64_t)j * f + i] = i == j ? T(1) : T(0);
            Q[(int64_t)j * f + i] = i == j ? T(1) : T(0);
        }
    if (t.a == t.b && threadIdx.x < 64 && i < w) piv[c0 + i] = c0 + piv[c0 + i];
}

// F22 <- F22 - (L21 D) U12 by 64 x 64 tiles (I0, J0 front rows/columns >= w), each entry's
// sum over k = 0, 1, ..., w - 1 in order. L21 D and U12 in chunks of 16 columns in LDS.
template <typename T>
__global__ void __launch_bounds__(256) k_lu_cb(DevSym S, const Task* __restrict__ tasks,
                                              const T* __restrict__ factor, const T* __restrict__ ufactor,
                                              T* __restrict__ cbpool, const T* __restrict__ dvec) {
    constexpr int KC = 16;
    __shared__ T Ws[KC][TILE];
    __shared__ T Us[KC][TILE];
    const Task t = tasks[blockIdx.x];
    const int s = t.s, f = S.fnrows[s], w = S.fncols[s], m = f - w;
    const int I0 = t.a, J0 = t.b;
    const int c0 = S.super_ptr[s];
    const T* L = factor + S.panel_off[s];
    const T* Q = ufactor + S.panel_off[s];
    T* C = cbpool + S.cb_off[s];
    const T* dd = dvec + c0;
    const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
    T acc[4][4];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[a][b] = T(0);
    // the thread's four (kk, c) staging slots, kk = (tid >> 6) + 4 u, c = tid & 63: the raw
    // values of chunk k0 + KC are loaded, clamped, while chunk k0 is multiplied
    const int c = tid & 63, ic = min(I0 + c, f - 1), jc = min(J0 + c, f - 1);
    T lv[4], dv[4], uv0[4];
    auto load_raw = [&](int k0) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int kc = min(k0 + (tid >> 6) + 4 * u, w - 1);
            lv[u] = L[(int64_t)kc * f + ic];
            dv[u] = dd[kc];
            uv0[u] = Q[(int64_t)kc * f + jc];
        }
    };
    load_raw(0);
    for (int k0 = 0; k0 < w; k0 += KC) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int kk = (tid >> 6) + 4 * u, k = k0 + kk;
            Ws[kk][c] = (k < w && I0 + c < f) ? lv[u] * dv[u] : T(0);
            Us[kk][c] = (k < w && J0 + c < f) ? uv0[u] : T(0);
        }
        __syncthreads();
        if (k0 + KC < w) load_raw(k0 + KC);
        const int kn = min(KC, w - k0);
        for (int kk = 0; kk < kn; ++kk) {
            T wv[4], uv[4];
#pragma unroll
            for (int a = 0; a < 4; ++a) wv[a] = Ws[kk][4 * ty + a];
#pragma unroll
            for (int b = 0; b < 4; ++b) uv[b] = Us[kk][4 * tx + b];
#pragma unroll
            for (int a = 0; a < 4; ++a)
#pragma unroll
                for (int b = 0; b < 4; ++b) acc[a][b] = acc[a][b] + wv[a] * uv[b];
        }
        __syncthreads();
    }
    // the tile's old values loaded together (clamped), then the masked stores
    T old[4][4];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const int i = min(I0 + 4 * ty + a, f - 1), j = min(J0 + 4 * tx + b, f - 1);
            old[a][b] = C[(int64_t)(j - w) * m + (i - w)];
        }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const int i = I0 + 4 * ty + a, j = J0 + 4 * tx + b;
            if (i < f && j < f) C[(int64_t)(j - w) * m + (i - w)] = old[a][b] - acc[a][b];
        }
}

// ---------------------------------------------------------------------------

template <typename T>
void launch_front_small_lu(hipStream_t st, const DevSym& S, const int32_t* fronts, int nfronts, int fmax,
                           const double* nz, T* factor, T* ufactor, T* cbpool, T* dvec, int32_t* piv, int8_t* kind,
                           int64_t* stats, int pivoting, double u, double eps, int scaled, const double* aux) {
    size_t lds = (size_t)fmax * fmax * sizeof(T);
    hipLaunchKernelGGL(k_front_small_lu<T>, dim3(nfronts), dim3(256), lds, st, S, fronts, nz, factor, ufactor, cbpool,
                       dvec, piv, kind, stats, pivoting, u, eps, scaled, aux);
}

template <typename T>
void launch_big_lu_zero(hipStream_t st, const DevSym& S, const Task* tasks, int n, T* factor, T* ufactor, T* cbpool) {
    hipLaunchKernelGGL(k_big_lu_zero<T>, dim3(n), dim3(256), 0, st, S, tasks, factor, ufactor, cbpool);
}

template <typename T>
void launch_big_lu_scatter(hipStream_t st, const DevSym& S, const Task* tasks, int n, const double* nz, T* factor,
                           T* ufactor) {
    hipLaunchKernelGGL(k_big_lu_scatter<T>, dim3(n), dim3(256), 0, st, S, tasks, nz, factor, ufactor);
}

template <typename T>
void launch_big_lu_extend_add(hipStream_t st, const DevSym& S, const Task* tasks, int n, T* factor, T* ufactor,
                              T* cbpool) {
    hipLaunchKernelGGL(k_big_lu_extend_add<T>, dim3(n), dim3(256), 0, st, S, tasks, factor, ufactor, cbpool);
}

template <typename T>
void launch_lu_pivot(hipStream_t st, const DevSym& S, const Task* tasks, int n, int k, T* factor, T* ufactor,
                     T* dvec, int32_t* piv, int8_t* kind, int64_t* stats, int pivoting, double u, double eps,
                     int scaled, const double* aux) {
    hipLaunchKernelGGL(k_lu_pivot<T>, dim3(n), dim3(1024), 0, st, S, tasks, k, factor, ufactor, dvec, piv, kind,
                       stats, pivoting, u, eps, scaled, aux);
}

template <typename T>
void launch_lu_update(hipStream_t st, const DevSym& S, const Task* tasks, int n, int k, T* factor, T* ufactor,
                      const T* dvec) {
    hipLaunchKernelGGL(k_lu_update<T>, dim3(n), dim3(256), 0, st, S, tasks, k, factor, ufactor, dvec);
}

template <typename T>
void launch_lu_finish(hipStream_t st, const DevSym& S, const Task* tasks, int n, T* factor, T* ufactor,
                      const T* dvec, int32_t* piv) {
    hipLaunchKernelGGL(k_lu_finish<T>, dim3(n), dim3(1024), 0, st, S, tasks, factor, ufactor, dvec, piv);
}

template <typename T>
void launch_lu_panel(hipStream_t st, const DevSym& S, const Task* tasks, int n, int k0, int cols, T* factor,
                     T* ufactor, T* dvec, int32_t* piv, int8_t* kind, int64_t* stats, int pivoting, double u,
                     double eps, int scaled, const double* aux) {
    const LuPrm p{pivoting, u, eps};
#define PANEL(R, C)                                                                                                  \
    hipLaunchKernelGGL((k_lu_panel<T, R, C>), dim3(n), dim3(512), 0, st, S, tasks, k0, factor, ufactor, dvec, piv,   \
                       kind, stats, p, scaled, aux)
    switch (cols) {
        case 32: PANEL(3, 32); break;
        case 16: PANEL(6, 16); break;
        case 8: PANEL(10, 8); break;
        default: PANEL(20, 4); break;
    }
#undef PANEL
}

// columns of the next panel of fronts with at most `rows` rows and `cols` columns left (0: too tall
// for the registers of one workgroup). The widest panel whose rows fit: a panel pays three launches
// and its loads and stores once, whatever its columns; no wider than the columns left need. Measured
// with all three launches: 32 columns 2.9 us a pivot, against 13.5 us of a launch pair.
int lu_panel_cols(int rows, int cols) {
    if (rows <= 3 * 512 && cols > 16) return 32;
    if (rows <= 6 * 512 && cols > 8) return 16;
    if (rows <= 10 * 512) return 8;
    return rows <= 20 * 512 ? 4 : 0;
}

template <typename T>
void launch_lu_urows(hipStream_t st, const DevSym& S, const Task* tasks, int n, int k0, int cols, const T* factor,
                     T* ufactor, const T* dvec, T* scratch) {
    hipLaunchKernelGGL(k_lu_urows<T>, dim3(n), dim3(64), 0, st, S, tasks, k0, cols, factor, ufactor, dvec, scratch);
}

template <typename T>
void launch_lu_trail(hipStream_t st, const DevSym& S, const Task* tasks, int n, int k0, int cols, T* factor,
                     T* ufactor, const T* scratch) {
    hipLaunchKernelGGL(k_lu_trail<T>, dim3(n), dim3(256), 0, st, S, tasks, k0, cols, factor, ufactor, scratch);
}

template <typename T>
void launch_lu_unit(hipStream_t st, const DevSym& S, const Task* tasks, int n, T* factor, T* ufactor, int32_t* piv) {
    hipLaunchKernelGGL(k_lu_unit<T>, dim3(n), dim3(256), 0, st, S, tasks, factor, ufactor, piv);
}

template <typename T>
void launch_lu_cb(hipStream_t st, const DevSym& S, const Task* tasks, int n, const T* factor, const T* ufactor,
                  T* cbpool, const T* dvec) {
    hipLaunchKernelGGL(k_lu_cb<T>, dim3(n), dim3(256), 0, st, S, tasks, factor, ufactor, cbpool, dvec);
}

#define INST(T)                                                                                                      \
    template void launch_front_small_lu<T>(hipStream_t, const DevSym&, const int32_t*, int, int, const double*, T*, \
                                           T*, T*, T*, int32_t*, int8_t*, int64_t*, int, double, double, int,       \
                                           const double*);                                                          \
    template void launch_big_lu_zero<T>(hipStream_t, const DevSym&, const Task*, int, T*, T*, T*);                  \
    template void launch_big_lu_scatter<T>(hipStream_t, const DevSym&, const Task*, int, const double*, T*, T*);    \
    template void launch_big_lu_extend_add<T>(hipStream_t, const DevSym&, const Task*, int, T*, T*, T*);            \
    template void launch_lu_cb<T>(hipStream_t, const DevSym&, const Task*, int, const T*, const T*, T*, const T*); \
    template void launch_lu_pivot<T>(hipStream_t, const DevSym&, const Task*, int, int, T*, T*, T*, int32_t*,      \
                                     int8_t*, int64_t*, int, double, double, int, const double*);                   \
    template void launch_lu_update<T>(hipStream_t, const DevSym&, const Task*, int, int, T*, T*, const T*);         \
    template void launch_lu_panel<T>(hipStream_t, const DevSym&, const Task*, int, int, int, T*, T*, T*, int32_t*, \
                                     int8_t*, int64_t*, int, double, double, int, const double*);                   \
    template void launch_lu_urows<T>(hipStream_t, const DevSym&, const Task*, int, int, int, const T*, T*,          \
                                     const T*, T*);                                                                 \
    template void launch_lu_trail<T>(hipStream_t, const DevSym&, const Task*, int, int, int, T*, T*, const T*);     \
    template void launch_lu_unit<T>(hipStream_t, const DevSym&, const Task*, int, T*, T*, int32_t*);                \
    template void launch_lu_finish<T>(hipStream_t, const DevSym&, const Task*, int, T*, T*, const T*, int32_t*);
INST(double)
INST(float)
#undef INST

}  // namespace sds
