// LDL^T factorization kernels (gfx950) with diagonal and Bunch-Kaufman pivoting inside
// each front's fully summed block, threshold test against the whole remaining column,
// best-1x1 fallback and static perturbation (+-eps, optionally with requested signs).
//
// Every floating-point operation of the factorization is the one the CPU reference
// performs, in the same order, with no fused multiply-add (the file is compiled with
// contraction off): a front's pivot decisions, factor, D and contribution block are
// bitwise those of src/reference/ldlt.jl in FP64. The pivot search reductions
// (column maxima, argmax with the first index on ties) are order-independent, so they
// run as parallel reductions.
//
// Small fronts (f x f fits the LDS) are assembled, factored and their contribution
// block formed in one workgroup; large fronts are assembled in global memory by the
// shared column-chunk and extend-add kernels and factored on the panel in place (the full
// w x w fully summed block lives in the panel's top rows, the upper triangle being the
// mirror the reference keeps), in panels of 4 to 16 pivot columns held in one workgroup's registers,
// each followed by its update of the columns after it by 64 x 64 tiles over the GPU (fronts too
// tall for that: one pivot per pair of launches); then their contribution block is updated by
// 64 x 64 tiles, each entry subtracting the terms W[i, k] L[j, k] in the order k = 0, 1, ... of the
// reference.
//
// Reference counterparts: ref_ldlt! and _ldlt_front! (src/reference/ldlt.jl:121-202,
// :384-454), _choose_pivot (:280-325), _best_1x1 (:264-276), the threshold test
// (:252-260), the 2x2 test (:240-248), W = L21 D and the Schur update (:206-231);
// device statistics src/numeric/ldlt.jl:1276-1356.
#pragma clang fp contract(off)
#include "k_front.h"
#include "k_panel.h"
#include "panel_plan.h"
#include "sds_common.h"
#include "sds_kernels.h"

namespace sds {

enum { PV_NONE = 0, PV_DIAG = 1, PV_BK = 2 };
enum { ST_NPOS = 0, ST_NNEG = 1, ST_NZERO = 2, ST_NPERT = 3, ST_N2X2 = 4, ST_INFO = 5 };

// max that propagates NaN, as Julia's max
__device__ inline double jmax(double a, double b) {
    if (a != a || b != b) return a + b;
    return a > b ? a : b;
}

// (value, index) pairs of the argmax reductions: index < 0 = no candidate; a larger value
// wins, equal values keep the smaller index (the first one a sequential scan meets)
__device__ inline bool vi_better(double ov, int oi, double v, int i) {
    if (oi < 0) return false;
    if (i < 0) return true;
    return ov > v || (ov == v && oi < i);
}

template <int NT>
struct RedBuf {
    double v[NT / 64];
    int i[NT / 64];
};

// (values >= 0) every lane gets the wave's maximum
__device__ inline double wave_jmax(double v) {
    const double m = last_lane(wave_max_last(v));
    return __any(v != v) ? __builtin_nan("") : m;
}

// (candidates' values >= 0) every lane gets the wave's best candidate; a NaN value, which every
// lane then holds, stays
__device__ inline void wave_argmax(double& v, int& i) {
    const double m = last_lane(wave_max_last(i >= 0 ? v : 0.0));
    const int first = __builtin_amdgcn_readlane(wave_min_last(i >= 0 && v == m ? i : 0x7fffffff), 63);
    if (first != 0x7fffffff) {
        v = m;
        i = first;
    }
}

// block-wide reductions: every thread gets the same result
template <int NT>
__device__ double block_jmax(double v, RedBuf<NT>& rb) {
    v = wave_jmax(v);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (lane == 0) rb.v[wv] = v;
    __syncthreads();
    double r = rb.v[0];
    for (int q = 1; q < NT / 64; ++q) r = jmax(r, rb.v[q]);
    __syncthreads();
    return r;
}

template <int NT>
__device__ void block_argmax(double& v, int& i, RedBuf<NT>& rb) {
    wave_argmax(v, i);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (lane == 0) {
        rb.v[wv] = v;
        rb.i[wv] = i;
    }
    __syncthreads();
    v = rb.v[0];
    i = rb.i[0];
    for (int q = 1; q < NT / 64; ++q)
        if (vi_better(rb.v[q], rb.i[q], v, i)) {
            v = rb.v[q];
            i = rb.i[q];
        }
    __syncthreads();
}

struct LdltPrm {
    int pivot;
    double u, eps;
};

// the front view of one factorization: F is f x f column-major (LDS or the panel), only
// columns < w are touched; lp is the local pivot order (original positions)
template <typename T, int NT>
struct Front {
    T* F;
    int f, w;
    int* lp;
    RedBuf<NT>* rb;
    double* skey = nullptr;  // LDS scratch of best_1x1_sorted (scap entries), or none
    int* sidx = nullptr;
    int scap = 0;
    __device__ double at(int i, int j) const { return (double)F[(int64_t)j * f + i]; }
    __device__ T& ref(int i, int j) const { return F[(int64_t)j * f + i]; }

    // largest |F[i, c]| over the rows k..f-1 but s1 and s2, NaN-propagating (ldlt.jl:240-260)
    __device__ double colmax(int c, int k, int s1, int s2) const {
        double m = 0.0;
        for (int i = k + threadIdx.x; i < f; i += NT)
            if (i != s1 && i != s2) m = jmax(m, fabs(at(i, c)));
        return block_jmax<NT>(m, *rb);
    }
    // d >= u max_{i in k..f-1, i != c} |F[i, c]| (the early exit of the reference is the same
    // predicate: the running maximum only grows)
    __device__ bool accept_1x1(int c, int k, const LdltPrm& p) const {
        const double d = fabs(at(c, c));
        if (!(d >= p.eps)) return false;
        return d >= p.u * colmax(c, k, c, -1);
    }
    __device__ bool nonsingular_2x2(int k, int r, const LdltPrm& p) const {
        const double det = at(k, k) * at(r, r) - at(k, r) * at(r, k);
        const double mx = jmax(jmax(fabs(at(k, k)), fabs(at(r, k))), fabs(at(r, r)));
        return det != 0.0 && isfinite(det) && mx >= p.eps;
    }
    __device__ bool accept_2x2(int k, int r, const LdltPrm& p) const {
        if (!nonsingular_2x2(k, r, p)) return false;
        const double det = at(k, k) * at(r, r) - at(k, r) * at(r, k);
        const double e11 = fabs(at(r, r) / det), e12 = fabs(at(k, r) / det), e21 = fabs(at(r, k) / det),
                     e22 = fabs(at(k, k) / det);
        const double m1 = colmax(k, k, k, r), m2 = colmax(r, k, r, k);
        return p.u * (e11 * m1 + e21 * m2) <= 1.0 && p.u * (e12 * m1 + e22 * m2) <= 1.0;
    }
    // acceptable 1x1 pivot of the block k..w-1 with the largest |a_jj|, first on ties; -1 if
    // none (ldlt.jl:264-276). One wave per candidate column; a column that cannot beat its
    // wave's current best is not tested (it cannot be the sequential scan's choice either).
    __device__ int best_1x1(int k, const LdltPrm& p) const {
        const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
        double bv = 0.0;
        int bi = -1;
        for (int j = k + wv; j < w; j += NT / 64) {
            const double a = fabs(at(j, j));
            if (!(a >= p.eps)) continue;
            if (bi >= 0 && !(a > bv)) continue;
            double m = 0.0;
            for (int i = k + lane; i < f; i += 64)
                if (i != j) m = jmax(m, fabs(at(i, j)));
            m = wave_jmax(m);
            if (!(a >= p.u * m)) continue;
            bv = a;
            bi = j;
        }
        // each wave's candidate is wave-uniform; combine across waves
        if (lane == 0) {
            rb->v[wv] = bv;
            rb->i[wv] = bi;
        }
        __syncthreads();
        double v = rb->v[0];
        int i = rb->i[0];
        for (int q = 1; q < NT / 64; ++q)
            if (vi_better(rb->v[q], rb->i[q], v, i)) {
                v = rb->v[q];
                i = rb->i[q];
            }
        __syncthreads();
        return i;
    }
    // best_1x1 for a large front: the candidates sorted by |a_jj| (largest first, the smaller
    // index first on ties; those below eps last), then tested sixteen at a time in that order
    // (one wave per column, the column maximum over all rows below): the first acceptable one
    // in the order is the one the sequential scan of the reference picks. Usually the first
    // round decides, where the scan of every column reads (w - k) f entries.
    __device__ int best_1x1_sorted(int k, const LdltPrm& p) const {
        const int n = w - k, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
        int np = 1;
        while (np < n) np <<= 1;
        for (int q = tid; q < np; q += NT) {
            double key = -1.0;
            if (q < n) {
                const double a = fabs(at(k + q, k + q));
                key = a >= p.eps ? a : -1.0;
            }
            skey[q] = key;
            sidx[q] = k + q;
        }
        __syncthreads();
        // bitonic sort into the order "before(x, y)": key larger, or equal key and smaller index
        for (int size = 2; size <= np; size <<= 1)
            for (int stride = size >> 1; stride > 0; stride >>= 1) {
                for (int i = tid; i < np; i += NT) {
                    const int l = i ^ stride;
                    if (l <= i) continue;
                    const bool lbefore = skey[l] > skey[i] || (skey[l] == skey[i] && sidx[l] < sidx[i]);
                    const bool ibefore = skey[i] > skey[l] || (skey[i] == skey[l] && sidx[i] < sidx[l]);
                    if ((i & size) == 0 ? lbefore : ibefore) {
                        const double tk = skey[i];
                        skey[i] = skey[l];
                        skey[l] = tk;
                        const int ti = sidx[i];
                        sidx[i] = sidx[l];
                        sidx[l] = ti;
                    }
                }
                __syncthreads();
            }
        for (int base = 0; base < n && skey[base] >= 0.0; base += NT / 64) {
            const int q = base + wv;
            int found = 0x7fffffff;
            if (q < n && skey[q] >= 0.0) {
                const int j = sidx[q];
                const double a = skey[q];
                double m = 0.0;
                for (int i = k + lane; i < f; i += 64)
                    if (i != j) m = jmax(m, fabs(at(i, j)));
                m = wave_jmax(m);
                if (a >= p.u * m) found = q;
            }
            if (lane == 0) rb->i[wv] = found;
            __syncthreads();
            int best = rb->i[0];
            for (int w2 = 1; w2 < NT / 64; ++w2) best = min(best, rb->i[w2]);
            __syncthreads();
            if (best != 0x7fffffff) return sidx[best];
        }
        return -1;
    }
    __device__ int best_1x1_any(int k, const LdltPrm& p) const {
        if (!skey || w - k > scap) return best_1x1(k, p);
        // the first candidate in the sorted order (largest |a_jj| >= eps, the smaller index on
        // ties) tested by the whole block first: it usually is the answer
        double v = -1.0;
        int bi = -1;
        for (int j = k + threadIdx.x; j < w; j += NT) {
            const double a = fabs(at(j, j));
            if (a >= p.eps && vi_better(a, j, v, bi)) {
                v = a;
                bi = j;
            }
        }
        block_argmax<NT>(v, bi, *rb);
        if (bi < 0) return -1;
        if (v >= p.u * colmax(bi, k, bi, -1)) return bi;
        return best_1x1_sorted(k, p);
    }
    // pivot choice at column k (ldlt.jl:280-325): c = pivot column, r = 2x2 partner or -1
    __device__ void choose(int k, const LdltPrm& p, int& c, int& r) const {
        r = -1;
        if (p.pivot == PV_NONE) {
            c = k;
            return;
        }
        if (p.pivot == PV_DIAG) {
            if (accept_1x1(k, k, p)) {
                c = k;
                return;
            }
            const int best = best_1x1_any(k, p);
            if (best >= 0) {
                c = best;
                return;
            }
            // the largest diagonal entry, first on ties; a NaN |a_kk| keeps k
            double v = fabs(at(k, k));
            int bi = k;
            for (int j = k + 1 + threadIdx.x; j < w; j += NT) {
                const double a = fabs(at(j, j));
                if (a > v) {
                    v = a;
                    bi = j;
                }
            }
            block_argmax<NT>(v, bi, *rb);
            c = fabs(at(bi, bi)) >= p.eps ? bi : k;
            return;
        }
        const double alpha = (1.0 + sqrt(17.0)) / 8.0;  // Bunch-Kaufman constant (ldlt.jl:22)
        double lambda = 0.0;
        int rr = -1;
        for (int i = k + 1 + threadIdx.x; i < w; i += NT) {
            const double a = fabs(at(i, k));
            if (a > lambda) {
                lambda = a;
                rr = i;
            }
        }
        block_argmax<NT>(lambda, rr, *rb);
        if (rr < 0) lambda = 0.0;
        const double akk = fabs(at(k, k));
        int bc = k, br = -1;
        if (rr < 0 || akk >= alpha * lambda) {
            bc = k;
        } else {
            double sigma = 0.0;
            for (int i = k + threadIdx.x; i < w; i += NT)
                if (i != rr) sigma = jmax(sigma, fabs(at(i, rr)));
            sigma = block_jmax<NT>(sigma, *rb);
            if (akk * sigma >= alpha * lambda * lambda)
                bc = k;
            else if (fabs(at(rr, rr)) >= alpha * sigma)
                bc = rr;
            else {
                bc = k;
                br = rr;
            }
        }
        const bool ok = br < 0 ? accept_1x1(bc, k, p) : accept_2x2(k, br, p);
        if (ok) {
            c = bc;
            r = br;
            return;
        }
        const int best = best_1x1_any(k, p);
        if (best >= 0) {
            c = best;
            return;
        }
        if (br >= 0 && nonsingular_2x2(k, br, p)) {
            c = bc;
            r = br;
            return;
        }
        c = bc;
    }
    // symmetric interchange of positions a and b: columns over all f rows, then rows over the
    // w fully summed columns (ldlt.jl:328-340)
    __device__ void swap(int a, int b) const {
        __syncthreads();  // the pivot choice's last reads of F are done
        if (a == b) return;
        for (int i = threadIdx.x; i < f; i += NT) {
            const T t = ref(i, a);
            ref(i, a) = ref(i, b);
            ref(i, b) = t;
        }
        __syncthreads();
        for (int j = threadIdx.x; j < w; j += NT) {
            const T t = ref(a, j);
            ref(a, j) = ref(b, j);
            ref(b, j) = t;
        }
        if (threadIdx.x == 0) {
            const int t = lp[a];
            lp[a] = lp[b];
            lp[b] = t;
        }
        __syncthreads();
    }
};

// Per-front outputs of the pivot loop.
template <typename T>
struct PivOut {
    int8_t* kind;  // w
    T* dd;         // w: D (1x1 value, or the 2x2 diagonal entries)
    T* ee;         // w: 2x2 subdiagonal at the first position
    int* st;       // NF statistics (shared)
};

// The pivot loop of one front (_ldlt_front!, ldlt.jl:384-454) run by all NT threads.
// sreq (nullable): requested sign of each original local position (psign of its row).
template <typename T, int NT>
__device__ void ldlt_front(const Front<T, NT>& Fr, const LdltPrm& p, const int8_t* sreq_row,
                           const int32_t* perm_c0, PivOut<T> out, double* sh) {
    const int f = Fr.f, w = Fr.w, tid = threadIdx.x;
    int k = 0;
    while (k < w) {
        int c, r;
        Fr.choose(k, p, c, r);
        if (r < 0) {
            Fr.swap(k, c);
            if (tid == 0) {
                double d = Fr.at(k, k);
                int8_t kd = KIND_1X1;
                if (!(fabs(d) >= p.eps) || d == 0.0) {
                    if (d == 0.0) out.st[ST_NZERO]++;
                    const int req = sreq_row ? (int)sreq_row[perm_c0[Fr.lp[k]]] : 0;
                    const double sg = req != 0 ? (double)req : (d < 0.0 ? -1.0 : 1.0);
                    d = sg * p.eps;
                    kd = KIND_PERTURBED;
                    out.st[ST_NPERT]++;
                    if (d == 0.0 && out.st[ST_INFO] == 0) out.st[ST_INFO] = Fr.lp[k] + 1;
                }
                Fr.ref(k, k) = T(d);
                out.kind[k] = kd;
                out.dd[k] = T(d);
                out.ee[k] = T(0);
                if (d > 0.0)
                    out.st[ST_NPOS]++;
                else if (d < 0.0)
                    out.st[ST_NNEG]++;
                sh[0] = d;
            }
            __syncthreads();
            const T d = T(sh[0]);
            for (int i = k + 1 + tid; i < f; i += NT) Fr.ref(i, k) = Fr.ref(i, k) / d;
            __syncthreads();
            const int R = f - k - 1, C = w - k - 1;
            for (int q = tid; q < R * C; q += NT) {
                const int j = k + 1 + q / R, i = k + 1 + q % R;
                Fr.ref(i, j) = Fr.ref(i, j) - Fr.ref(i, k) * Fr.ref(k, j);
            }
            __syncthreads();
            k += 1;
        } else {
            Fr.swap(k + 1, r);
            if (tid == 0) {
                const T a = Fr.ref(k, k), b = Fr.ref(k + 1, k), c2 = Fr.ref(k + 1, k + 1);
                const T up = b;
                Fr.ref(k, k + 1) = up;
                const T det = a * c2 - up * b;
                sh[0] = (double)(c2 / det);
                sh[1] = (double)(-up / det);
                sh[2] = (double)(-b / det);
                sh[3] = (double)(a / det);
                out.kind[k] = KIND_2X2_FIRST;
                out.kind[k + 1] = KIND_2X2_SECOND;
                out.dd[k] = a;
                out.dd[k + 1] = c2;
                out.ee[k] = b;
                out.ee[k + 1] = T(0);
                out.st[ST_N2X2]++;
                if (det < T(0)) {
                    out.st[ST_NPOS]++;
                    out.st[ST_NNEG]++;
                } else if (a > T(0)) {
                    out.st[ST_NPOS] += 2;
                } else {
                    out.st[ST_NNEG] += 2;
                }
                Fr.ref(k + 1, k) = T(0);  // the reference clears it; nobody reads it below
            }
            __syncthreads();
            const T e11 = T(sh[0]), e12 = T(sh[1]), e21 = T(sh[2]), e22 = T(sh[3]);
            for (int i = k + 2 + tid; i < f; i += NT) {
                const T x1 = Fr.ref(i, k), x2 = Fr.ref(i, k + 1);
                Fr.ref(i, k) = x1 * e11 + x2 * e21;
                Fr.ref(i, k + 1) = x1 * e12 + x2 * e22;
            }
            __syncthreads();
            const int R = f - k - 2, C = w - k - 2;
            for (int q = tid; q < R * C; q += NT) {
                const int j = k + 2 + q / R, i = k + 2 + q % R;
                Fr.ref(i, j) = Fr.ref(i, j) - (Fr.ref(i, k) * Fr.ref(k, j) + Fr.ref(i, k + 1) * Fr.ref(k + 1, j));
            }
            __syncthreads();
            k += 2;
        }
    }
}

// W[i, k] = (L21 D)[i, k] for row i of L (column-major, ld f) given the pivot kinds and D
// (ldlt.jl:206-231); k is a factor column of the front
template <typename T>
__device__ inline T w_entry(const T* L, int64_t f, int i, int k, const int8_t* kind, const T* dd, const T* ee) {
    const int8_t kd = kind[k];
    if (kd == KIND_2X2_FIRST) {
        const T x1 = L[(int64_t)k * f + i], x2 = L[(int64_t)(k + 1) * f + i];
        return x1 * dd[k] + x2 * ee[k];
    }
    if (kd == KIND_2X2_SECOND) {
        const T x1 = L[(int64_t)(k - 1) * f + i], x2 = L[(int64_t)k * f + i];
        return x1 * ee[k - 1] + x2 * dd[k];
    }
    return L[(int64_t)k * f + i] * dd[k];
}

template <typename T>
__device__ inline double eps_eff(double eps, int scaled, const double* aux) {
    if (!scaled) return eps;
    const double a = aux[0];
    return a > 0 ? eps * a : eps;
}

// ---------------------------------------------------------------------------
// small fronts: one workgroup, the dense front in LDS

constexpr int LDLT_SMALL_W = 128;  // largest front of the small class (f <= this)

template <typename T>
__global__ void __launch_bounds__(256) k_front_small_ldlt(DevSym S, const int32_t* __restrict__ fronts,
                                                         const double* __restrict__ nz, T* __restrict__ factor,
                                                         T* __restrict__ cbpool, T* __restrict__ dvec,
                                                         int32_t* __restrict__ piv, int8_t* __restrict__ pkind,
                                                         int64_t* __restrict__ stats, LdltPrm prm, int scaled,
                                                         const double* __restrict__ aux,
                                                         const int8_t* __restrict__ psign) {
    constexpr int NT = 256;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    T* F = reinterpret_cast<T*>(smem_raw);
    __shared__ RedBuf<NT> rb;
    __shared__ int lp[LDLT_SMALL_W];
    __shared__ int8_t kind[LDLT_SMALL_W];
    __shared__ T dd[LDLT_SMALL_W], ee[LDLT_SMALL_W];
    __shared__ int st[NF];
    __shared__ double sh[4];
    const int s = fronts[blockIdx.x];
    const int f = S.fnrows[s], w = S.fncols[s], m = f - w;
    const int c0 = S.super_ptr[s];
    const int tid = threadIdx.x;
    prm.eps = eps_eff<T>(prm.eps, scaled, aux);
    for (int k = tid; k < w; k += NT) {
        lp[k] = k;
        kind[k] = 0;
        dd[k] = ee[k] = T(0);
    }
    if (tid < NF) st[tid] = 0;
    assemble_dense<T>(S, s, nz, cbpool, F, f, 0);
    // the upper triangle of the fully summed block mirrors the lower one
    for (int q = tid; q < w * w; q += NT) {
        const int j = q / w, i = q - j * w;
        if (i > j) F[i * f + j] = F[j * f + i];
    }
    __syncthreads();
    Front<T, NT> Fr{F, f, w, lp, &rb};
    ldlt_front<T, NT>(Fr, prm, psign, S.perm + c0, PivOut<T>{kind, dd, ee, st}, sh);
    // W = L21 D, then the lower triangle of F22 <- F22 - W L21^T, k in order
    const int64_t co = S.cb_off[s];
    if (co >= 0) {
        T* C = cbpool + co;
        for (int q = tid; q < m * m; q += NT) {
            const int jj = q / m, ii = q - jj * m;
            if (ii < jj) continue;
            T acc = F[(w + jj) * f + w + ii];
            for (int k = 0; k < w; ++k) acc = acc - w_entry<T>(F, f, w + ii, k, kind, dd, ee) * F[k * f + w + jj];
            C[q] = acc;
        }
    }
    T* P = factor + S.panel_off[s];
    for (int q = tid; q < f * w; q += NT) {
        const int j = q / f, i = q - j * f;
        P[q] = i > j ? F[q] : (i == j ? T(1) : T(0));
    }
    for (int k = tid; k < w; k += NT) {
        const int g = c0 + k;
        piv[g] = c0 + lp[k];
        pkind[g] = kind[k];
        dvec[g] = dd[k];
        dvec[S.n + g] = ee[k];
    }
    if (tid < NF) stats[(int64_t)s * NF + tid] = st[tid];
}

// ---------------------------------------------------------------------------
// large fronts, one pivot per pair of launches over the whole GPU: k_ldlt_pivot (one
// workgroup per front) chooses the pivot of the front's next column, swaps, sets D and
// scales the pivot column(s); k_ldlt_update (64 x 64 tiles over every front of the level)
// applies that pivot's rank-1 or rank-2 update to the remaining fully summed columns (all
// rows). Each entry goes through the operations of ldlt_front above, in the same order. A
// 2x2 pivot takes two columns in one pair, so the number of pairs a front needs is only
// known on the device: the launch pairs run to the level's widest front and a front whose
// columns are done skips them. lstep[3 s ..]: the step's first column, its size (1, 2, or 0
// when the front is done) and the next column.

// launch pair t: the next pivot of every large front. task: (s)
template <typename T>
__global__ void __launch_bounds__(1024) k_ldlt_pivot(DevSym S, const Task* __restrict__ tasks, int t,
                                                    T* __restrict__ factor, T* __restrict__ dvec,
                                                    int32_t* __restrict__ piv, int8_t* __restrict__ pkind,
                                                    int64_t* __restrict__ stats, int32_t* __restrict__ lstep,
                                                    LdltPrm prm, int scaled, const double* __restrict__ aux,
                                                    const int8_t* __restrict__ psign) {
    constexpr int NT = 1024;
    constexpr int SCAP = 2048;  // candidates of the sorted best-1x1 scan
    __shared__ RedBuf<NT> rb;
    __shared__ double sh[4];
    __shared__ double skey[SCAP];
    __shared__ int sidx[SCAP];
    const int s = tasks[blockIdx.x].s;
    const int f = S.fnrows[s], w = S.fncols[s];
    const int c0 = S.super_ptr[s];
    const int tid = threadIdx.x;
    prm.eps = eps_eff<T>(prm.eps, scaled, aux);
    T* P = factor + S.panel_off[s];
    int* lp = piv + c0;
    int8_t* kind = pkind + c0;
    T* dd = dvec + c0;
    T* ee = dvec + S.n + c0;
    int64_t* st = stats + (int64_t)s * NF;
    int32_t* ls = lstep + 3 * s;
    int k;
    if (t == 0) {
        for (int q = tid; q < w; q += NT) {
            lp[q] = q;
            kind[q] = 0;
            dd[q] = ee[q] = T(0);
        }
        if (tid < NF) st[tid] = 0;
        // (the upper triangle of the fully summed square, the reference's full square, was
        // mirrored from the lower one by k_ldlt_mirror)
        k = 0;
    } else {
        k = ls[2];
    }
    __syncthreads();
    if (k >= w) {
        if (tid == 0) ls[1] = 0;
        return;
    }
    Front<T, NT> Fr{P, f, w, lp, &rb, skey, sidx, SCAP};
    // The usual step in one pass over column k: its entries k..f-1 in registers (the loads
    // issued together), one combined reduction giving the Bunch-Kaufman partner search (the
    // largest |a_ik| over rows k+1..w-1, first index on ties) and the threshold test's column
    // maximum (rows k+1..f-1, NaN-propagating). When column k is its own acceptable 1x1 pivot
    // (the first outcome of choose: no partner needed, the threshold test passes) the step
    // takes it and scales the column from the registers; otherwise choose decides from the
    // panel with the same predicates.
    constexpr int CR = 8;  // column entries per thread held in registers
    __shared__ double smx[NT / 64];
    T x[CR];
    bool fast = false;
    if (f - k <= CR * NT) {
        const T* col = P + (int64_t)k * f;
#pragma unroll
        for (int u = 0; u < CR; ++u) x[u] = col[min(k + tid + NT * u, f - 1)];
        const double akk = fabs((double)col[k]);
        __builtin_amdgcn_sched_barrier(0);
        double lam = 0.0, m = 0.0;
        int rr = -1;
#pragma unroll
        for (int u = 0; u < CR; ++u) {
            const int i = k + tid + NT * u;
            if (i > k && i < f) {
                const double a = fabs((double)x[u]);
                m = jmax(m, a);
                if (i < w && a > lam) {
                    lam = a;
                    rr = i;
                }
            }
        }
        wave_argmax(lam, rr);
        m = wave_jmax(m);
        const int lane = tid & 63, wv = tid >> 6;
        if (lane == 0) {
            rb.v[wv] = lam;
            rb.i[wv] = rr;
            smx[wv] = m;
        }
        __syncthreads();
        lam = rb.v[0];
        rr = rb.i[0];
        m = smx[0];
        for (int q = 1; q < NT / 64; ++q) {
            if (vi_better(rb.v[q], rb.i[q], lam, rr)) {
                lam = rb.v[q];
                rr = rb.i[q];
            }
            m = jmax(m, smx[q]);
        }
        __syncthreads();
        if (rr < 0) lam = 0.0;
        if (prm.pivot == PV_NONE) {
            fast = true;
        } else {
            const double alpha = (1.0 + sqrt(17.0)) / 8.0;  // Bunch-Kaufman constant (ldlt.jl:22)
            const bool self = prm.pivot == PV_DIAG || rr < 0 || akk >= alpha * lam;
            fast = self && akk >= prm.eps && akk >= prm.u * m;
        }
    }
    int c = k, r = -1;
    if (!fast) Fr.choose(k, prm, c, r);
    const int8_t* sreq_row = psign;
    const int32_t* perm_c0 = S.perm + c0;
    if (r < 0) {
        Fr.swap(k, c);
        if (tid == 0) {
            // (thread 0 holds a_kk in x[0] on the one-pass step; the sign counts are added by
            // atomics whose result is not waited for)
            double d = fast ? (double)x[0] : Fr.at(k, k);
            int8_t kd = KIND_1X1;
            if (!(fabs(d) >= prm.eps) || d == 0.0) {
                if (d == 0.0) st[ST_NZERO]++;
                const int req = sreq_row ? (int)sreq_row[perm_c0[lp[k]]] : 0;
                const double sg = req != 0 ? (double)req : (d < 0.0 ? -1.0 : 1.0);
                d = sg * prm.eps;
                kd = KIND_PERTURBED;
                st[ST_NPERT]++;
                if (d == 0.0 && st[ST_INFO] == 0) st[ST_INFO] = lp[k] + 1;
            }
            Fr.ref(k, k) = T(d);
            kind[k] = kd;
            dd[k] = T(d);
            ee[k] = T(0);
            if (d > 0.0)
                atomicAdd(reinterpret_cast<unsigned long long*>(st + ST_NPOS), 1ull);
            else if (d < 0.0)
                atomicAdd(reinterpret_cast<unsigned long long*>(st + ST_NNEG), 1ull);
            sh[0] = d;
            ls[0] = k;
            ls[1] = 1;
            ls[2] = k + 1;
        }
        __syncthreads();
        const T d = T(sh[0]);
        if (fast) {
            T* col = P + (int64_t)k * f;
#pragma unroll
            for (int u = 0; u < CR; ++u) {
                const int i = k + tid + NT * u;
                if (i > k && i < f) col[i] = x[u] / d;
            }
        } else {
            for (int i = k + 1 + tid; i < f; i += NT) Fr.ref(i, k) = Fr.ref(i, k) / d;
        }
    } else {
        Fr.swap(k + 1, r);
        if (tid == 0) {
            const T a = Fr.ref(k, k), b = Fr.ref(k + 1, k), c2 = Fr.ref(k + 1, k + 1);
            const T up = b;
            Fr.ref(k, k + 1) = up;
            const T det = a * c2 - up * b;
            sh[0] = (double)(c2 / det);
            sh[1] = (double)(-up / det);
            sh[2] = (double)(-b / det);
            sh[3] = (double)(a / det);
            kind[k] = KIND_2X2_FIRST;
            kind[k + 1] = KIND_2X2_SECOND;
            dd[k] = a;
            dd[k + 1] = c2;
            ee[k] = b;
            ee[k + 1] = T(0);
            st[ST_N2X2]++;
            if (det < T(0)) {
                st[ST_NPOS]++;
                st[ST_NNEG]++;
            } else if (a > T(0)) {
                st[ST_NPOS] += 2;
            } else {
                st[ST_NNEG] += 2;
            }
            Fr.ref(k + 1, k) = T(0);
            ls[0] = k;
            ls[1] = 2;
            ls[2] = k + 2;
        }
        __syncthreads();
        const T e11 = T(sh[0]), e12 = T(sh[1]), e21 = T(sh[2]), e22 = T(sh[3]);
        for (int i = k + 2 + tid; i < f; i += NT) {
            const T x1 = Fr.ref(i, k), x2 = Fr.ref(i, k + 1);
            Fr.ref(i, k) = x1 * e11 + x2 * e21;
            Fr.ref(i, k + 1) = x1 * e12 + x2 * e22;
        }
    }
}

// before the pivot launches: the upper triangle of each large front's fully summed square
// mirrors the lower one (the reference's full square). task: (s, I0, J0), the 64 x 64 tile of
// rows I0.. and columns J0.. with I0 >= J0, written transposed through LDS (both sides
// coalesced)
template <typename T>
__global__ void __launch_bounds__(256) k_ldlt_mirror(DevSym S, const Task* __restrict__ tasks, T* __restrict__ factor) {
    __shared__ T tl[64][65];
    const Task t = tasks[blockIdx.x];
    const int s = t.s, f = S.fnrows[s], w = S.fncols[s];
    const int I0 = t.a, J0 = t.b, ni = min(64, w - I0), nj = min(64, w - J0);
    T* P = factor + S.panel_off[s];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    {
        T v[16];
#pragma unroll
        for (int q = 0; q < 16; ++q)
            v[q] = P[(int64_t)(J0 + min(wv + 4 * q, nj - 1)) * f + I0 + min(lane, ni - 1)];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < 16; ++q) tl[wv + 4 * q][lane] = v[q];  // tl[j][i] = A(I0 + i, J0 + j)
    }
    __syncthreads();
    // A(J0 + j, I0 + i) = A(I0 + i, J0 + j) for I0 + i > J0 + j: lanes along j
#pragma unroll
    for (int q = 0; q < 16; ++q) {
        const int i = wv + 4 * q, j = lane;
        if (i < ni && j < nj && I0 + i > J0 + j) P[(int64_t)(I0 + i) * f + J0 + j] = tl[j][i];
    }
}

// launch pair t: the update of each front's pivot of that pair on the fully summed columns
// after it (every row below). task: (s, I0, J0), a 64 x 64 tile, lanes along the rows
template <typename T>
__global__ void __launch_bounds__(256) k_ldlt_update(DevSym S, const Task* __restrict__ tasks, T* __restrict__ factor,
                                                     const int32_t* __restrict__ lstep) {
    const Task t = tasks[blockIdx.x];
    const int s = t.s, f = S.fnrows[s], w = S.fncols[s];
    const int32_t* ls = lstep + 3 * s;
    const int sz = ls[1];
    if (sz == 0) return;
    const int k = ls[0], k2 = k + sz;
    const int i = t.a + (threadIdx.x & 63);
    if (i < k2 || i >= f) return;
    T* P = factor + S.panel_off[s];
    const T* ck = P + (int64_t)k * f;
    const int j1 = min(t.b + 64, w);
    if (sz == 1) {
        // the thread's sixteen columns: every load in flight together (clamped to the tile's
        // last column), then the updates and the stores; row k is not written here
        const int jb = max(t.b, k2) + (threadIdx.x >> 6);
        if (jb >= j1) return;
        const T lk = ck[i];
        T a[16], u[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const int64_t o = (int64_t)min(jb + 4 * q, j1 - 1) * f;
            a[q] = P[o + i];
            u[q] = P[o + k];
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < 16; ++q)
            if (jb + 4 * q < j1) P[(int64_t)(jb + 4 * q) * f + i] = a[q] - lk * u[q];
    } else {
        const T l1 = ck[i], l2 = ck[f + i];
        for (int j = max(t.b, k2) + (threadIdx.x >> 6); j < j1; j += 4) {
            T& a = P[(int64_t)j * f + i];
            a = a - (l1 * P[(int64_t)j * f + k] + l2 * P[(int64_t)j * f + k + 1]);
        }
    }
}

// ---------------------------------------------------------------------------
// large fronts in panels: k_ldlt_panel (one workgroup per front) takes the pivots of a panel of
// NBP columns with the columns held in registers: thread t holds the rows k0 + t + NT u of every
// panel column (R rows, R NBP entries). The usual pivot (column k its own acceptable 1x1 pivot)
// is one pass: the column's two maxima by lane reductions, one barrier (LDS only: the L column's
// global stores stay in flight), the scaling and the rank-1 update of the panel's later columns,
// which moves each column one register to the left. Everything after the panel keeps its values
// of the panel's start; k_ldlt_trail then applies the panel's pivots to it over the GPU.
//
// Any other pivot (a 2x2, an interchange, a perturbation) is decided from the panel memory: the
// columns the choice reads are formed when it reads them, by applying the panel's pivots to the
// stored values in the reference's order: x - L(i, p) U(p, j) for a 1x1 pivot p, x - (L(i, p) U(p, j) +
// L(i, p + 1) U(p + 1, j)) for a 2x2 one. U(p, j), the row of pivot p in column j at the time of
// pivot p (the upper mirror entry the reference's update reads), is formed for a run of usual
// pivots at once, before such a pivot and at the panel's end. Every entry thus goes through the
// operations of ldlt_front in the same order: the factor is bitwise that of one pivot at a time.
// The symmetric interchanges act on the stored values, as in the reference; a row interchange of
// two positions at or after the current pivot commutes with the pending updates, since it
// exchanges the L rows of the panel's pivots too. After such a pivot the rest of the panel is
// loaded again and brought up to date.

constexpr int LP_NB = 16;           // most columns of a panel (a 2x2 pivot at its end takes one more)
constexpr int LP_MAXP = LP_NB + 1;  // pivot rows of one panel

// scratch of one front during a panel (element offsets from its base): the pivot rows U (LP_MAXP x
// w, U[q w + j] = U(k0 + q, j)), the current diagonal DG (w) and the saved panel columns V (cols x f)
inline int64_t lp_scratch(int f, int w, int cols) { return (int64_t)(LP_MAXP + 1) * w + (int64_t)cols * f; }

// a front during a panel, as its NT threads see it
template <typename T, int NT, int R, int MAXP>
struct PanelFront {
    Global<T>* P;
    int f, w, k0;
    Global<int>* lp;
    RedBuf<NT>* rb;
    Global<T>*U, *DG;
    Global<T>* V;  // the panel's columns kv, kv + 1, ... (MAXP - 1 of them, ld f) as they were before the pivot kv
    // the panel's pivot steps, bit q for column k0 + q: the 1x1 pivots, the first columns of 2x2 ones
    uint32_t one, two;
    // LDS
    T* Uc;          // U(., j) of the column being formed
    T* Lr;          // L(r, .) of the pivot row whose U row is being formed
    T (*Ls)[MAXP];  // Ls[r][q] = L(k0 + r, k0 + q), q < r, of the panel's pivots
    double* pk;     // picked entries (pick)
    double (*mx3)[NT / 64];  // the waves' maxima, three at a time

    // x minus the panel's first np pivots in order, l(q) = L(row, k0 + q) and u(q) = U(k0 + q,
    // column) (the operations and their order of ldlt_front's updates); eight pivots' entries are
    // loaded together (the ninth: the second column of a 2x2)
    template <class LF, class UF>
    __device__ __attribute__((always_inline)) T apply(T x, int np, LF l, UF u) const {
#pragma unroll 1
        for (int q0 = 0; q0 < np; q0 += 8) {
            T lv[9], uv[9];
#pragma unroll
            for (int q = 0; q < 9; ++q) {
                lv[q] = l(min(q0 + q, np - 1));
                uv[q] = u(min(q0 + q, np - 1));
            }
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                if (one >> (q0 + q) & 1)
                    x = x - lv[q] * uv[q];
                else if (two >> (q0 + q) & 1)
                    x = x - (lv[q] * uv[q] + lv[q + 1] * uv[q + 1]);
            }
        }
        return x;
    }
    __device__ __attribute__((always_inline)) PanelRows<NT, (int)sizeof(T)> rows() const { return {k0, f}; }
    // the thread and the slot of row i
    __device__ __attribute__((always_inline)) void owner(int i, int& t, int& u) const {
        const int o = uni(i - k0);
        u = o / NT;
        t = o - u * NT;
    }
    // the thread's rows of a column
    __device__ __attribute__((always_inline)) void load_rows(const Global<T>* col, T (&y)[R]) const {
        const auto rw = rows();
#pragma unroll
        for (int u = 0; u < R; ++u) y[u] = load_at(col, rw.clamped(u));
    }
    __device__ __attribute__((always_inline)) void store_rows(Global<T>* col, const T (&y)[R]) const {
        const auto rw = rows();
        const int nf = rw.count(f);
#pragma unroll
        for (int u = 0; u < R; ++u)
            if (u < nf) store_at(col, rw.off(u), y[u]);
    }
    // current values of column j at the thread's rows (all threads; ends with a barrier): from V for
    // a column of the panel, else the L entries of G pivots in flight together
    __device__ __attribute__((always_inline)) void form_col(int j, int np, T (&y)[R]) const {
        if (j < k0 + MAXP - 1) {
            load_rows(V + (int64_t)(j - k0 - np) * f, y);
            __syncthreads();
            return;
        }
        constexpr int G = R <= 3 ? 8 : R <= 6 ? 4 : 2;
        for (int q = threadIdx.x; q < np; q += NT) Uc[q] = U[(int64_t)q * w + j];
        __syncthreads();
        load_rows(P + (int64_t)j * f, y);
#pragma unroll 1
        for (int q0 = 0; q0 < np; q0 += G) {
            const auto rw = rows();
            T l[G][R];
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const Global<T>* cq = P + (int64_t)(k0 + min(q0 + g, np - 1)) * f;
#pragma unroll
                for (int u = 0; u < R; ++u) l[g][u] = load_at(cq, rw.clamped(u));
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int g = 0; g < G; ++g) {
                if (one >> (q0 + g) & 1) {
                    const T v = Uc[q0 + g];
#pragma unroll
                    for (int u = 0; u < R; ++u) y[u] = y[u] - l[g][u] * v;
                } else if (two >> (q0 + g) & 1) {
                    const T v = Uc[q0 + g], v2 = Uc[q0 + g + 1];
                    const Global<T>* c2 = P + (int64_t)(k0 + q0 + g + 1) * f;
#pragma unroll
                    for (int u = 0; u < R; ++u) y[u] = y[u] - (l[g][u] * v + load_at(c2, rw.clamped(u)) * v2);
                }
            }
        }
        __syncthreads();
    }
    // entry of row i of a column in registers, into pk[slot] (a barrier later)
    __device__ __attribute__((always_inline)) void pick(const T (&y)[R], int i, int slot) const {
        int t, us;
        owner(i, t, us);
        // (each entry hidden from the optimizer: as plain selects they become one load by a variable index,
        // and the column a scratch array)
        T v = y[0];
#pragma unroll
        for (int u = 1; u < R; ++u) {
            T z = y[u];
            asm("" : "+v"(z));
            v = u == us ? z : v;
        }
        if ((int)threadIdx.x == t) pk[slot] = (double)v;
    }
    // rows a and b of a column in registers exchanged (pk[sa], pk[sb]: its entries there)
    __device__ __attribute__((always_inline)) void exchange(T (&y)[R], int a, int b, int sa, int sb) const {
        const T va = T(pk[sa]), vb = T(pk[sb]);
        int ta, ua, tb, ub;
        owner(a, ta, ua);
        owner(b, tb, ub);
        const bool ma = (int)threadIdx.x == ta, mb = (int)threadIdx.x == tb;
#pragma unroll
        for (int u = 0; u < R; ++u) {
            y[u] = ma && u == ua ? vb : y[u];
            y[u] = mb && u == ub ? va : y[u];
        }
    }
    // largest |y_i| over the thread's rows k..end-1 but s1 and s2, NaN-propagating (ldlt.jl:240-260)
    __device__ __attribute__((always_inline)) double rows_max(const T (&y)[R], int k, int end, int s1, int s2) const {
        // (rows above k: only among the first slot's, the panel is narrower than the block)
        double m = 0.0;
        const int n = rows().count(end);
        int t1, u1, t2, u2;
        owner(s1, t1, u1);
        owner(s2, t2, u2);
        const bool up = (int)threadIdx.x >= k - k0, m1 = (int)threadIdx.x == t1, m2 = (int)threadIdx.x == t2;
#pragma unroll
        for (int u = 0; u < R; ++u) {
            bool on = u < n;
            if (u == 0) on = on && up;
            if (u == u1) on = on && !m1;
            if (u == u2) on = on && !m2;
            m = on ? jmax(m, fabs((double)y[u])) : m;
        }
        return m;
    }
    // the same over the whole front
    __device__ __attribute__((always_inline)) double colmax(const T (&y)[R], int k, int end, int s1, int s2) const {
        return block_jmax<NT>(rows_max(y, k, end, s1, s2), *rb);
    }
    // current diagonal entries of the columns k..w-1 into DG (all threads; ends with a barrier)
    __device__ __attribute__((always_inline)) void form_diag(int k) const {
        for (int j = k + threadIdx.x; j < w; j += NT)
            DG[j] = apply(P[(int64_t)j * f + j], k - k0, [&](int q) { return P[(int64_t)(k0 + q) * f + j]; },
                          [&](int q) { return U[(int64_t)q * w + j]; });
        __syncthreads();
    }
    // U row of the pivot row r (a position at or after the current pivot, before the current
    // pivot's own step is recorded) for the columns j0..w-1 (all threads; ends with a barrier)
    __device__ __attribute__((always_inline)) void form_urow(int r, int j0) const {
        const int np = r - k0;
        for (int q = threadIdx.x; q < np; q += NT) Lr[q] = P[(int64_t)(k0 + q) * f + r];
        __syncthreads();
        Global<T>* ur = U + (int64_t)np * w;
        for (int j = j0 + threadIdx.x; j < w; j += NT)
            ur[j] = apply(P[(int64_t)j * f + r], np, [&](int q) { return Lr[q]; },
                          [&](int q) { return U[(int64_t)q * w + j]; });
        __syncthreads();
    }
    // U rows n0..n1-1 (all of them 1x1 pivots) for the columns k0 + n1..w-1, the rows before n0 being
    // there: a thread per column, eight rows at a time (all threads; ends with a barrier)
    __device__ __attribute__((always_inline)) void form_urows(int n0, int n1) const {
        for (int j = k0 + n1 + threadIdx.x; j < w; j += NT) {
            const Global<T>* cj = P + (int64_t)j * f + k0;
#pragma unroll 1
            for (int b0 = n0; b0 < n1; b0 += 8) {
                T a[8];
#pragma unroll
                for (int r = 0; r < 8; ++r) a[r] = cj[min(b0 + r, n1 - 1)];
#pragma unroll 1
                for (int q0 = 0; q0 < b0; q0 += 8) {
                    T uv[9];
#pragma unroll
                    for (int q = 0; q < 9; ++q) uv[q] = U[(int64_t)min(q0 + q, b0 - 1) * w + j];
#pragma unroll
                    for (int q = 0; q < 8; ++q) {
                        if (q0 + q >= b0) break;
                        if (one >> (q0 + q) & 1) {
#pragma unroll
                            for (int r = 0; r < 8; ++r) a[r] = a[r] - Ls[min(b0 + r, n1 - 1)][q0 + q] * uv[q];
                        } else if (two >> (q0 + q) & 1) {
#pragma unroll
                            for (int r = 0; r < 8; ++r)
                                a[r] = a[r] - (Ls[min(b0 + r, n1 - 1)][q0 + q] * uv[q] +
                                               Ls[min(b0 + r, n1 - 1)][q0 + q + 1] * uv[q + 1]);
                        }
                    }
                }
#pragma unroll
                for (int r = 0; r < 8; ++r) {
                    if (b0 + r >= n1) break;
                    U[(int64_t)(b0 + r) * w + j] = a[r];
#pragma unroll
                    for (int r2 = r + 1; r2 < 8; ++r2) a[r2] = a[r2] - Ls[min(b0 + r2, n1 - 1)][b0 + r] * a[r];
                }
            }
        }
        __syncthreads();
    }
    // the update of the pivot at q = k - k0 (1x1: its L column la; TWO: a 2x2's la and lb) on V's later
    // columns, G columns in flight together
    template <bool TWO>
    __device__ __attribute__((always_inline)) void update_v(int q, const T (&la)[R], const T (&lb)[R]) const {
        constexpr int G = R <= 3 ? 8 : R <= 6 ? 4 : R <= 12 ? 2 : 1;
        const int n = min(MAXP - 1, w - k0) - q;  // V's columns inside the panel
        const Global<T>* u0 = U + (int64_t)q * w + k0 + q;
#pragma unroll 1
        for (int c0 = TWO ? 2 : 1; c0 < n; c0 += G) {
            const auto rw = rows();
            const int nf = rw.count(f);
            T v[G][R], ua[G], ub[G];
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const int c = min(c0 + g, n - 1);
                ua[g] = u0[c];
                ub[g] = TWO ? u0[w + c] : T(0);
#pragma unroll
                for (int u = 0; u < R; ++u) v[g][u] = load_at(V + (int64_t)c * f, rw.clamped(u));
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int g = 0; g < G; ++g) {
                if (c0 + g < n) {
#pragma unroll
                    for (int u = 0; u < R; ++u) {
                        const T x = TWO ? v[g][u] - (la[u] * ua[g] + lb[u] * ub[g]) : v[g][u] - la[u] * ua[g];
                        if (u < nf) store_at(V + (int64_t)(c0 + g) * f, rw.off(u), x);
                    }
                }
            }
        }
    }
    // the current entries (rows i[t], columns j[c]) of NC columns from their stored ones in x, by one wave; the
    // columns share the loads of L, four pivots' at a time. ul[c]: U(., j[c]), a pivot a lane
    template <int NC, int NR>
    __device__ __attribute__((always_inline)) void wave_apply(int np, const int (&i)[NR], const T (&ul)[NC],
                                                              T (&x)[NC][NR]) const {
#pragma unroll 1
        for (int q0 = 0; q0 < np; q0 += 4) {
            T l[5][NR];  // (the fifth: the second column of a 2x2)
#pragma unroll
            for (int g = 0; g < 5; ++g)
#pragma unroll
                for (int t = 0; t < NR; ++t) l[g][t] = P[(int64_t)(k0 + min(q0 + g, np - 1)) * f + i[t]];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int q1 = min(q0 + g, np - 1), q2 = min(q0 + g + 1, np - 1);
                if (one >> (q0 + g) & 1) {
#pragma unroll
                    for (int c = 0; c < NC; ++c)
#pragma unroll
                        for (int t = 0; t < NR; ++t) x[c][t] = x[c][t] - l[g][t] * lane_bcast(ul[c], q1);
                } else if (two >> (q0 + g) & 1) {
#pragma unroll
                    for (int c = 0; c < NC; ++c)
#pragma unroll
                        for (int t = 0; t < NR; ++t)
                            x[c][t] = x[c][t] - (l[g][t] * lane_bcast(ul[c], q1) + l[g + 1][t] * lane_bcast(ul[c], q2));
                }
            }
        }
    }
    // the best acceptable 1x1 pivot among the columns k..w-1 but `first`, their current diagonal in DG, each
    // tested by one wave unless it cannot beat the wave's best: eight columns together on 64 rows, where
    // most of those that fail do, the others on all rows. A column passes where a = |a_jj| >= u |a_ij| for
    // every other row, which is the test of the largest (a product with u is monotone). All threads get
    // the answer (-1 if none)
    __device__ __attribute__((always_inline)) int search_1x1(int k, int first, const LdltPrm& p) const {
        constexpr int NC = 8;
        const int wv = uni(threadIdx.x >> 6), lane = threadIdx.x & 63, np = k - k0;
        double bv = -1.0;
        int bj = -1;
#pragma unroll 1
        for (int j0 = k + NC * wv; j0 < w; j0 += NC * (NT / 64)) {
            double a[NC];
            T x[NC][1], ul[NC];
            const int i[1] = {min(k + lane, f - 1)};
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                const int j = min(j0 + c, w - 1);
                a[c] = fabs((double)DG[j]);
                x[c][0] = P[(int64_t)j * f + i[0]];
                ul[c] = np > 0 ? U[(int64_t)min(lane, np - 1) * w + j] : T(0);
            }
            __builtin_amdgcn_sched_barrier(0);
            wave_apply(np, i, ul, x);
            uint32_t left = 0;
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                const int j = j0 + c;
                const bool live = j < w && j != first && a[c] >= p.eps && (bj < 0 || a[c] > bv);
                const bool fails = i[0] != j && !(a[c] >= p.u * fabs((double)x[c][0]));
                if (uni(live) && !__any(fails)) left |= 1u << c;
            }
#pragma unroll 1
            for (; left; left &= left - 1) {
                const int j = j0 + __builtin_ctz(left);
                const double aj = fabs((double)DG[j]);
                if (uni(bj >= 0 && !(aj > bv))) continue;
                const T ur[1] = {np > 0 ? U[(int64_t)min(lane, np - 1) * w + j] : T(0)};
                bool ok = true;
#pragma unroll 1
                for (int i0 = k + 64; ok && i0 < f; i0 += 256) {
                    int ir[4];
                    T xr[1][4];
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        ir[t] = min(i0 + 64 * t + lane, f - 1);
                        xr[0][t] = P[(int64_t)j * f + ir[t]];
                    }
                    wave_apply(np, ir, ur, xr);
                    bool fails = false;
#pragma unroll
                    for (int t = 0; t < 4; ++t) fails |= ir[t] != j && !(aj >= p.u * fabs((double)xr[0][t]));
                    ok = !__any(fails);
                }
                if (ok) {
                    bv = aj;
                    bj = j;
                }
            }
        }
        if (lane == 0) {
            rb->v[wv] = bv;
            rb->i[wv] = bj;
        }
        __syncthreads();
        bv = rb->v[0];
        bj = rb->i[0];
        for (int q = 1; q < NT / 64; ++q)
            if (vi_better(rb->v[q], rb->i[q], bv, bj)) {
                bv = rb->v[q];
                bj = rb->i[q];
            }
        __syncthreads();
        return uni(bj);
    }
    // best_1x1 (ldlt.jl:264-276) on the current diagonal (formed here): the acceptable 1x1 pivot of
    // k..w-1 with the largest |a_jj|, first on ties, -1 if none; on return y holds the answer's current
    // column. The largest candidate (|a_jj| >= eps) is tested first, by the whole block: it is usually the
    // answer (KKT, n = 12,000: in 367 of 619 searches). Where it is not, the others are tested by a wave
    // each. (One candidate after another by the whole block: a front of 600 columns under a threshold that
    // nearly all of them fail took 89 ms instead of 16.)
    __device__ __attribute__((always_inline)) int best_1x1(int k, const LdltPrm& p, T (&y)[R]) const {
        form_diag(k);
        double v = -1.0;
        int bi = -1;
        for (int j = k + threadIdx.x; j < w; j += NT) {
            const double a = fabs((double)DG[j]);
            if (a >= p.eps && vi_better(a, j, v, bi)) {
                v = a;
                bi = j;
            }
        }
        block_argmax<NT>(v, bi, *rb);
        bi = uni(bi);
        bool tested = false;
#pragma unroll 1
        while (bi >= 0) {
            form_col(bi, k - k0, y);
            if (tested || uni(v >= p.u * colmax(y, k, f, bi, bi))) return bi;
            tested = true;
            bi = search_1x1(k, bi, p);
        }
        return -1;
    }
    // pivot choice at column k (ldlt.jl:280-325), as Front::choose on the current columns, column k
    // in xa: c = pivot column, r = 2x2 partner or -1; on return the column c is in xa (1x1), or the
    // columns k and r are in xa and xb (2x2)
    __device__ __attribute__((always_inline)) void choose(int k, const LdltPrm& p, int& c, int& r, T (&xa)[R],
                                                          T (&xb)[R]) const {
        const int np = k - k0;
        r = -1;
        c = k;
        if (p.pivot == PV_NONE) return;
        pick(xa, k, 0);
        double mk = rows_max(xa, k, f, k, k), akk;
        bool ok, two2 = false;
        double det = 0.0, mx = 0.0;
        int rr = -1;
        if (p.pivot == PV_DIAG) {
            mk = block_jmax<NT>(mk, *rb);
            akk = fabs(pk[0]);
            ok = akk >= p.eps && akk >= p.u * mk;
        } else {
            const double alpha = (1.0 + sqrt(17.0)) / 8.0;  // Bunch-Kaufman constant (ldlt.jl:22)
            double lambda = 0.0;
            {
                const int n = rows().count(w);
                const bool up = (int)threadIdx.x > k - k0;
#pragma unroll
                for (int u = 0; u < R; ++u) {
                    const double a = fabs((double)xa[u]);
                    if (u < n && (u > 0 || up) && a > lambda) {
                        lambda = a;
                        rr = u;
                    }
                }
                if (rr >= 0) rr = k0 + (int)threadIdx.x + NT * rr;
            }
            mk = wave_jmax(mk);
            if ((threadIdx.x & 63) == 0) mx3[0][threadIdx.x >> 6] = mk;
            block_argmax<NT>(lambda, rr, *rb);
            mk = mx3[0][0];
            for (int q = 1; q < NT / 64; ++q) mk = jmax(mk, mx3[0][q]);
            akk = fabs(pk[0]);
            rr = uni(rr);
            if (rr < 0) lambda = 0.0;
            if (rr < 0 || uni(akk >= alpha * lambda)) {
                ok = akk >= p.eps && akk >= p.u * mk;
            } else {
                form_col(rr, np, xb);
                pick(xa, rr, 1);
                pick(xb, k, 2);
                pick(xb, rr, 3);
                // the maxima of column rr's fully summed rows and of the two columns below a 2x2 pivot together
                double m[3] = {rows_max(xb, k, w, rr, rr), rows_max(xa, k, f, k, rr), rows_max(xb, k, f, rr, k)};
#pragma unroll
                for (int q = 0; q < 3; ++q) {
                    m[q] = wave_jmax(m[q]);
                    if ((threadIdx.x & 63) == 0) mx3[q][threadIdx.x >> 6] = m[q];
                }
                __syncthreads();
#pragma unroll
                for (int q = 0; q < 3; ++q) {
                    m[q] = mx3[q][0];
                    for (int v = 1; v < NT / 64; ++v) m[q] = jmax(m[q], mx3[q][v]);
                }
                const double sigma = m[0], arr = pk[3], ark = pk[1], akr = pk[2];
                if (uni(akk * sigma >= alpha * lambda * lambda)) {
                    ok = akk >= p.eps && akk >= p.u * mk;
                } else if (uni(fabs(arr) >= alpha * sigma)) {
                    c = rr;
                    ok = fabs(arr) >= p.eps && fabs(arr) >= p.u * jmax(m[2], fabs(akr));
                } else {
                    two2 = true;
                    det = pk[0] * arr - akr * ark;
                    mx = jmax(jmax(akk, fabs(ark)), fabs(arr));
                    ok = det != 0.0 && isfinite(det) && mx >= p.eps;
                    if (uni(ok)) {
                        const double e11 = fabs(arr / det), e12 = fabs(akr / det), e21 = fabs(ark / det),
                                     e22 = fabs(pk[0] / det);
                        ok = p.u * (e11 * m[1] + e21 * m[2]) <= 1.0 && p.u * (e12 * m[1] + e22 * m[2]) <= 1.0;
                    }
                }
            }
        }
        if (!uni(ok)) {
            T y[R];
            int best = best_1x1(k, p, y);
            if (best < 0 && p.pivot == PV_DIAG) {
                // the largest diagonal entry, first on ties; a NaN |a_kk| keeps k (DG was formed by
                // best_1x1)
                double v = akk;
                int bi = k;
                for (int j = k + 1 + threadIdx.x; j < w; j += NT) {
                    const double a = fabs((double)DG[j]);
                    if (a > v) {
                        v = a;
                        bi = j;
                    }
                }
                block_argmax<NT>(v, bi, *rb);
                best = uni(fabs((double)DG[bi]) >= p.eps ? bi : k);
                if (best == k) return;
                form_col(best, np, y);
            }
            if (best >= 0) {
                c = best;
#pragma unroll
                for (int u = 0; u < R; ++u) xa[u] = y[u];
                return;
            }
            two2 = uni(two2 && det != 0.0 && isfinite(det) && mx >= p.eps);  // (a singular 2x2: k as a 1x1)
        }
        if (two2) {
            r = rr;
        } else if (c != k) {
#pragma unroll
            for (int u = 0; u < R; ++u) xa[u] = xb[u];
        }
    }
    // symmetric interchange of the positions a (the pivot position, whose column is written next)
    // and b (ldlt.jl:328-340): the stored column of a moves to b, the rows a and b of every other
    // stored column, of V and of the columns in registers are exchanged, and the pivot rows' entries
    // (xa, with TWO also xb; np pivots taken, the current pivot is k0 + np; ends with a barrier)
    template <bool TWO>
    __device__ __attribute__((always_inline)) void swap(int a, int b, int np, T (&xa)[R], T (&xb)[R]) const {
        if (a == b) return;
        pick(xa, a, 0);
        pick(xa, b, 1);
        const int kv = k0 + np;
        T col[R];
        load_rows(P + (int64_t)a * f, col);
        for (int q = threadIdx.x; q < np; q += NT) {
            const T t = U[(int64_t)q * w + a];
            U[(int64_t)q * w + a] = U[(int64_t)q * w + b];
            U[(int64_t)q * w + b] = t;
        }
        store_rows(P + (int64_t)b * f, col);
        if (b < k0 + MAXP - 1) {
            load_rows(V + (int64_t)(a - kv) * f, col);
            store_rows(V + (int64_t)(b - kv) * f, col);
        }
        __syncthreads();
        for (int c = threadIdx.x; c < MAXP - 1; c += NT) {
            const T t = V[(int64_t)c * f + a];
            V[(int64_t)c * f + a] = V[(int64_t)c * f + b];
            V[(int64_t)c * f + b] = t;
        }
        exchange(xa, a, b, 0, 1);
        if (TWO) {
            pick(xb, a, 2);
            pick(xb, b, 3);
            __syncthreads();
            exchange(xb, a, b, 2, 3);
        }
        for (int j = threadIdx.x; j < w; j += NT) {
            const T t = P[(int64_t)j * f + a];
            P[(int64_t)j * f + a] = P[(int64_t)j * f + b];
            P[(int64_t)j * f + b] = t;
        }
        if (threadIdx.x == 0) {
            const int t = lp[a];
            lp[a] = lp[b];
            lp[b] = t;
        }
        __syncthreads();
    }
};

// the state of a panel's usual pivots
template <typename T, int R, int NBP>
struct PanelRegs {
    T x[R][NBP];  // x[u][c] = entry (k0 + tid + NT u, k + c)
    int nr;       // row slots in use
    int buf;
    int npos, nneg;
};

// usual pivots k, k + 1, ... of the panel while the panel's remaining columns number more than W - 8
// (of W registers per row); false: column k is not its own acceptable 1x1 pivot
template <typename T, int NT, int R, int NBP, int W, class Z>
__device__ __attribute__((always_inline)) inline bool panel_pivots(PanelRegs<T, R, NBP>& X, const Z& F, int& k, int kend,
                                                                   const LdltPrm& p, double (*red)[NT / 64][2],
                                                                   T (*urow)[NBP], int* ctype, Global<int8_t>* kind,
                                                                   Global<T>* dd) {
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, f = F.f, w = F.w, k0 = F.k0;
    const double alpha = (1.0 + sqrt(17.0)) / 8.0;  // Bunch-Kaufman constant (ldlt.jl:22)
    const int kstop = min(kend, k0 + NBP - (W > 8 ? W - 8 : 0));
    while (k < kstop) {
        // the largest |a_ik| below the pivot: fully summed rows, then the others
        double lam = 0.0, mx = 0.0;
        bool nan = false;
        const auto rw = F.rows();
        const int nf = rw.count(f), nw = rw.count(w);
        const bool up = tid > k - k0;  // (the pivot's row is among the first slot's)
#pragma unroll
        for (int u = 0; u < R; ++u) {
            if (u < X.nr) {  // (only the last slot can hold rows past the front's end)
                double a = (double)X.x[u][0];
                if (u == 0) a = up ? a : 0.0;
                if (u + 1 == X.nr) a = u < nf ? a : 0.0;
                nan |= a != a;
                mx = max_abs(mx, a);
                if (NT * u < w - k0) lam = max_abs(lam, u < nw ? a : 0.0);
            }
        }
        lam = wave_max_last(lam);
        mx = wave_max_last(mx);
        if (__any(nan)) mx = __builtin_nan("");
        X.buf ^= 1;
        if (lane == 63) {
            red[X.buf][wv][0] = lam;
            red[X.buf][wv][1] = mx;
        }
        if (tid == k - k0) {
#pragma unroll
            for (int c = 0; c < W; ++c) urow[X.buf][c] = X.x[0][c];
        }
        __syncthreads();  // (waits for LDS only: the L columns' stores stay in flight)
        nan = false;
        lam = 0.0;
        mx = 0.0;
#pragma unroll
        for (int q = 0; q < NT / 64; ++q) {
            lam = max_abs(lam, red[X.buf][q][0]);
            const double v = red[X.buf][q][1];
            nan |= v != v;
            mx = max_abs(mx, v);
        }
        const T d = urow[X.buf][0];
        const double akk = fabs((double)d);
        bool fast = akk >= p.eps && d != T(0);
        if (p.pivot != PV_NONE) fast = fast && !nan && akk >= p.u * mx;
        if (p.pivot == PV_BK) fast = fast && akk >= alpha * lam;
        if (!uni(fast)) return false;
        Global<T>* col = F.P + (int64_t)k * f;
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
                    if (u0 + u == 0 && up && tid < NBP) F.Ls[tid][k - k0] = l[0];
                    shift_update<W>(X.x[u0 + u], l[u], urow[X.buf]);
                }
            }
        }
        if (tid == 0) {
            kind[k] = KIND_1X1;
            dd[k] = d;
            ctype[k - k0] = 1;
        }
        if (d > T(0))
            X.npos++;
        else
            X.nneg++;
        ++k;
    }
    return true;
}

// a front's arrays during a panel
template <typename T>
struct PanelArgs {
    T *P, *U, *dd, *ee;
    int f, w, k0;
    int* lp;
    int8_t* kind;
    int64_t* st;
    const int8_t* sreq_row;
    const int32_t* perm_c0;
    LdltPrm prm;
};
// the LDS words of a panel. The front's arrays are kept here too: panel_general reads them back, so that they
// take no scalar registers during the usual pivots. ctype: per column q of the panel (k0 + q) the kind
// of its pivot step: 0 none yet, 1 a 1x1, 2 the first and 3 the second column of a 2x2
template <typename T, int NBP>
struct PanelLds {
    PanelArgs<T> args;
    RedBuf<512> rb;
    double pk[4], mx3[3][512 / 64];
    int ctype[NBP + 1];
    T Uc[NBP + 1], Lr[NBP + 1];
    T Ls[NBP + 1][NBP + 1];
    __align__(16) double red[2][512 / 64][2];
    __align__(16) T urow[2][NBP];
};
template <typename T, int NBP>
__device__ inline PanelLds<T, NBP>& panel_lds() {
    __shared__ PanelLds<T, NBP> lds;
    return lds;
}
template <typename T, int R, int NBP>
__device__ __attribute__((always_inline)) inline PanelFront<T, 512, R, NBP + 1> panel_front() {
    PanelLds<T, NBP>& S = panel_lds<T, NBP>();
    const PanelArgs<T>& A = S.args;
    const int w = uni(A.w), lane = threadIdx.x & 63, ct = S.ctype[min(lane, NBP)];
    Global<T>*U = uni_ptr(A.U), *DG = U + (int64_t)LP_MAXP * w;
    return PanelFront<T, 512, R, NBP + 1>{uni_ptr(A.P), uni(A.f), w, uni(A.k0), uni_ptr(A.lp), &S.rb, U, DG, DG + w,
                                          (uint32_t)__ballot(lane <= NBP && ct == 1),
                                          (uint32_t)__ballot(lane <= NBP && ct == 2), S.Uc, S.Lr, S.Ls, S.pk, S.mx3};
}

// any pivot but the usual one, at column k, from the panel memory (V holds the panel's columns from k
// on, nu pivot rows are formed); returns the next column. Part of the kernel: the panel's registers are free
// meanwhile. (As a function of its own, its pointers in a struct, it had its columns and the caller's
// registers in scratch memory and every access a flat one: a dense front of 1,500 columns with hardly a
// usual pivot took 41.7 ms, 24.5 now, 26.6 with one pivot per launch pair.)
template <typename T, int R, int NBP>
__device__ __attribute__((always_inline)) inline int panel_general(int k, int nu) {
    const auto Z = panel_front<T, R, NBP>();
    PanelLds<T, NBP>& S = panel_lds<T, NBP>();
    const PanelArgs<T>& A = S.args;
    const LdltPrm prm = {uni(A.prm.pivot), A.prm.u, A.prm.eps};
    const int tid = threadIdx.x, f = Z.f, k0 = Z.k0;
    k = uni(k);
    nu = uni(nu);
    Global<T>*P = Z.P, *dd = uni_ptr(A.dd), *ee = uni_ptr(A.ee);
    Global<int>* lp = Z.lp;
    int* ctype = S.ctype;
    double* pk = S.pk;
    Global<int8_t>* kind = uni_ptr(A.kind);
    Global<int64_t>* st = uni_ptr(A.st);
    T xa[R], xb[R];
    Z.load_rows(Z.V, xa);
    if (nu < k - k0) Z.form_urows(nu, k - k0);
    int c, r;
    Z.choose(k, prm, c, r, xa, xb);
    __syncthreads();
    Global<T>* ck = P + (int64_t)k * f;
    if (r < 0) {
        Z.template swap<false>(k, c, k - k0, xa, xb);
        Z.pick(xa, k, 0);
        __syncthreads();
        if (tid == 0) {
            double d = pk[0];
            int8_t kd = KIND_1X1;
            if (!(fabs(d) >= prm.eps) || d == 0.0) {
                if (d == 0.0) st[ST_NZERO]++;
                const int req = A.sreq_row ? (int)A.sreq_row[A.perm_c0[lp[k]]] : 0;
                const double sg = req != 0 ? (double)req : (d < 0.0 ? -1.0 : 1.0);
                d = sg * prm.eps;
                kd = KIND_PERTURBED;
                st[ST_NPERT]++;
                if (d == 0.0 && st[ST_INFO] == 0) st[ST_INFO] = lp[k] + 1;
            }
            ck[k] = T(d);
            kind[k] = kd;
            dd[k] = T(d);
            if (d > 0.0)
                st[ST_NPOS]++;
            else if (d < 0.0)
                st[ST_NNEG]++;
            pk[1] = d;
            ctype[k - k0] = 0;
        }
        __syncthreads();
        const T d = T(pk[1]);
        const auto rw = Z.rows();
        const int nf = rw.count(f);
#pragma unroll
        for (int u = 0; u < R; ++u) {
            xa[u] = xa[u] / d;
            if (u < nf && (u > 0 || tid > k - k0)) store_at(ck, rw.off(u), xa[u]);
        }
        Z.form_urow(k, k + 1);
        Z.template update_v<false>(k - k0, xa, xb);
        if (tid == 0) ctype[k - k0] = 1;
        k += 1;
    } else {
        Z.template swap<true>(k + 1, r, k - k0, xa, xb);
        Z.pick(xa, k, 0);
        Z.pick(xa, k + 1, 1);
        Z.pick(xb, k + 1, 2);
        __syncthreads();
        const T a = T(pk[0]), b = T(pk[1]), c2 = T(pk[2]);
        const T up = b;
        const T det = a * c2 - up * b;
        const T e11 = c2 / det, e12 = -up / det, e21 = -b / det, e22 = a / det;
        if (tid == 0) {
            kind[k] = KIND_2X2_FIRST;
            kind[k + 1] = KIND_2X2_SECOND;
            dd[k] = a;
            dd[k + 1] = c2;
            ee[k] = b;
            st[ST_N2X2]++;
            if (det < T(0)) {
                st[ST_NPOS]++;
                st[ST_NNEG]++;
            } else if (a > T(0)) {
                st[ST_NPOS] += 2;
            } else {
                st[ST_NNEG] += 2;
            }
            ck[k] = a;
            ck[f + k + 1] = c2;
            ck[k + 1] = T(0);  // the reference clears it
        }
        const auto rw = Z.rows();
        const int nf = rw.count(f);
#pragma unroll
        for (int u = 0; u < R; ++u) {
            const T x1 = xa[u], x2 = xb[u];
            xa[u] = x1 * e11 + x2 * e21;
            xb[u] = x1 * e12 + x2 * e22;
            if (u < nf && (u > 0 || tid > k + 1 - k0)) {
                store_at(ck, rw.off(u), xa[u]);
                store_at(ck + f, rw.off(u), xb[u]);
            }
        }
        Z.form_urow(k, k + 2);
        Z.form_urow(k + 1, k + 2);
        Z.template update_v<true>(k - k0, xa, xb);
        if (tid == 0) {
            ctype[k - k0] = 2;
            ctype[k + 1 - k0] = 3;
        }
        k += 2;
    }
    __syncthreads();
    return k;
}

// the next panel of every large front of a level: its pivots until NBP columns are taken or the
// front is done (the first panel also sets up the front; the upper triangle of the fully summed
// square was mirrored by k_ldlt_mirror). task: (s, scratch offset).
//
// Bound: latency, one workgroup per front walks the pivots one after another. NT = 512 (two waves
// per SIMD) leaves 256 registers a thread, 192 of them for the panel: NBP R <= 96. KKT, n = 12,000,
// FP64, one pivot in six not a usual one: a launch takes 78 us (16 columns, 3 rows a thread), 113 (6 rows), 64
// (8 columns), 43 (4), refactorization and solve 98 ms (157 with one pivot per launch pair). A
// usual pivot takes 3.5 us, another about 23 us with 3 rows a thread and 35 with 6.
template <typename T, int R, int NBP>
__global__ void __launch_bounds__(512) k_ldlt_panel(DevSym S, const Task* __restrict__ tasks, int first,
                                                    T* __restrict__ factor, T* __restrict__ dvec,
                                                    int32_t* __restrict__ piv, int8_t* __restrict__ pkind,
                                                    int64_t* __restrict__ stats, int32_t* __restrict__ lstep,
                                                    T* __restrict__ scratch, LdltPrm prm, int scaled,
                                                    const double* __restrict__ aux, const int8_t* __restrict__ psign) {
    constexpr int NT = 512;
    constexpr int MAXP = NBP + 1;
    static_assert(NBP == 4 || NBP == 8 || NBP == 16, "the usual pivots come in two runs: of NBP columns, then of 8");
    const Task tk = tasks[blockIdx.x];
    const int s = tk.s;
    const int f = S.fnrows[s], w = S.fncols[s];
    const int c0 = S.super_ptr[s];
    const int tid = threadIdx.x;
    prm.eps = eps_eff<T>(prm.eps, scaled, aux);
    T* P = factor + S.panel_off[s];
    int* lp = piv + c0;
    int8_t* kind = pkind + c0;
    T* dd = dvec + c0;
    T* ee = dvec + S.n + c0;
    int64_t* st = stats + (int64_t)s * NF;
    int32_t* ls = lstep + 3 * s;
    int k;
    if (first) {
        for (int q = tid; q < w; q += NT) {
            lp[q] = q;
            kind[q] = 0;
            dd[q] = ee[q] = T(0);
        }
        if (tid < NF) st[tid] = 0;
        k = 0;
    } else {
        k = uni(ls[2]);
    }
    __syncthreads();
    if (k >= w) {
        if (tid == 0) ls[1] = 0;
        return;
    }
    const int k0 = k, kend = min(w, k0 + NBP);
    PanelLds<T, NBP>& D = panel_lds<T, NBP>();
    for (int q = tid; q < MAXP; q += NT) D.ctype[q] = 0;
    if (tid == 0) D.args = {P, scratch + (int64_t)tk.a * PANEL_SCR_UNIT, dd, ee, f, w, k0, lp, kind, st, psign, S.perm + c0, prm};
    const int nr = (f - k0 + NT - 1) / NT;
    int nu = 0;  // U rows formed
    int kv = k0;  // the last general pivot
    int npos = 0, nneg = 0;
    while (k < kend) {
        __syncthreads();
        const auto Z = panel_front<T, R, NBP>();
        PanelRegs<T, R, NBP> X;
        X.nr = nr;
        X.buf = 0;
        X.npos = X.nneg = 0;
        // the panel's columns k.. in registers: the stored values, or after a general pivot V's
        const int np = k - k0, last = k - kv;  // (last: columns of that pivot, 0 at the panel's start)
        for (int q = tid; q < MAXP * np; q += NT) {
            const int pp = q / MAXP, r = q - pp * MAXP;
            if (r > pp && k0 + r < f) D.Ls[r][pp] = Z.P[(int64_t)(k0 + pp) * f + k0 + r];
        }
        const Global<T>* src = last ? Z.V + (int64_t)last * f : Z.P + (int64_t)k * f;
        const int cmax = last ? NBP - 1 - last : w - 1 - k;
        {
            const auto rw = Z.rows();
#pragma unroll
            for (int u = 0; u < R; ++u) {
                const uint32_t off = rw.clamped(u);
#pragma unroll
                for (int c = 0; c < NBP; ++c) X.x[u][c] = load_at(src + (int64_t)max(min(c, cmax), 0) * f, off);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __syncthreads();
        bool go = true;
        Global<int8_t>* gkind = uni_ptr(D.args.kind);
        Global<T>* gdd = uni_ptr(D.args.dd);
        if constexpr (NBP > 8) go = panel_pivots<T, NT, R, NBP, NBP>(X, Z, k, kend, prm, D.red, D.urow, D.ctype, gkind, gdd);
        if (go) go = panel_pivots<T, NT, R, NBP, (NBP < 8 ? NBP : 8)>(X, Z, k, kend, prm, D.red, D.urow, D.ctype, gkind, gdd);
        __syncthreads();  // the L columns are stored, the LDS words of the last pivot read
        npos += X.npos;
        nneg += X.nneg;
        if (go) break;
        // any other pivot, from the panel memory
        kv = k;
        {
            const auto rw = Z.rows();
            const int nf = rw.count(f);
#pragma unroll
            for (int u = 0; u < R; ++u) {
                if (u < nf) {
#pragma unroll
                    for (int c = 0; c < NBP; ++c) store_at(Z.V + (int64_t)c * f, rw.off(u), X.x[u][c]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __syncthreads();
        k = uni(panel_general<T, R, NBP>(k, nu));
        nu = k - k0;
    }
    // the rest of the pivot rows for the columns after the panel
    if (nu < k - k0 && k < w) panel_front<T, R, NBP>().form_urows(nu, k - k0);
    if (tid == 0) {
        st[ST_NPOS] += npos;
        st[ST_NNEG] += nneg;
        ls[0] = k0;
        ls[1] = k - k0;
        ls[2] = k;
    }
}

// the update of a panel's pivots on the columns after it: the tile rows [I0, I0 + 64) x columns
// [J0, J0 + 64) of the entries at or after the panel's end (every row below, the fully summed
// square's upper mirror included), each entry applying the panel's pivots in order as ldlt_front
// does. task: (s, I0, J0, scratch offset). Lanes along the rows, sixteen columns a wave: the
// thread's sixteen entries are loaded together, its row of L eight pivots at a time, the U rows
// come from LDS by broadcast. Bound: HBM / L2 (two accesses per entry and panel): 9.2 us a launch at n
// = 12,000 where one pivot's update took 6.
template <typename T>
__global__ void __launch_bounds__(256) k_ldlt_trail(DevSym S, const Task* __restrict__ tasks, T* __restrict__ factor,
                                                   const int8_t* __restrict__ pkind, const int32_t* __restrict__ lstep,
                                                   const T* __restrict__ scratch) {
    __shared__ __align__(16) T Us[LP_MAXP][TILE];
    __shared__ int8_t ks[LP_MAXP + 1];
    const Task t = tasks[blockIdx.x];
    const int s = t.s, f = S.fnrows[s], w = S.fncols[s];
    const int32_t* ls = lstep + 3 * s;
    const int np = ls[1];
    if (np == 0) return;
    const int k0 = ls[0], kend = ls[2];
    const int I0 = t.a, J0 = t.b;
    if (I0 + TILE <= kend || J0 + TILE <= kend) return;
    T* P = factor + S.panel_off[s];
    const int8_t* kind = pkind + S.super_ptr[s];
    const T* U = scratch + (int64_t)t.c * PANEL_SCR_UNIT;
    const int tid = threadIdx.x, i = I0 + (tid & 63), ic = min(i, f - 1), cb = (tid >> 6) * 16;
    for (int q = tid; q < np * TILE; q += 256) {
        const int pp = q / TILE, c = q - pp * TILE;
        Us[pp][c] = U[(int64_t)pp * w + min(J0 + c, w - 1)];
    }
    if (tid < np) ks[tid] = kind[k0 + tid];
    T x[16];
#pragma unroll
    for (int c = 0; c < 16; ++c) x[c] = P[(int64_t)min(J0 + cb + c, w - 1) * f + ic];
    __syncthreads();
    const T* Li = P + (int64_t)k0 * f + ic;
    for (int q0 = 0; q0 < np; q0 += 8) {
        T l[9];  // (one past the eight: the second column of a 2x2 pivot)
#pragma unroll
        for (int q = 0; q < 9; ++q) l[q] = Li[(int64_t)min(q0 + q, np - 1) * f];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            if (q0 + q >= np) break;
            const int kd = ks[q0 + q];
            if (kd == KIND_2X2_SECOND) continue;
            if (kd == KIND_2X2_FIRST) {
#pragma unroll
                for (int c = 0; c < 16; ++c)
                    x[c] = x[c] - (l[q] * Us[q0 + q][cb + c] + l[q + 1] * Us[q0 + q + 1][cb + c]);
            } else {
#pragma unroll
                for (int c = 0; c < 16; ++c) x[c] = x[c] - l[q] * Us[q0 + q][cb + c];
            }
        }
    }
    if (i < kend || i >= f) return;
#pragma unroll
    for (int c = 0; c < 16; ++c) {
        const int j = J0 + cb + c;
        if (j >= kend && j < w) P[(int64_t)j * f + i] = x[c];
    }
}

// after the last pair: unit diagonal, empty upper triangle and the global pivot order.
// task: (s)
template <typename T>
__global__ void __launch_bounds__(1024) k_ldlt_finish(DevSym S, const Task* __restrict__ tasks,
                                                     T* __restrict__ factor, int32_t* __restrict__ piv) {
    constexpr int NT = 1024;
    const int s = tasks[blockIdx.x].s;
    const int f = S.fnrows[s], w = S.fncols[s], c0 = S.super_ptr[s], tid = threadIdx.x;
    T* P = factor + S.panel_off[s];
    for (int q = tid; q < w * w; q += NT) {
        const int j = q / w, i = q - j * w;
        if (i <= j) P[(int64_t)j * f + i] = i == j ? T(1) : T(0);
    }
    for (int q = tid; q < w; q += NT) piv[c0 + q] = c0 + piv[c0 + q];
}

// Contribution block of a large front: the 64 x 64 tile (I0, J0) (front rows, I0 >= J0 >= w)
// of the lower triangle of F22 <- F22 - W L21^T, each entry subtracting W[i, k] L[j, k] for
// k = 0, 1, ..., w - 1 in order. Chunks of 16 columns of W and L21 are staged in LDS.
// Thread (ty, tx) owns rows I0 + 4 ty + a and columns J0 + 4 tx + b (a, b < 4).
template <typename T>
__global__ void __launch_bounds__(256) k_ldlt_cb(DevSym S, const Task* __restrict__ tasks,
                                                const T* __restrict__ factor, T* __restrict__ cbpool,
                                                const T* __restrict__ dvec, const int8_t* __restrict__ pkind) {
    constexpr int KC = 16;
    __shared__ T Ws[KC][TILE];
    __shared__ T Ls[KC][TILE];
    const Task t = tasks[blockIdx.x];
    const int s = t.s, f = S.fnrows[s], w = S.fncols[s], m = f - w;
    const int I0 = t.a, J0 = t.b;
    const int c0 = S.super_ptr[s];
    const T* L = factor + S.panel_off[s];
    T* C = cbpool + S.cb_off[s];
    const int8_t* kind = pkind + c0;
    const T* dd = dvec + c0;
    const T* ee = dvec + S.n + c0;
    const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
    T acc[4][4];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const int i = min(I0 + 4 * ty + a, f - 1), j = min(J0 + 4 * tx + b, f - 1);
            acc[a][b] = C[(int64_t)(j - w) * m + (i - w)];  // (clamped; entries j > i are not stored)
        }
    // the thread's four (kk, c) staging slots, kk = (tid >> 6) + 4 u, c = tid & 63: the raw
    // values of chunk k0 + KC (the L entries W(i, k) may combine, D, the pivot kinds, L(j, k))
    // are loaded, clamped, while chunk k0 is multiplied; W(i, k) is formed as w_entry forms it
    const int c = tid & 63, ic = min(I0 + c, f - 1), jc = min(J0 + c, f - 1);
    T l0[4], lm[4], lq[4], d0[4], e0[4], em[4], lj[4];
    int kd[4];
    auto load_raw = [&](int k0) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int kc = min(k0 + (tid >> 6) + 4 * u, w - 1), km = max(kc - 1, 0), kq = min(kc + 1, w - 1);
            kd[u] = kind[kc];
            l0[u] = L[(int64_t)kc * f + ic];
            lm[u] = L[(int64_t)km * f + ic];
            lq[u] = L[(int64_t)kq * f + ic];
            d0[u] = dd[kc];
            e0[u] = ee[kc];
            em[u] = ee[km];
            lj[u] = L[(int64_t)kc * f + jc];
        }
    };
    load_raw(0);
    for (int k0 = 0; k0 < w; k0 += KC) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int kk = (tid >> 6) + 4 * u, k = k0 + kk;
            const T wv = kd[u] == KIND_2X2_FIRST    ? l0[u] * d0[u] + lq[u] * e0[u]
                         : kd[u] == KIND_2X2_SECOND ? lm[u] * em[u] + l0[u] * d0[u]
                                                    : l0[u] * d0[u];
            Ws[kk][c] = (k < w && I0 + c < f) ? wv : T(0);
            Ls[kk][c] = (k < w && J0 + c < f) ? lj[u] : T(0);
        }
        __syncthreads();
        if (k0 + KC < w) load_raw(k0 + KC);
        const int kn = min(KC, w - k0);
        for (int kk = 0; kk < kn; ++kk) {
            T wv[4], lv[4];
#pragma unroll
            for (int a = 0; a < 4; ++a) wv[a] = Ws[kk][4 * ty + a];
#pragma unroll
            for (int b = 0; b < 4; ++b) lv[b] = Ls[kk][4 * tx + b];
#pragma unroll
            for (int a = 0; a < 4; ++a)
#pragma unroll
                for (int b = 0; b < 4; ++b) acc[a][b] = acc[a][b] - wv[a] * lv[b];
        }
        __syncthreads();
    }
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const int i = I0 + 4 * ty + a, j = J0 + 4 * tx + b;
            if (i < f && j <= i) C[(int64_t)(j - w) * m + (i - w)] = acc[a][b];
        }
}

// aux[0] = max |nzval| (the scale of pivot_epsilon_alg = "algo1"): non-negative doubles
// order like their bit patterns, so an integer atomic max is exact; a NaN wins, as the
// reference's NaN-propagating max. aux[0] must be zero on entry.
__global__ void k_absmax(int64_t nnz, const double* __restrict__ nz, unsigned long long* __restrict__ aux) {
    unsigned long long m = 0;
    for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < nnz; q += (int64_t)gridDim.x * blockDim.x) {
        const unsigned long long b = __double_as_longlong(fabs(nz[q]));
        m = b > m ? b : m;
    }
    for (int o = 32; o > 0; o >>= 1) {
        const unsigned long long x = __shfl_xor(m, o);
        m = x > m ? x : m;
    }
    if ((threadIdx.x & 63) == 0) atomicMax(aux, m);
}

// info[0] = the smallest failed factor column (1-based; 0 = none) over the fronts'
// statistics (ldlt.jl:208-216)
__global__ void __launch_bounds__(256) k_info_from_stats(DevSym S, const int64_t* __restrict__ stats,
                                                        int64_t* __restrict__ part) {
    __shared__ int64_t best[256];
    int64_t mn = INT64_MAX;
    for (int64_t s = blockIdx.x * 256 + threadIdx.x; s < S.ns; s += (int64_t)gridDim.x * 256) {
        const int64_t fi = stats[s * NF + ST_INFO];
        if (fi > 0) mn = min(mn, (int64_t)S.super_ptr[s] + fi);
    }
    best[threadIdx.x] = mn;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if (threadIdx.x < h) best[threadIdx.x] = min(best[threadIdx.x], best[threadIdx.x + h]);
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = best[0];
}

// ---------------------------------------------------------------------------

template <typename T>
void launch_front_small_ldlt(hipStream_t st, const DevSym& S, const int32_t* fronts, int nfronts, int fmax,
                             const double* nz, T* factor, T* cbpool, T* dvec, int32_t* piv, int8_t* kind,
                             int64_t* stats, int pivot, double u, double eps, int scaled, const double* aux,
                             const int8_t* psign) {
    size_t lds = (size_t)fmax * fmax * sizeof(T);
    LdltPrm p{pivot, u, eps};
    hipLaunchKernelGGL(k_front_small_ldlt<T>, dim3(nfronts), dim3(256), lds, st, S, fronts, nz, factor, cbpool, dvec,
                       piv, kind, stats, p, scaled, aux, psign);
}

template <typename T>
void launch_ldlt_pivot(hipStream_t st, const DevSym& S, const Task* tasks, int n, int t, T* factor, T* dvec,
                       int32_t* piv, int8_t* kind, int64_t* stats, int32_t* lstep, int pivot, double u, double eps,
                       int scaled, const double* aux, const int8_t* psign) {
    LdltPrm p{pivot, u, eps};
    hipLaunchKernelGGL(k_ldlt_pivot<T>, dim3(n), dim3(1024), 0, st, S, tasks, t, factor, dvec, piv, kind, stats,
                       lstep, p, scaled, aux, psign);
}

template <typename T>
void launch_ldlt_panel(hipStream_t st, const DevSym& S, const Task* tasks, int n, int first, int cols, int rows,
                       T* factor, T* dvec, int32_t* piv, int8_t* kind, int64_t* stats, int32_t* lstep, T* scratch, int pivot,
                       double u, double eps, int scaled, const double* aux, const int8_t* psign) {
    LdltPrm p{pivot, u, eps};
#define PANEL(R, C)                                                                                                  \
    hipLaunchKernelGGL((k_ldlt_panel<T, R, C>), dim3(n), dim3(512), 0, st, S, tasks, first, factor, dvec, piv, kind, \
                       stats, lstep, scratch, p, scaled, aux, psign)
    switch (cols) {
        case 16:  // (3 rows a thread do half the work of 6: 78 us a launch instead of 113)
            if (rows <= 3 * 512)
                PANEL(3, 16);
            else
                PANEL(6, 16);
            break;
        case 8: PANEL(10, 8); break;
        default: PANEL(14, 4); break;
    }
#undef PANEL
}

template <typename T>
void launch_ldlt_trail(hipStream_t st, const DevSym& S, const Task* tasks, int n, T* factor, const int8_t* kind,
                       const int32_t* lstep, const T* scratch) {
    hipLaunchKernelGGL(k_ldlt_trail<T>, dim3(n), dim3(256), 0, st, S, tasks, factor, kind, lstep, scratch);
}

int64_t ldlt_panel_scratch(int f, int w, int cols) { return lp_scratch(f, w, cols); }
// columns of the next panel of fronts with at most `rows` rows and `cols` columns left (0: too tall
// for the registers of one workgroup). The widest panel whose rows fit: a panel pays two launches
// and its loads and stores once, whatever its columns; no wider than the columns left need. Measured
// per column on the KKT fronts, with the update: 16 columns 5.4 to 7.6 us, 8 columns 9, 4 columns (5,121 to
// 7,168 rows) 13 us against 17.9 us of a launch pair; taller fronts do not fit the registers. Where hardly a pivot is
// a usual one (a dense front with zero diagonal) panels take 0.76 to 1.0 of the pairs' time, under a
// threshold that most of the diagonal fails up to 1.2 (n = 2,000, 0.9).
int ldlt_panel_cols(int rows, int cols) {
    if (rows <= 6 * 512 && cols > 8) return 16;
    if (rows <= 10 * 512) return 8;
    return rows <= 14 * 512 ? 4 : 0;
}

template <typename T>
void launch_ldlt_mirror(hipStream_t st, const DevSym& S, const Task* tasks, int n, T* factor) {
    hipLaunchKernelGGL(k_ldlt_mirror<T>, dim3(n), dim3(256), 0, st, S, tasks, factor);
}

template <typename T>
void launch_ldlt_update(hipStream_t st, const DevSym& S, const Task* tasks, int n, T* factor, const int32_t* lstep) {
    hipLaunchKernelGGL(k_ldlt_update<T>, dim3(n), dim3(256), 0, st, S, tasks, factor, lstep);
}

template <typename T>
void launch_ldlt_finish(hipStream_t st, const DevSym& S, const Task* tasks, int n, T* factor, int32_t* piv) {
    hipLaunchKernelGGL(k_ldlt_finish<T>, dim3(n), dim3(1024), 0, st, S, tasks, factor, piv);
}

template <typename T>
void launch_ldlt_cb(hipStream_t st, const DevSym& S, const Task* tasks, int n, const T* factor, T* cbpool,
                    const T* dvec, const int8_t* kind) {
    hipLaunchKernelGGL(k_ldlt_cb<T>, dim3(n), dim3(256), 0, st, S, tasks, factor, cbpool, dvec, kind);
}

void launch_absmax(hipStream_t st, int64_t nnz, const double* nz, double* aux) {
    hipLaunchKernelGGL(k_absmax, dim3((unsigned)std::min<int64_t>(std::max<int64_t>((nnz + 255) / 256, 1), 1024)),
                       dim3(256), 0, st, nnz, nz, reinterpret_cast<unsigned long long*>(aux));
}

void launch_info_from_stats(hipStream_t st, const DevSym& S, const int64_t* stats, int64_t* info) {
    // block minima at info + 8, then the smallest into info[0]
    const int blocks = (int)std::max<int64_t>(1, std::min<int64_t>(INFO_BLOCKS, (S.ns + 255) / 256));
    hipLaunchKernelGGL(k_info_from_stats, dim3(blocks), dim3(256), 0, st, S, stats, info + 8);
    launch_info_final(st, blocks, info);
}

#define INST(T)                                                                                                    \
    template void launch_front_small_ldlt<T>(hipStream_t, const DevSym&, const int32_t*, int, int, const double*, \
                                             T*, T*, T*, int32_t*, int8_t*, int64_t*, int, double, double, int,   \
                                             const double*, const int8_t*);                                        \
    template void launch_ldlt_cb<T>(hipStream_t, const DevSym&, const Task*, int, const T*, T*, const T*,         \
                                    const int8_t*);                                                                \
    template void launch_ldlt_pivot<T>(hipStream_t, const DevSym&, const Task*, int, int, T*, T*, int32_t*,        \
                                       int8_t*, int64_t*, int32_t*, int, double, double, int, const double*,       \
                                       const int8_t*);                                                             \
    template void launch_ldlt_update<T>(hipStream_t, const DevSym&, const Task*, int, T*, const int32_t*);        \
    template void launch_ldlt_mirror<T>(hipStream_t, const DevSym&, const Task*, int, T*);                        \
    template void launch_ldlt_panel<T>(hipStream_t, const DevSym&, const Task*, int, int, int, int, T*, T*,        \
                                       int32_t*, int8_t*, int64_t*, int32_t*, T*, int, double, double, int, const double*,   \
                                       const int8_t*);                                                             \
    template void launch_ldlt_trail<T>(hipStream_t, const DevSym&, const Task*, int, T*, const int8_t*,           \
                                       const int32_t*, const T*);                                                  \
    template void launch_ldlt_finish<T>(hipStream_t, const DevSym&, const Task*, int, T*, int32_t*);
INST(double)
INST(float)
#undef INST

}  // namespace sds
