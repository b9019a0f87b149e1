// Device helpers of the pivot panels held in one workgroup's registers (LDL^T, LU): lane reductions
// without an LDS round trip per step, addressing with a scalar base, and the register-rotating
// rank-1 update. The including files compile with contraction off.
#pragma once
#include "sds_common.h"

namespace sds {

// a value every lane holds, as a scalar
__device__ inline int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }

// max(m, |a|), a NaN in a passed over (fmax would first quiet both operands)
__device__ inline double max_abs(double m, double a) {
    double r;
    asm("v_max_f64 %0, %1, |%2|" : "=v"(r) : "v"(m), "v"(a));
    return r;
}
// a wave's largest v (v >= 0 in every lane; a NaN is passed over) in its last lane: row shifts and
// row broadcasts, no LDS round trip per step
template <int CTRL, int ROWS>
__device__ inline double dpp_max_step(double v) {
    const int2 x = __builtin_bit_cast(int2, v);
    int2 y;
    y.x = __builtin_amdgcn_update_dpp(0, x.x, CTRL, ROWS, 0xf, true);
    y.y = __builtin_amdgcn_update_dpp(0, x.y, CTRL, ROWS, 0xf, true);
    return max_abs(v, __builtin_bit_cast(double, y));
}
__device__ inline double wave_max_last(double v) {
    v = dpp_max_step<0x111, 0xf>(v);  // row_shr 1, 2, 4, 8
    v = dpp_max_step<0x112, 0xf>(v);
    v = dpp_max_step<0x114, 0xf>(v);
    v = dpp_max_step<0x118, 0xf>(v);
    v = dpp_max_step<0x142, 0xa>(v);  // row_bcast 15, 31
    return dpp_max_step<0x143, 0xc>(v);
}
__device__ inline double last_lane(double v) {
    int2 x = __builtin_bit_cast(int2, v);
    x.x = __builtin_amdgcn_readlane(x.x, 63);
    x.y = __builtin_amdgcn_readlane(x.y, 63);
    return __builtin_bit_cast(double, x);
}
// a wave's smallest i in its last lane
template <int CTRL, int ROWS>
__device__ inline int dpp_min_step(int v) {
    return min(v, __builtin_amdgcn_update_dpp(0x7fffffff, v, CTRL, ROWS, 0xf, false));
}
__device__ inline int wave_min_last(int v) {
    v = dpp_min_step<0x111, 0xf>(v);
    v = dpp_min_step<0x112, 0xf>(v);
    v = dpp_min_step<0x114, 0xf>(v);
    v = dpp_min_step<0x118, 0xf>(v);
    v = dpp_min_step<0x142, 0xa>(v);
    return dpp_min_step<0x143, 0xc>(v);
}

// pointers into global memory that say so: one that was itself read from memory is otherwise taken for
// a pointer to anything, its accesses become flat ones, and those are waited for together with the LDS
template <typename T>
using Global = __attribute__((address_space(1))) T;
// such a pointer from an address every lane holds, in scalar registers
template <typename T>
__device__ inline Global<T>* uni_ptr(T* p) {
    const uint64_t a = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((int)a), hi = __builtin_amdgcn_readfirstlane((int)(a >> 32));
    return (Global<T>*)((uint64_t)hi << 32 | lo);
}

// entry `off` bytes into the column `col` (a wave-uniform address: scalar base, 32-bit offset)
template <typename T>
__device__ inline T load_at(const T* col, uint32_t off) {
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(col) + off);
}
template <typename T>
__device__ inline T load_at(const Global<T>* col, uint32_t off) {
    return *(const Global<T>*)((const Global<char>*)col + off);
}
template <typename T>
__device__ inline void store_at(T* col, uint32_t off, T v) {
    *reinterpret_cast<T*>(reinterpret_cast<char*>(col) + off) = v;
}
template <typename T>
__device__ inline void store_at(Global<T>* col, uint32_t off, T v) {
    *(Global<T>*)((Global<char>*)col + off) = v;
}

// a thread's rows k0 + tid + NT u of a front: their byte offsets in a column and how many lie above an
// end. Both start from values hidden from the optimizer (empty asm): hoisted out of the pivot loop, the
// R comparisons of every loop would take R scalar register pairs each.
template <int NT, int SIZE>
struct PanelRows {
    uint32_t o0, olast;
    int left;  // k0 + tid
    __device__ __attribute__((always_inline)) PanelRows(int k0, int f) {
        left = k0 + (int)threadIdx.x;
        asm volatile("" : "+v"(left));
        o0 = (uint32_t)left * SIZE;
        olast = (uint32_t)(f - 1) * SIZE;
    }
    __device__ uint32_t off(int u) const { return o0 + (uint32_t)(NT * SIZE) * u; }
    __device__ uint32_t clamped(int u) const { return min(off(u), olast); }
    // slots u < count(end) hold rows below end
    __device__ int count(int end) const { return (end - left + NT - 1) >> (NT == 512 ? 9 : NT == 1024 ? 10 : 8); }
};

// N values computed here, not where they are used next (empty asm statements, which also order the
// memory accesses around them): without it the register allocator meets the loads of a whole panel
// update before the first of its sums, and the panel spills
template <int N, typename T>
__device__ __attribute__((always_inline)) inline void pin(T* v) {
#pragma unroll
    for (int c = 0; c < N; ++c) asm volatile("" : "+v"(v[c])::"memory");
}
// x[c - 1] = x[c] - l u[c] for 1 <= c < W: a row's rank-1 update, each column moving one register left;
// eight entries of u in flight together
template <int W, int C0 = 1, int N, typename T>
__device__ __attribute__((always_inline)) inline void shift_update(T (&x)[N], T l, const T* u) {
    constexpr int C1 = C0 + 8 < W ? C0 + 8 : W;
#pragma unroll
    for (int c = C0; c < C1; ++c) x[c - 1] = x[c] - l * u[c];
    pin<C1 - C0>(x + C0 - 1);
    if constexpr (C1 < W) shift_update<W, C1>(x, l, u);
}

}  // namespace sds
