// dpp_fma.h -- rank-1 updates of a register row with the other factor taken
// from a lane of the wavefront by DPP.
#pragma once

#include "kernels.h"

namespace magma_amd {

// a += x l, x lane K of x's 16 lanes: one v_fmac_f64 with a row_newbcast
// operand, where a readlane pair and an fma take three issues.  Every lane of
// the wavefront must be active, and x must have passed dpp_operand().
template <int K>
__device__ __forceinline__ void fmac_bcast(double &a, double x, double l)
{
    asm("v_fmac_f64_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf" : "+v"(a) : "v"(x), "v"(l), "n"(K));
}

template <int K>
__device__ __forceinline__ void fmac_bcast(float &a, float x, float l)
{
    asm("v_fmac_f32_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf" : "+v"(a) : "v"(x), "v"(l), "n"(K));
}

// a[K] += x[K] l for K0 <= K < K1, x[K] lane K % 16 of x0 (K < 16) or x1
template <int K0, int K1, int N, class T>
__device__ __forceinline__ void fmac_row(T (&a)[N], T x0, T x1, T l)
{
    if constexpr (K0 < K1) {
        fmac_bcast<(K0 & 15)>(a[K0], K0 < 16 ? x0 : x1, l);
        fmac_row<K0 + 1, K1>(a, x0, x1, l);
    }
}

// A DPP operand needs two wait states after a VALU write; the compiler does not
// look for it inside the asm above.
template <class T>
__device__ __forceinline__ void dpp_operand(T &x0, T &x1) { asm volatile("s_nop 1" : "+v"(x0), "+v"(x1)); }

// lane K of each row of 16 lanes, in all of them
template <int K>
__device__ __forceinline__ double row_bcast(double x)
{
    asm volatile("s_nop 1" : "+v"(x));      // x may come from the asm above
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, 0x150 + K, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x150 + K, 0xF, 0xF, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// The value with nothing known of how it was computed, so that addresses and
// masks derived from it are formed where they are used: hoisted out of loops
// they cost a hundred registers in the kernels that hold a block column.
__device__ __forceinline__ GDoublePtr opaque(GDoublePtr p)
{
    asm volatile("" : "+v"(p));
    return p;
}
__device__ __forceinline__ int opaque(int x)
{
    asm volatile("" : "+v"(x));
    return x;
}

}  // namespace magma_amd
