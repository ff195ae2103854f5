// dpp_fma.h -- rank-1 updates of a register row with the other factor taken
// from a lane of the wavefront by DPP.
#pragma once

#include "kernels.h"

namespace magma_amd {

// a[K0 + i] += x l, x lane (K0 + i) % 16 of x's 16 lanes, for i < C: v_fmac with a
// row_newbcast operand, where a readlane pair and an fma take three issues.
// Every lane of the wavefront must be active.
//
// One asm statement, the wait states first: a DPP operand needs two after a VALU
// write, and the compiler, which does not look for them inside an asm, may put a
// copy of x right before any statement that reads it.
#define MAGMA_FMAC(T, i) "\n\tv_fmac_" T "_dpp %" #i ", %[x], %[l] row_newbcast:%[k]+" #i " row_mask:0xf bank_mask:0xf"
#define MAGMA_FMAC1(T) MAGMA_FMAC(T, 0)
#define MAGMA_ACC1 "+&v"(a[K0])
#define MAGMA_FMAC2(T) MAGMA_FMAC1(T) MAGMA_FMAC(T, 1)
#define MAGMA_ACC2 MAGMA_ACC1, "+&v"(a[K0 + 1])
#define MAGMA_FMAC3(T) MAGMA_FMAC2(T) MAGMA_FMAC(T, 2)
#define MAGMA_ACC3 MAGMA_ACC2, "+&v"(a[K0 + 2])
#define MAGMA_FMAC4(T) MAGMA_FMAC3(T) MAGMA_FMAC(T, 3)
#define MAGMA_ACC4 MAGMA_ACC3, "+&v"(a[K0 + 3])
#define MAGMA_FMAC5(T) MAGMA_FMAC4(T) MAGMA_FMAC(T, 4)
#define MAGMA_ACC5 MAGMA_ACC4, "+&v"(a[K0 + 4])
#define MAGMA_FMAC6(T) MAGMA_FMAC5(T) MAGMA_FMAC(T, 5)
#define MAGMA_ACC6 MAGMA_ACC5, "+&v"(a[K0 + 5])
#define MAGMA_FMAC7(T) MAGMA_FMAC6(T) MAGMA_FMAC(T, 6)
#define MAGMA_ACC7 MAGMA_ACC6, "+&v"(a[K0 + 6])
#define MAGMA_FMAC8(T) MAGMA_FMAC7(T) MAGMA_FMAC(T, 7)
#define MAGMA_ACC8 MAGMA_ACC7, "+&v"(a[K0 + 7])
#define MAGMA_FMAC9(T) MAGMA_FMAC8(T) MAGMA_FMAC(T, 8)
#define MAGMA_ACC9 MAGMA_ACC8, "+&v"(a[K0 + 8])
#define MAGMA_FMAC10(T) MAGMA_FMAC9(T) MAGMA_FMAC(T, 9)
#define MAGMA_ACC10 MAGMA_ACC9, "+&v"(a[K0 + 9])
#define MAGMA_FMAC11(T) MAGMA_FMAC10(T) MAGMA_FMAC(T, 10)
#define MAGMA_ACC11 MAGMA_ACC10, "+&v"(a[K0 + 10])
#define MAGMA_FMAC12(T) MAGMA_FMAC11(T) MAGMA_FMAC(T, 11)
#define MAGMA_ACC12 MAGMA_ACC11, "+&v"(a[K0 + 11])
#define MAGMA_FMAC13(T) MAGMA_FMAC12(T) MAGMA_FMAC(T, 12)
#define MAGMA_ACC13 MAGMA_ACC12, "+&v"(a[K0 + 12])
#define MAGMA_FMAC14(T) MAGMA_FMAC13(T) MAGMA_FMAC(T, 13)
#define MAGMA_ACC14 MAGMA_ACC13, "+&v"(a[K0 + 13])
#define MAGMA_FMAC15(T) MAGMA_FMAC14(T) MAGMA_FMAC(T, 14)
#define MAGMA_ACC15 MAGMA_ACC14, "+&v"(a[K0 + 14])
#define MAGMA_FMAC16(T) MAGMA_FMAC15(T) MAGMA_FMAC(T, 15)
#define MAGMA_ACC16 MAGMA_ACC15, "+&v"(a[K0 + 15])
#define MAGMA_FMAC_CASE(C0)                                                                                     \
    if constexpr (C == C0 && sizeof(T) == 8)                                                                    \
        asm("s_nop 1" MAGMA_FMAC##C0("f64") : MAGMA_ACC##C0 : [x] "v"(x), [l] "v"(l), [k] "n"(K0 & 15));        \
    else if constexpr (C == C0)                                                                                 \
        asm("s_nop 1" MAGMA_FMAC##C0("f32") : MAGMA_ACC##C0 : [x] "v"(x), [l] "v"(l), [k] "n"(K0 & 15));
template <int K0, int C, int N, class T>
__device__ __forceinline__ void fmac_group(T (&a)[N], T x, T l)
{
    static_assert(C >= 0 && (K0 & 15) + C <= 16 && K0 + C <= N);
    MAGMA_FMAC_CASE(1) MAGMA_FMAC_CASE(2) MAGMA_FMAC_CASE(3) MAGMA_FMAC_CASE(4)
    MAGMA_FMAC_CASE(5) MAGMA_FMAC_CASE(6) MAGMA_FMAC_CASE(7) MAGMA_FMAC_CASE(8)
    MAGMA_FMAC_CASE(9) MAGMA_FMAC_CASE(10) MAGMA_FMAC_CASE(11) MAGMA_FMAC_CASE(12)
    MAGMA_FMAC_CASE(13) MAGMA_FMAC_CASE(14) MAGMA_FMAC_CASE(15) MAGMA_FMAC_CASE(16)
}

// a[K] += x[K] l for K0 <= K < K1, x[K] lane K % 16 of x0 (K < 16) or x1
template <int K0, int K1, int N, class T>
__device__ __forceinline__ void fmac_row(T (&a)[N], T x0, T x1, T l)
{
    if constexpr (K0 < K1) {
        constexpr int C = (K1 - K0 < 16 - (K0 & 15)) ? K1 - K0 : 16 - (K0 & 15);
        fmac_group<K0, C>(a, K0 < 16 ? x0 : x1, l);
        fmac_row<K0 + C, K1>(a, x0, x1, l);
    }
}

// lane K of each row of 16 lanes, in all of them
template <int K>
__device__ __forceinline__ double row_bcast(double x)
{
    asm volatile("s_nop 1" : "+v"(x));      // x may come from the asm above; a copy after this is the compiler's to see
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
__device__ __forceinline__ LDoublePtr opaque(LDoublePtr p)
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
