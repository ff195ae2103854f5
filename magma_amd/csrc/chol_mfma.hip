// chol_mfma.hip -- Cholesky, lower, FP64, 64 < n <= 512: one workgroup per
// matrix, one thread per row, left-looking by block columns of 32 columns.
//
//   update  C = A(j0.., block) in registers in the MFMA result layout,
//           wavefront w the 16-row tiles w, w + W, ...; C -= L(:, 0..j0)
//           L(block, 0..j0)' on v_mfma_f64_16x16x4f64, 16 columns of L a step
//           with the next step's operands in flight.  No barrier: both operands
//           are finished columns in memory.
//   panel   through LDS into one row per thread.  Every wavefront holds the
//           32 x 32 diagonal block too (lane li of each 16: rows li and 16 + li)
//           and factors it as it goes, so a column is a square root, a
//           reciprocal and rank-1 updates with DPP operands: nothing crosses
//           wavefronts and there is no barrier between columns.
//   store   the rows of the block column.
//
// What bounds it: the panel's chain (square root, reciprocal, the first update
// of a column) and, with three wavefronts per SIMD, their vector issue: at order
// 149 a wavefront waits 0.44 of its time, waits to issue 0.33 and issues VALU
// work 0.19 of it, about half of that work the diagonal block that every
// wavefront factors for itself; the matrix cores are 18% busy.  The form before,
// a right-looking panel of 16 columns with three barriers per column and the
// trailing matrix rewritten per panel: 2000 of order 149 0.606 -> 0.369 ms, 4096 of
// order 128 0.849 -> 0.350 ms, 256 of order 512 3.57 -> 0.955 ms, one of order 256
// 0.42 -> 0.125 ms.
//
// Replaces the reference's lg Cholesky (src/zpotrf_batched.cpp:20-221) for
// these sizes with one launch.
//
// Rounding: an entry gets fma(-l_ck, l_ik, a) in increasing k (the MFMA applies
// its four k terms as the sequential chain), then times 1 / l_cc: the netlib
// order.  The reference BLAS skips a zero l_ck; that can differ only where
// l_ik is not finite, and then row i's own diagonal entry stops the
// factorization at or before it, so no entry of the leading block that is
// final depends on it.
#include "dpp_fma.h"
#include "kernels.h"

#include <type_traits>

namespace magma_amd {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));

constexpr int PW = 32;              // columns of a block column
constexpr int TPW = 4;              // 16-row tiles per wavefront

__device__ __forceinline__ int pick(const int *arr, int fixed, int id) { return arr ? arr[id] : fixed; }

// Column K of the panel: the diagonal block's rows d0 (li), d1 (16 + li) and
// this thread's row a.
template <int K>
__device__ __forceinline__ void panel_columns(double (&d0)[16], double (&d1)[PW], double (&a)[PW], int row, int nb,
                                              int &fail)
{
    if constexpr (K < PW) {
        double dkk;
        if constexpr (K < 16) dkk = row_bcast<K>(d0[K]);
        else dkk = row_bcast<K - 16>(d1[K]);
        if (K < nb && !(dkk > 0.0)) fail = min(fail, K);
        const double ljj = sqrt(dkk), rc = 1.0 / ljj;
        double x0 = 0.0, x1;
        d1[K] = rc * d1[K];
        x1 = -d1[K];
        if constexpr (K < 16) {
            d0[K] = rc * d0[K];
            x0 = -d0[K];
        }
        const double l = rc * a[K];
        a[K] = row == K ? ljj : l;
        if constexpr (K < 16) fmac_row<K + 1, 16>(d0, x0, x1, d0[K]);
        fmac_row<K + 1, PW>(d1, x0, x1, d1[K]);
        fmac_row<K + 1, PW>(a, x0, x1, l);
        panel_columns<K + 1>(d0, d1, a, row, nb, fail);
    }
}

// Column K of the left half of the panel: the diagonal block's rows d0 (li) and
// d1 (16 + li), and this thread's row a.
template <int K>
__device__ __forceinline__ void left_columns(double (&d0)[16], double (&d1)[16], double (&a)[16], int row, int nb,
                                             int &fail)
{
    if constexpr (K < 16) {
        const double dkk = row_bcast<K>(d0[K]);
        if (K < nb && !(dkk > 0.0)) fail = min(fail, K);
        const double ljj = sqrt(dkk), rc = 1.0 / ljj;
        d0[K] = rc * d0[K];
        d1[K] = rc * d1[K];
        const double x0 = -d0[K];
        const double l = rc * a[K];
        a[K] = row == K ? ljj : l;
        fmac_row<K + 1, 16>(d0, x0, x0, d0[K]);
        fmac_row<K + 1, 16>(d1, x0, x0, d1[K]);
        fmac_row<K + 1, 16>(a, x0, x0, l);
        left_columns<K + 1>(d0, d1, a, row, nb, fail);
    }
}

// Column K of the left half taken from the right half: e the rows 16 + li, b this
// thread's row, d1 and a their entries in the left half.
template <int K>
__device__ __forceinline__ void apply_columns(double (&e)[16], double (&b)[16], const double (&d1)[16],
                                              const double (&a)[16])
{
    if constexpr (K < 16) {
        const double x = -d1[K];
        fmac_row<0, 16>(e, x, x, d1[K]);
        fmac_row<0, 16>(b, x, x, a[K]);
        apply_columns<K + 1>(e, b, d1, a);
    }
}

// Column 16 + K.
template <int K>
__device__ __forceinline__ void right_columns(double (&e)[16], double (&b)[16], int row, int nb, int &fail)
{
    if constexpr (K < 16) {
        const double dkk = row_bcast<K>(e[K]);
        if (16 + K < nb && !(dkk > 0.0)) fail = min(fail, 16 + K);
        const double ljj = sqrt(dkk), rc = 1.0 / ljj;
        e[K] = rc * e[K];
        const double x = -e[K];
        const double l = rc * b[K];
        b[K] = row == 16 + K ? ljj : l;
        fmac_row<K + 1, 16>(e, x, x, e[K]);
        fmac_row<K + 1, 16>(b, x, x, l);
        right_columns<K + 1>(e, b, row, nb, fail);
    }
}

// At 192 rows the LDS leaves room for three workgroups per CU but 206 registers
// only for two: there the panel goes in two halves of 16 columns and the update
// in steps of 8, which takes 150 (2000 of order 149 0.437 -> 0.383 ms, of order
// 192 0.530 -> 0.472 ms; 0.369 at order 149 since each row's updates are one statement).  At 128, 256 and 512 rows the LDS holds no more
// wavefronts than two per SIMD anyway, and the halves cost 3%.
template <int MT> constexpr bool three_per_simd() { return MT == 192; }

template <int MT>
__global__ void __launch_bounds__(MT) __attribute__((amdgpu_waves_per_eu(three_per_simd<MT>() ? 3 : 2))) potrf_mfma_kernel(MatSet s)
{
    constexpr int W = MT / 64;
    constexpr bool HALVES = three_per_simd<MT>();
    constexpr int KS = HALVES ? 8 : 16;         // columns of L per update step
    __shared__ double P[PW][MT + 1];
    __shared__ int failed;

    int tid = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    int li = tid & 15, lk = (tid >> 4) & 3;
    const int cnt = item_count(s);
    const int *idx = item_index(s);
    for (int item = blockIdx.x; item < cnt; item += gridDim.x) {
        const int id = idx ? idx[item] : item;
        const int n = pick(s.n_arr, s.n, id);
        const long lda = pick(s.lda_arr, s.lda, id);
        const GDoublePtr A = (GDoublePtr)s.A[id];
        int info = 0;
        __syncthreads();
        if (tid == 0) failed = PW;

        for (int j0 = 0; j0 < n; j0 += PW) {
            tid = opaque(tid);
            li = opaque(li);
            lk = opaque(lk);
            const int nb = min(PW, n - j0);
            // tiles with a row of the block column
            auto live = [&](int b) { return 16 * (w + W * b) + 16 > j0 && 16 * (w + W * b) < n; };
            int rowc[TPW];
#pragma unroll
            for (int b = 0; b < TPW; ++b) rowc[b] = min(16 * (w + W * b) + li, n - 1);
            // C: entry (row, column 16 t + lk + 4 i of the block) in c[b][t][i]
            d4 c[TPW][2];
            {
                GDoublePtr pc = opaque(A + min(j0 + lk, n - 1) * lda);
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
#pragma unroll
                        for (int b = 0; b < TPW; ++b) c[b][t][i] = pc[rowc[b]];
                        pc += j0 + 16 * t + lk + 4 * i + 4 < n ? 4 * lda : 0;
                        __builtin_amdgcn_sched_barrier(0);
                    }
            }
            // ------------------------------------------------ update -------
            // L(row, k) and -L(block row, k), k = k0 + 4 s + lk
            double lb[2][TPW][KS / 4], ua[2][2][KS / 4];
            const int r0 = min(j0 + li, n - 1), r1 = min(j0 + 16 + li, n - 1);
            auto load = [&](int k0, double (&l)[TPW][KS / 4], double (&u)[2][KS / 4]) {
                GDoublePtr pl = opaque(A + (k0 + lk) * lda);
#pragma unroll
                for (int k = 0; k < KS / 4; ++k) {
                    u[0][k] = pl[r0];
                    u[1][k] = pl[r1];
#pragma unroll
                    for (int b = 0; b < TPW; ++b) l[b][k] = pl[rowc[b]];
                    pl += 4 * lda;
                }
            };
            auto update = [&](const double (&l)[TPW][KS / 4], const double (&u)[2][KS / 4]) {
#pragma unroll
                for (int b = 0; b < TPW; b += 2)
                    if (live(b) || live(b + 1)) {
#pragma unroll
                        for (int k = 0; k < KS / 4; ++k)
#pragma unroll
                            for (int d = 0; d < 2; ++d)
#pragma unroll
                                for (int t = 0; t < 2; ++t)
                                    c[b + d][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(-u[t][k], l[b + d][k], c[b + d][t],
                                                                                       0, 0, 0);
                    }
            };
            if (j0 > 0) {
                load(0, lb[0], ua[0]);
#pragma unroll 1
                for (int k0 = 0; k0 < j0; k0 += 2 * KS) {       // j0 is a multiple of 32
                    load(k0 + KS, lb[1], ua[1]);
                    update(lb[0], ua[0]);
                    if (k0 + 2 * KS < j0) load(k0 + 2 * KS, lb[0], ua[0]);
                    update(lb[1], ua[1]);
                }
            }
            // ------------------------------------------------ panel --------
            li = opaque(li);
            lk = opaque(lk);
#pragma unroll
            for (int b = 0; b < TPW; ++b) {
                const int row = 16 * (w + W * b) + li;
                if (live(b) && row < n) {
#pragma unroll
                    for (int t = 0; t < 2; ++t)
#pragma unroll
                        for (int i = 0; i < 4; ++i) P[16 * t + lk + 4 * i][row] = c[b][t][i];
                }
            }
            __syncthreads();
            if (64 * w + 64 > j0 && 64 * w < n) {       // wavefronts with a row of the block column
                int fail = PW;
                if constexpr (HALVES) {
                    double a[16], b[16], d1[16], e[16];
                    const int q0 = min(j0 + li, n - 1), q1 = min(j0 + 16 + li, n - 1);
                    {
                        double d0[16];
#pragma unroll
                        for (int k = 0; k < 16; ++k) {
                            a[k] = P[k][tid];
                            d0[k] = P[k][q0];
                            d1[k] = P[k][q1];
                        }
                        left_columns<0>(d0, d1, a, tid - j0, nb, fail);
                    }
                    const int kn0 = min(nb, fail);
                    GDoublePtr pa = opaque(A + j0 * lda + tid);
                    auto store = [&](const double (&v)[16], int k0, int kn) {
#pragma unroll
                        for (int k = 0; k < 16; ++k) {
                            if (tid < n && tid >= j0 + k0 + k && k0 + k < kn) *pa = v[k];
                            pa += lda;
                        }
                    };
                    store(a, 0, kn0);
                    // row K's own entry of the left half holds l_kk: its right half is above the diagonal
#pragma unroll
                    for (int k = 0; k < 16; ++k) {
                        b[k] = P[16 + k][tid];
                        e[k] = P[16 + k][q1];
                    }
                    apply_columns<0>(e, b, d1, a);
                    right_columns<0>(e, b, tid - j0, nb, fail);
                    store(b, 16, min(nb, fail));
                } else {
                    double a[PW], d0[16], d1[PW];
                    const int q0 = min(j0 + li, n - 1), q1 = min(j0 + 16 + li, n - 1);
#pragma unroll
                    for (int k = 0; k < PW; ++k) {
                        a[k] = P[k][tid];
                        d1[k] = P[k][q1];
                        if (k < 16) d0[k] = P[k][q0];
                    }
                    panel_columns<0>(d0, d1, a, tid - j0, nb, fail);
                    const int kn = min(nb, fail);
                    GDoublePtr pa = opaque(A + j0 * lda + tid);
#pragma unroll
                    for (int k = 0; k < PW; ++k) {
                        if (tid < n && tid >= j0 + k && k < kn) *pa = a[k];
                        pa += lda;
                    }
                }
                if (fail < PW) failed = fail;           // the same in every wavefront
            }
            __syncthreads();
            if (failed < PW) {
                info = j0 + failed + 1;
                break;
            }
        }
        if (tid == 0) s.info[id] = info;
    }
}

}  // namespace

template <int MT>
static magma_int_t launch_mt(const MatSet &s, hipStream_t st)
{
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, potrf_mfma_kernel<MT>, MT, 0) != hipSuccess || nb < 1) nb = 1;
    potrf_mfma_kernel<MT><<<persistent_grid(s.count, nb), MT, 0, st>>>(s);
    MAGMA_LAUNCH_CHECK();
    return MAGMA_SUCCESS;
}

// 64 < n <= 512, by the order that a workgroup's rows cover
magma_int_t launch_potrf_mfma(const MatSet &s, int max_n, hipStream_t st)
{
    if (s.count <= 0) return MAGMA_SUCCESS;
    if (max_n > 512) return MAGMA_ERR_NOT_SUPPORTED;
    if (max_n <= 128) return launch_mt<128>(s, st);
    if (max_n <= 192) return launch_mt<192>(s, st);
    if (max_n <= 256) return launch_mt<256>(s, st);
    return launch_mt<512>(s, st);
}

}  // namespace magma_amd
