// trsm_mfma.hip -- batched triangular solves and inverses on the register
// sweeps of tri_mfma.h, for triangles of order up to 512.
//
// magmablas_dtrsm_batched: six of its eight side / triangle / transpose cases
// (Left: not Trans with Lower; Right: not NoTrans with Lower).  In these the
// terms of an entry become final in the order in which the reference BLAS adds
// them, so the sweep gives its bits (up to the sign of a zero); the other two add the newest term first
// and stay with the lane-per-vector loops of blas_batched.hip.  Right-hand
// sides are the columns of B (Left) or its rows (Right), 16 to a work item.
//
// magma_dgetri_outofplace_batched: the row-interchanged identity is set up in
// LDS and both sweeps run on it, so the inverse is written once; before, the
// identity, the L solve and the U solve each made a pass over it.
//
// Bound: at order 64 the chain of the 4 x 4 triangles (one wavefront per 16
// vectors), with the factor read once per 16 vectors.  20,000 matrices of order
// 64: trsm with 16 vectors 1583 -> 185 us (3.6 TB/s of the 0.66 GB that has to
// move), the inverse 10.7 -> 0.81 ms.  Small triangles, and few vectors in large
// batches, stay with the lane-per-vector loops: blas_batched.hip draws the line.
#include <algorithm>

#include "kernels.h"
#include "tri_mfma.h"
#include "trsm_vector.h"

namespace magma_amd {
namespace {

constexpr int kTrsmMfmaMax = 512;

template <bool LEFT, int W, int NB>
__global__ void __launch_bounds__(64 * W, NB <= 2 || W == 1 ? 4 : NB == 4 ? 3 : 2)
trsm_mfma_kernel(int m, int n, double alpha, double **A_array, int lda, double **B_array, int ldb, bool lower,
                 bool trans, bool unit, int count, int nchunks)
{
    extern __shared__ double X[];
    const int tid = threadIdx.x, lane = tid & 63, w = W == 1 ? 0 : tid >> 6;
    const int L = LEFT ? m : n, nv = LEFT ? n : m;
    // the sweep's view: x_j -= A(k, j) x_k from the right is a transposed access
    const bool vtrans = LEFT ? trans : !trans;
    const double pre = LEFT || !trans ? alpha : 1.0, post = !LEFT && trans ? alpha : 1.0;
    for (long item = blockIdx.x; item < (long)count * nchunks; item += gridDim.x) {
        const int id = (int)(item / nchunks), v0 = 16 * (int)(item % nchunks);
        const int nc = min(16, nv - v0);
        const GDoublePtr A = (GDoublePtr)A_array[id];
        const GDoublePtr B = (GDoublePtr)B_array[id];
        // Left: lanes along a column of B; Right: 16 lanes along a column, four columns
        if (LEFT) {
#pragma unroll 1
            for (int c = w; c < 16; c += W)
#pragma unroll 4
                for (int k = lane; k < L; k += 64) {
                    const double b = c < nc ? B[k + (size_t)(v0 + c) * ldb] : 0.0;
                    X[k * kTriPitch + c] = pre != 1.0 ? pre * b : b;
                }
        } else {
#pragma unroll 4
            for (int k = tid >> 4; k < L; k += 4 * W) {
                const int c = tid & 15;
                const double b = c < nc ? B[v0 + c + (size_t)k * ldb] : 0.0;
                X[k * kTriPitch + c] = pre != 1.0 ? pre * b : b;
            }
        }
        __syncthreads();
        const bool fits = tri_fits(lda, L);
        if (fits) {
            const TriView v{A, lda, lower, vtrans};
            if (unit) tri_sweep<W, NB, kTriUnit>(v, L, X);
            else tri_sweep<W, NB, LEFT ? kTriDivide : kTriReciprocal>(v, L, X);
        }
        bool bad = !fits;
        for (int e = tid; e < L * 16; e += 64 * W) bad |= !__builtin_isfinite(X[(e >> 4) * kTriPitch + (e & 15)]);
        if (__syncthreads_or(bad)) {
            // the reference loops with their skips, on B itself
            const double *a = A_array[id];
            double *b = B_array[id];
            if (tid < nc) {
                const int v = v0 + tid;
                if (LEFT) {
                    auto x = [&](int k) -> double & { return b[k + (size_t)v * ldb]; };
                    if (!trans && lower) trsm_vector<'L', 'L', 'N'>(m, n, alpha, a, lda, unit, x);
                    else if (!trans) trsm_vector<'L', 'U', 'N'>(m, n, alpha, a, lda, unit, x);
                    else trsm_vector<'L', 'U', 'T'>(m, n, alpha, a, lda, unit, x);
                } else {
                    auto x = [&](int k) -> double & { return b[v + (size_t)k * ldb]; };
                    if (!trans) trsm_vector<'R', 'U', 'N'>(m, n, alpha, a, lda, unit, x);
                    else if (lower) trsm_vector<'R', 'L', 'T'>(m, n, alpha, a, lda, unit, x);
                    else trsm_vector<'R', 'U', 'T'>(m, n, alpha, a, lda, unit, x);
                }
            }
        } else if (LEFT) {
#pragma unroll 1
            for (int c = w; c < nc; c += W)
#pragma unroll 4
                for (int k = lane; k < L; k += 64) B[k + (size_t)(v0 + c) * ldb] = X[k * kTriPitch + c];
        } else {
            const int c = tid & 15;
            if (c < nc)
#pragma unroll 4
                for (int k = tid >> 4; k < L; k += 4 * W) {
                    const double x = X[k * kTriPitch + c];
                    B[v0 + c + (size_t)k * ldb] = post != 1.0 ? post * x : x;
                }
        }
        __syncthreads();
    }
}

// Columns 16 c .. 16 c + 15 of the inverse: U^-1 L^-1 P applied to those
// columns of the identity.  info (from the first work item of a matrix) is the
// first zero on U's diagonal, 1-based, or 0.
template <int W, int NB>
__global__ void __launch_bounds__(64 * W, NB <= 2 || W == 1 ? 4 : NB == 4 ? 3 : 2)
getri_mfma_kernel(int n, double **A_array, int lda, int **ipiv_array, double **I_array, int ldi, int *info, int count,
                  int nchunks)
{
    extern __shared__ double X[];
    int *pos = reinterpret_cast<int *>(X + (size_t)n * kTriPitch);
    __shared__ int first;
    const int tid = threadIdx.x, lane = tid & 63, w = W == 1 ? 0 : tid >> 6;
    for (long item = blockIdx.x; item < (long)count * nchunks; item += gridDim.x) {
        const int id = (int)(item / nchunks), v0 = 16 * (int)(item % nchunks);
        const int nc = min(16, n - v0);
        const GDoublePtr A = (GDoublePtr)A_array[id];
        final_positions<W, (16 * NB + 63) / 64>(ipiv_array[id], n, pos);
        if (tid == 0) first = n + 1;
        // one round for the identity, one more if the result is not finite
        auto identity = [&](int pitch, int step) {
            for (int e = tid; e < n * kTriPitch; e += 64 * W) X[e] = 0.0;
            __syncthreads();
            if (tid < nc) X[pos[v0 + tid] * pitch + tid * step] = 1.0;
            __syncthreads();
        };
        __syncthreads();
        identity(kTriPitch, 1);
        if (v0 == 0) {
            for (int i = tid; i < n; i += 64 * W)
                if (A[i + (size_t)i * lda] == 0.0) atomicMin(&first, i + 1);
        }
        const bool fits = tri_fits(lda, n);
        if (fits) {
            tri_sweep<W, NB, kTriUnit>(TriView{A, lda, true, false}, n, X);
            tri_sweep<W, NB, kTriDivide>(TriView{A, lda, false, false}, n, X);
        }
        bool bad = !fits;
        for (int e = tid; e < n * 16; e += 64 * W) bad |= !__builtin_isfinite(X[(e >> 4) * kTriPitch + (e & 15)]);
        const GDoublePtr V = (GDoublePtr)I_array[id];
        if (__syncthreads_or(bad)) {
            identity(1, n);
            reference_sweep(A_array[id], lda, n, X, n, nc, true, false, true);
            reference_sweep(A_array[id], lda, n, X, n, nc, false, false, false);
#pragma unroll 1
            for (int c = w; c < nc; c += W)
                for (int r = lane; r < n; r += 64) V[r + (size_t)(v0 + c) * ldi] = X[r + c * n];
        } else {
#pragma unroll 1
            for (int c = w; c < nc; c += W)
#pragma unroll 4
                for (int r = lane; r < n; r += 64) V[r + (size_t)(v0 + c) * ldi] = X[r * kTriPitch + c];
        }
        if (v0 == 0 && tid == 0 && info) info[id] = first > n ? 0 : first;
        __syncthreads();
    }
}

// One workgroup per work item; wavefronts per matrix and 16-row blocks per
// wavefront by the order of the triangle.
template <class F>
void by_order(int n, F &&go)
{
    if (n <= 64) go(std::integral_constant<int, 1>(), std::integral_constant<int, 4>());
    else if (n <= 128) go(std::integral_constant<int, 4>(), std::integral_constant<int, 2>());
    else if (n <= 256) go(std::integral_constant<int, 4>(), std::integral_constant<int, 4>());
    else go(std::integral_constant<int, 4>(), std::integral_constant<int, 8>());
}

}  // namespace

// The cases and orders above, alpha != 0; MAGMA_ERR_NOT_SUPPORTED for the others.
magma_int_t launch_trsm_mfma(bool left, bool lower, bool trans, bool unit, int m, int n, double alpha, double **A,
                             int lda, double **B, int ldb, int count, hipStream_t st)
{
    const int L = left ? m : n, nv = left ? n : m;
    if (L > kTrsmMfmaMax || alpha == 0.0 || (lower && left == trans)) return MAGMA_ERR_NOT_SUPPORTED;
    const int nchunks = ceil_div(nv, 16);
    const size_t lds = sizeof(double) * kTriPitch * (size_t)L;
    const int grid = (int)std::min((long)count * nchunks, 1l << 20);
    by_order(L, [&](auto W, auto NB) {
        constexpr int w = decltype(W)::value, nb = decltype(NB)::value;
        if (left)
            trsm_mfma_kernel<true, w, nb><<<grid, 64 * w, lds, st>>>(m, n, alpha, A, lda, B, ldb, lower, trans, unit,
                                                                     count, nchunks);
        else
            trsm_mfma_kernel<false, w, nb><<<grid, 64 * w, lds, st>>>(m, n, alpha, A, lda, B, ldb, lower, trans, unit,
                                                                      count, nchunks);
    });
    MAGMA_LAUNCH_CHECK();
    return MAGMA_SUCCESS;
}

// n <= 512; MAGMA_ERR_NOT_SUPPORTED above.
magma_int_t launch_getri_mfma(int n, double **A, int lda, int **ipiv, double **inv, int ldi, int *info, int count,
                              hipStream_t st)
{
    if (n > kTrsmMfmaMax) return MAGMA_ERR_NOT_SUPPORTED;
    const int nchunks = ceil_div(n, 16);
    const size_t lds = (sizeof(double) * kTriPitch + sizeof(int)) * (size_t)n;
    const int grid = (int)std::min((long)count * nchunks, 1l << 20);
    by_order(n, [&](auto W, auto NB) {
        constexpr int w = decltype(W)::value, nb = decltype(NB)::value;
        getri_mfma_kernel<w, nb><<<grid, 64 * w, lds, st>>>(n, A, lda, ipiv, inv, ldi, info, count, nchunks);
    });
    MAGMA_LAUNCH_CHECK();
    return MAGMA_SUCCESS;
}

}  // namespace magma_amd
