// solve.hip -- triangular solves with LU / Cholesky factors (getrs, potrs), one
// launch and no workspace.  Replaces the reference's getrs/potrs chains
// (src/zgetrs_batched.cpp:86-273, src/zpotrs_batched.cpp:70-249:
// laswp_rowserial + trsv, or trtri_diag + trsm_outofplace GEMMs with a 128x128
// dinvA workspace per matrix).
//
//   n <= 512  16 right-hand sides at a time in the registers of one (n <= 64)
//             or four wavefronts: the sweeps of tri_mfma.h.
//             The 512 rows are what four wavefronts hold beside the factor
//             tiles in flight (256 registers a lane).  Against the kernel below
//             at its sizes: potrs 2000 x (149, 16 rhs) 1.13 -> 0.18 ms, getrs
//             256 x (500, 7 rhs) 1.90 -> 0.25 ms, getrs 8192 x (256, 1 rhs)
//             1.92 -> 1.19 ms (3.6 TB/s of the factor).
//   above     one 256-thread workgroup per matrix, up to 8 right-hand sides in
//             LDS, one barrier per column.  Also the tiniest systems.
//
// For the no-transpose L and U solves the order of an entry's terms is the
// reference BLAS dtrsm loop order, so results are bit-identical (in the register
// sweeps up to the sign of a zero) to LAPACK's dgetrs / dpotrs forward sweep; the transposed sweeps associate their sums in
// the opposite order to dtrsm's dot-product form and agree to rounding.
#include <algorithm>
#include <type_traits>

#include "kernels.h"
#include "tri_mfma.h"

namespace magma_amd {
namespace {

constexpr int kThreads = 256;
constexpr int kChunk = 8;

__device__ __forceinline__ int pick(const int *arr, int fixed, int id) { return arr ? arr[id] : fixed; }

// MODE 'N' getrs no-trans, 'T' getrs trans, 'C' potrs (triangle: lower);
// n <= 16 W NB.  A work item is a matrix and every nchunks-th group of 16 of
// its right-hand sides.
template <char MODE, int W, int NB>
__global__ void __launch_bounds__(64 * W, NB <= 2 || W == 1 ? 4 : NB == 4 ? 3 : 2) solve_mfma_kernel(MatSet s, bool lower, int nchunks)
{
    extern __shared__ double X[];
    constexpr char mode = MODE;
    const int cnt = item_count(s);
    const int *idx = item_index(s);
    const int tid = threadIdx.x, lane = tid & 63, w = W == 1 ? 0 : tid >> 6;
    constexpr bool lu = MODE != 'C';
    for (long item = blockIdx.x; item < (long)cnt * nchunks; item += gridDim.x) {
        const int seq = (int)(item / nchunks);
        const int id = idx ? idx[seq] : seq;
        const int n = __builtin_amdgcn_readfirstlane(pick(s.n_arr, s.n, id));
        const int lda = __builtin_amdgcn_readfirstlane(pick(s.lda_arr, s.lda, id));
        const int nrhs = __builtin_amdgcn_readfirstlane(pick(s.nrhs_arr, s.nrhs, id));
        const int ldb = __builtin_amdgcn_readfirstlane(pick(s.ldb_arr, s.ldb, id));
        const GDoublePtr A = (GDoublePtr)s.A[id];
        const GDoublePtr B = (GDoublePtr)s.B[id];
        if (n <= 0) continue;
        // after a fused factorization: no solve with a singular factor (dgesv/dposv)
        if (s.info && s.info[id] != 0) continue;
        // row r of B goes to row pos[r] of X ('N'), row pos[r] of X to row r of B ('T')
        int *pos = reinterpret_cast<int *>(X + (size_t)n * kTriPitch);
        if (lu) final_positions<W, (16 * NB + 63) / 64>(s.ipiv[id], n, pos);
        __syncthreads();
        for (int c0 = 16 * (int)(item % nchunks); c0 < nrhs; c0 += 16 * nchunks) {
            const int nc = min(16, nrhs - c0);
#pragma unroll 1
            for (int c = w; c < 16; c += W)
#pragma unroll 4
                for (int r = lane; r < n; r += 64)
                    X[(mode == 'N' ? pos[r] : r) * kTriPitch + c] = c < nc ? B[r + (size_t)(c0 + c) * ldb] : 0.0;
            __syncthreads();
            const bool fits = tri_fits(lda, n);
            if (!fits) {
            } else if (mode == 'N') {
                tri_sweep<W, NB, kTriUnit>(TriView{A, lda, true, false}, n, X);
                tri_sweep<W, NB, kTriDivide>(TriView{A, lda, false, false}, n, X);
            } else if (mode == 'T') {
                tri_sweep<W, NB, kTriDivide>(TriView{A, lda, false, true}, n, X);
                tri_sweep<W, NB, kTriUnit>(TriView{A, lda, true, true}, n, X);
            } else {
                tri_sweep<W, NB, kTriDivide>(TriView{A, lda, lower, !lower}, n, X);
                tri_sweep<W, NB, kTriDivide>(TriView{A, lda, lower, lower}, n, X);
            }
            bool bad = !fits;
            for (int e = tid; e < n * 16; e += 64 * W) bad |= !__builtin_isfinite(X[(e >> 4) * kTriPitch + (e & 15)]);
            if (__syncthreads_or(bad)) {
                // the reference loops and their skips, on the right-hand sides again
                const double *a = s.A[id];
                for (int c = w; c < nc; c += W)
                    for (int r = lane; r < n; r += 64)
                        X[c * n + (mode == 'N' ? pos[r] : r)] = B[r + (size_t)(c0 + c) * ldb];
                __syncthreads();
                for (int k = 0; k < 2; ++k) {
                    const bool first = k == 0;
                    const bool lo = mode == 'N' ? first : mode == 'T' ? !first : lower;
                    const bool tr = mode == 'T' || (mode == 'C' && first != lower);
                    reference_sweep(a, lda, n, X, n, nc, lo, tr, lu && lo);
                }
                for (int c = w; c < nc; c += W)
                    for (int r = lane; r < n; r += 64)
                        B[r + (size_t)(c0 + c) * ldb] = X[c * n + (mode == 'T' ? pos[r] : r)];
            } else {
                for (int c = w; c < nc; c += W)
#pragma unroll 4
                    for (int r = lane; r < n; r += 64)
                        B[r + (size_t)(c0 + c) * ldb] = X[(mode == 'T' ? pos[r] : r) * kTriPitch + c];
            }
            __syncthreads();
        }
    }
}

// mode: 'N' getrs no-trans, 'T' getrs trans, 'L' potrs lower, 'U' potrs upper.
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4))) solve_kernel(MatSet s, char mode, int chunk)
{
    extern __shared__ double X[];
    const int cnt = item_count(s);
    const int *idx = item_index(s);
    for (int item = blockIdx.x; item < cnt; item += gridDim.x) {
        const int id = idx ? idx[item] : item;
        const int n = pick(s.n_arr, s.n, id);
        const int lda = pick(s.lda_arr, s.lda, id);
        const int nrhs = pick(s.nrhs_arr, s.nrhs, id);
        const int ldb = pick(s.ldb_arr, s.ldb, id);
        const double *A = s.A[id];
        double *B = s.B[id];
        const int *ipiv = (mode == 'N' || mode == 'T') ? s.ipiv[id] : nullptr;
        const int tid = threadIdx.x;
        const int ldx = n;
        if (n <= 0) continue;
        // after a fused factorization: no solve with a singular factor (dgesv/dposv)
        if (s.info && s.info[id] != 0) continue;

        // the interchanges staged in LDS (after the right-hand-side chunk), so
        // the serial dlaswp chain below waits on LDS, not on a global load per step
        int *piv = reinterpret_cast<int *>(X + (size_t)n * chunk);
        if (ipiv) {
            for (int k = tid; k < n; k += kThreads) piv[k] = ipiv[k];
        }
        for (int c0 = 0; c0 < nrhs; c0 += chunk) {
            const int nc = min(chunk, nrhs - c0);
            for (int e = tid; e < n * nc; e += kThreads) {
                const int i = e % n, c = e / n;
                X[(size_t)c * ldx + i] = B[i + (size_t)(c0 + c) * ldb];
            }
            __syncthreads();
            if (mode == 'N') {
                // dlaswp forward: interchanges in order, one thread per column
                if (tid < nc)
                    for (int k = 0; k < n; ++k) {
                        const int p = piv[k] - 1;
                        if (p != k && p >= 0 && p < n) {
                            double *x = X + (size_t)tid * ldx;
                            const double t = x[k];
                            x[k] = x[p];
                            x[p] = t;
                        }
                    }
                __syncthreads();
                reference_sweep(A, lda, n, X, ldx, nc, true, false, true);
                reference_sweep(A, lda, n, X, ldx, nc, false, false, false);
            } else if (mode == 'T') {
                reference_sweep(A, lda, n, X, ldx, nc, false, true, false);
                reference_sweep(A, lda, n, X, ldx, nc, true, true, true);
                if (tid < nc)
                    for (int k = n - 1; k >= 0; --k) {
                        const int p = piv[k] - 1;
                        if (p != k && p >= 0 && p < n) {
                            double *x = X + (size_t)tid * ldx;
                            const double t = x[k];
                            x[k] = x[p];
                            x[p] = t;
                        }
                    }
                __syncthreads();
            } else if (mode == 'L') {
                reference_sweep(A, lda, n, X, ldx, nc, true, false, false);
                reference_sweep(A, lda, n, X, ldx, nc, true, true, false);
            } else {
                reference_sweep(A, lda, n, X, ldx, nc, false, true, false);
                reference_sweep(A, lda, n, X, ldx, nc, false, false, false);
            }
            for (int e = tid; e < n * nc; e += kThreads) {
                const int i = e % n, c = e / n;
                B[i + (size_t)(c0 + c) * ldb] = X[(size_t)c * ldx + i];
            }
            __syncthreads();
        }
        __syncthreads();
    }
}

// largest order whose 16 vectors fit the registers of four wavefronts
constexpr int kSolveMfmaMax = 512;

}  // namespace

static magma_int_t launch_solve(const MatSet &s, char mode, int max_n, hipStream_t st)
{
    if (s.count <= 0 || max_n <= 0) return MAGMA_SUCCESS;
    // A system of two to eight rows and a few right-hand sides fills neither a
    // tile nor a chain of 16 rows: the kernel below (sweeps / kernel below, 20,000
    // systems: n 2, 1 and 8 rhs 1.4 to 1.7 and 1.1 to 1.4; n 4, 1 rhs 1.0 to 1.2,
    // 4 rhs 0.8 to 1.0; n 8, 2 rhs 0.6 to 0.7.  64 systems: n 2, 16 rhs 1.1 to 1.2;
    // n 4, 8 rhs 1.0 to 1.2; n 6, 8 rhs 0.9 to 1.1; n 8, 4 rhs 0.9 to 1.05).
    const bool full = s.count > 4096;
    const bool tiny = !s.n_arr && !s.nrhs_arr && max_n <= (full ? 4 : 8) &&
                      (long)max_n * s.nrhs <= (full ? 16 : 32);
    if (max_n <= kSolveMfmaMax && !tiny) {
        const int nchunks = s.nrhs_arr ? 1 : std::max(1, ceil_div(s.nrhs, 16));
        const size_t lds = (size_t)max_n * (sizeof(double) * kTriPitch + sizeof(int));
        const long items = (long)s.count * nchunks;
        auto go = [&](auto kernel, int threads) {
            // one workgroup per item (the hardware keeps as many on a CU as fit);
            // a device-resident work list has fewer items than its bound
            const int grid = s.dev_count ? persistent_grid(items, 8) : (int)std::min(items, 1l << 20);
            kernel<<<grid, threads, lds, st>>>(s, mode == 'L', nchunks);
        };
        auto by_order = [&](auto tag) {
            constexpr char M = decltype(tag)::value;
            if (max_n <= 64) go(solve_mfma_kernel<M, 1, 4>, 64);
            else if (max_n <= 128) go(solve_mfma_kernel<M, 4, 2>, 256);
            else if (max_n <= 256) go(solve_mfma_kernel<M, 4, 4>, 256);
            else go(solve_mfma_kernel<M, 4, 8>, 256);
        };
        if (mode == 'N') by_order(std::integral_constant<char, 'N'>());
        else if (mode == 'T') by_order(std::integral_constant<char, 'T'>());
        else by_order(std::integral_constant<char, 'C'>());
        MAGMA_LAUNCH_CHECK();
        return MAGMA_SUCCESS;
    }
    // right-hand-side columns per pass: as many as fit 64 KB of LDS, at most kChunk
    const int chunk = std::min<long>(kChunk, (64 * 1024) / (sizeof(double) * (size_t)max_n));
    if (chunk < 1) return MAGMA_ERR_NOT_SUPPORTED;
    const size_t lds = sizeof(double) * (size_t)max_n * chunk + sizeof(int) * (size_t)max_n;
    const int grid = s.dev_count ? persistent_grid(s.count, 4) : s.count;
    solve_kernel<<<grid, kThreads, lds, st>>>(s, mode, chunk);
    MAGMA_LAUNCH_CHECK();
    return MAGMA_SUCCESS;
}

magma_int_t launch_getrs(const MatSet &s, char trans, int max_n, int max_nrhs, hipStream_t st)
{
    (void)max_nrhs;
    return launch_solve(s, trans == 'N' ? 'N' : 'T', max_n, st);
}

magma_int_t launch_potrs(const MatSet &s, char uplo, int max_n, int max_nrhs, hipStream_t st)
{
    (void)max_nrhs;
    return launch_solve(s, uplo == 'L' ? 'L' : 'U', max_n, st);
}

}  // namespace magma_amd
