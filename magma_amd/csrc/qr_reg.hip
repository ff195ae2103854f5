// qr_reg.hip -- batched Householder QR with the matrix in registers, for
// m, n <= 128.
//
// W wavefronts hold one matrix as a grid of RG row lanes by 64 / RG column
// lanes per wavefront; a lane keeps RL rows of CL columns (64 doubles at most)
// from the load to the store.  Rows are dealt in pairs, columns cyclically, so
// the finished rows and columns drop out of the unrolled loops as the
// factorization moves down the diagonal.
//
// Per column i: the lanes that hold it sum its squares (a few lane-local fmas
// and a DPP sum over the RG row lanes), the reflector goes to the other lanes
// through one LDS row (RG different addresses per read, the rest broadcast),
// and every lane forms its columns' partial dot products, the DPP sums over
// the row lanes and the update.  No barrier while one wavefront holds the
// matrix; one per column with four (the row is double-buffered by parity).
//
// Bound: the chain of a column (sum, square root, two divisions, LDS hand-off,
// dot, update) on two wavefronts per SIMD.  A workgroup per matrix with the
// matrix in LDS, which this replaces at these sizes, spent its time in the two
// workgroup reductions and four barriers of each column: 20,000 matrices of
// order 64 took 9.40 ms, and take 0.89 ms here (1.5 TB/s of the 1.32 GB that
// has to move; a wavefront issues VALU work 0.42 of its time and waits 0.20).  At 128 the grid of four wavefronts still holds the matrix
// (64 doubles a lane); above, the workgroup kernel of blas_batched.hip runs.
//
// Numerics: netlib dgeqr2's reflectors (dlarfg's beta = -sign(alpha)
// hypot(alpha, ||x||), tau = (beta - alpha) / beta, v = (1; x / (alpha - beta))).
// The sum of squares is taken directly while it is well inside the exponent
// range and else as max |x| times the root of the scaled sum, so no square
// over- or underflows; the direct sum has fewer roundings than the scaled one.
#include <cfloat>
#include <cmath>

#include "kernels.h"

namespace magma_amd {
namespace {

template <int CTRL>
__device__ __forceinline__ double dpp_f64(double x)
{
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xF, 0xF, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// sum over the RG lanes of a group (4: a quad, 8: half a row of 16), in all of them
template <int RG>
__device__ __forceinline__ double group_sum(double x)
{
    x += dpp_f64<0xB1>(x);                          // quad_perm [1,0,3,2]
    x += dpp_f64<0x4E>(x);                          // quad_perm [2,3,0,1]
    if constexpr (RG == 8) x += dpp_f64<0x141>(x);  // row_half_mirror
    return x;
}

template <int RG>
__device__ __forceinline__ double group_max(double x)
{
    x = fmax(x, dpp_f64<0xB1>(x));
    x = fmax(x, dpp_f64<0x4E>(x));
    if constexpr (RG == 8) x = fmax(x, dpp_f64<0x141>(x));
    return x;
}

__device__ __forceinline__ double lane_value(double x, int lane)
{
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_readlane((int)b, lane), hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

template <int W>
__device__ __forceinline__ void matrix_sync()
{
    if constexpr (W == 1) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    } else {
        __syncthreads();
    }
}

// m <= RG RL, n <= 64 / RG * W * CL.
template <int RG, int RL, int CL, int W>
__global__ void __launch_bounds__(64 * W, 2) geqrf_reg_kernel(int m, int n, double **A_array, int lda,
                                                              double **tau_array, int *info, int count)
{
    constexpr int CG = 64 / RG;          // column lanes per wavefront
    constexpr int CW = CG * W;           // columns per local column
    constexpr int MT = RG * RL;
    __shared__ double2 vbuf[2][MT / 2 + 1];      // the reflector; then tau
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int g = lane % RG, cpos = wave * CG + lane / RG;
    // The last row has no reflector (rows past m may hold NaN by then).
    const int k = min(m - 1, n);
    for (int id = blockIdx.x; id < count; id += gridDim.x) {
        GDoublePtr A = (GDoublePtr)A_array[id];
        GDoublePtr tau = (GDoublePtr)tau_array[id];
        if (tid == 0 && info) info[id] = 0;
        if (tid == 0 && m <= n) tau[m - 1] = 0.0;
        double a[CL][RL];
#pragma unroll
        for (int c = 0; c < CL; ++c)
#pragma unroll
            for (int l = 0; l < RL; ++l) {
                const int r = 2 * RG * (l / 2) + 2 * g + (l & 1), col = CW * c + cpos;
                a[c][l] = (r < m && col < n) ? A[r + (size_t)col * lda] : 0.0;
            }
#pragma unroll
        for (int lc = 0; lc < CL; ++lc) {
            // local rows below L0 are finished, those below L1 hold the diagonal
            constexpr int kR2 = 2 * RG;
            const int L0 = 2 * (CW * lc / kR2), L1 = 2 * ((CW * (lc + 1) + kR2 - 1) / kR2);
#pragma unroll 1
            for (int p = 0; p < CW; ++p) {
                const int i = CW * lc + p;
                if (i >= k) break;
                double2 *vb = vbuf[i & 1];
                if (W == 1 || wave == p / CG) {
                    const int owner = (p % CG) * RG;       // first lane of the column
                    double s0 = 0.0, s1 = 0.0, al = 0.0;
#pragma unroll
                    for (int l = 0; l < RL; ++l) {
                        if (l < L0) continue;
                        const int r = 2 * RG * (l / 2) + 2 * g + (l & 1);
                        const double x = a[lc][l];
                        double y = x;
                        if (l < L1) {
                            al = (r == i) ? x : al;
                            y = (r > i) ? x : 0.0;
                        }
                        if (l & 1) s1 = fma(y, y, s1);
                        else s0 = fma(y, y, s0);
                    }
                    const double ss = lane_value(group_sum<RG>(s0 + s1), owner);
                    const double alpha = lane_value(al, owner + (i / 2) % RG);
                    double t = 0.0, beta = alpha, sc = 0.0;
                    const double hh = fma(alpha, alpha, ss);
                    if (ss > 0x1p-900 && hh < 0x1p+1000) {
                        beta = -copysign(sqrt(hh), alpha);
                        t = (beta - alpha) / beta;
                        sc = 1.0 / (alpha - beta);
                    } else {
                        double mx = 0.0;
#pragma unroll
                        for (int l = 0; l < RL; ++l) {
                            if (l < L0) continue;
                            const int r = 2 * RG * (l / 2) + 2 * g + (l & 1);
                            mx = fmax(mx, r > i ? fabs(a[lc][l]) : 0.0);
                        }
                        const double amax = lane_value(group_max<RG>(mx), owner);
                        double sq = 0.0;
                        if (amax > 0.0) {
#pragma unroll
                            for (int l = 0; l < RL; ++l) {
                                if (l < L0) continue;
                                const int r = 2 * RG * (l / 2) + 2 * g + (l & 1);
                                const double y = r > i ? a[lc][l] / amax : 0.0;
                                sq = fma(y, y, sq);
                            }
                        }
                        // fmax drops a NaN: where it is all the column has, amax is 0
                        const double xnorm = ss == ss ? amax * sqrt(lane_value(group_sum<RG>(sq), owner)) : ss;
                        if (xnorm != 0.0) {
                            const double xa = fabs(alpha), wmax = fmax(xa, xnorm), wmin = fmin(xa, xnorm);
                            // fmax and fmin would drop a NaN
                            const double hyp = (xa == xa && xnorm == xnorm)
                                                   ? wmax * sqrt(1.0 + (wmin / wmax) * (wmin / wmax)) : xa + xnorm;
                            beta = -copysign(hyp, alpha);
                            t = (beta - alpha) / beta;
                            sc = 1.0 / (alpha - beta);
                        }
                    }
                    if (cpos == p) {
                        if (t != 0.0) {
#pragma unroll
                            for (int l = 0; l < RL; l += 2) {
                                if (l < L0) continue;
                                double v[2];
#pragma unroll
                                for (int h = 0; h < 2; ++h) {
                                    const int r = 2 * RG * (l / 2) + 2 * g + h;
                                    const double x = a[lc][l + h], y = x * sc;
                                    v[h] = y;
                                    if (l < L1) {
                                        a[lc][l + h] = r > i ? y : (r == i ? beta : x);
                                        v[h] = r > i ? y : (r == i ? 1.0 : 0.0);
                                    } else {
                                        a[lc][l + h] = y;
                                    }
                                }
                                vb[RG * (l / 2) + g] = make_double2(v[0], v[1]);
                            }
                        }
                        if (g == 0) {
                            tau[i] = t;
                            vb[MT / 2].x = t;
                        }
                    }
                }
                matrix_sync<W>();
                const double t = vb[MT / 2].x;
                if (t != 0.0) {
                    double v[RL];
#pragma unroll
                    for (int l = 0; l < RL; l += 2) {
                        if (l < L0) continue;
                        const double2 y = vb[RG * (l / 2) + g];
                        v[l] = y.x;
                        v[l + 1] = y.y;
                    }
                    double w[CL];
#pragma unroll
                    for (int c = 0; c < CL; ++c) w[c] = 0.0;
#pragma unroll
                    for (int l = 0; l < RL; ++l) {
                        if (l < L0) continue;
                        const int r = 2 * RG * (l / 2) + 2 * g + (l & 1);
                        // rows of R are not touched, whatever they hold
                        if (l >= L1 || r >= i) {
#pragma unroll
                            for (int c = 0; c < CL; ++c)
                                if (c >= lc) w[c] = fma(v[l], a[c][l], w[c]);
                        }
                    }
#pragma unroll
                    for (int c = 0; c < CL; ++c)
                        if (c >= lc) w[c] = -t * group_sum<RG>(w[c]);
                    if (cpos > p) {
#pragma unroll
                        for (int l = 0; l < RL; ++l) {
                            if (l < L0) continue;
                            const int r = 2 * RG * (l / 2) + 2 * g + (l & 1);
                            if (l >= L1 || r >= i) a[lc][l] = fma(w[lc], v[l], a[lc][l]);
                        }
                    }
#pragma unroll
                    for (int l = 0; l < RL; ++l) {
                        if (l < L0) continue;
                        const int r = 2 * RG * (l / 2) + 2 * g + (l & 1);
                        if (l >= L1 || r >= i) {
#pragma unroll
                            for (int c = 0; c < CL; ++c)
                                if (c > lc) a[c][l] = fma(w[c], v[l], a[c][l]);
                        }
                    }
                }
                if constexpr (W == 1) matrix_sync<W>();
            }
        }
#pragma unroll
        for (int c = 0; c < CL; ++c)
#pragma unroll
            for (int l = 0; l < RL; ++l) {
                const int r = 2 * RG * (l / 2) + 2 * g + (l & 1), col = CW * c + cpos;
                if (r < m && col < n) A[r + (size_t)col * lda] = a[c][l];
            }
        // the next matrix's first column reuses a row of vbuf
        if constexpr (W > 1) __syncthreads();
    }
}

}  // namespace

// m, n <= 128 (MAGMA_ERR_NOT_SUPPORTED above); also clears info.
magma_int_t launch_geqrf_reg(int m, int n, double **A, int lda, double **tau, int *info, int count, hipStream_t st)
{
    if (m > 128 || n > 128) return MAGMA_ERR_NOT_SUPPORTED;
    const int grid1 = persistent_grid(count, 8);
    if (m <= 16 && n <= 16)
        geqrf_reg_kernel<4, 4, 1, 1><<<persistent_grid(count, 32), 64, 0, st>>>(m, n, A, lda, tau, info, count);
    else if (m <= 32 && n <= 32)
        geqrf_reg_kernel<4, 8, 2, 1><<<persistent_grid(count, 24), 64, 0, st>>>(m, n, A, lda, tau, info, count);
    else if (m <= 64 && n <= 16)
        geqrf_reg_kernel<4, 16, 1, 1><<<persistent_grid(count, 16), 64, 0, st>>>(m, n, A, lda, tau, info, count);
    else if (m <= 64 && n <= 64)
        geqrf_reg_kernel<4, 16, 4, 1><<<grid1, 64, 0, st>>>(m, n, A, lda, tau, info, count);
    else if (n <= 32)
        geqrf_reg_kernel<8, 16, 4, 1><<<grid1, 64, 0, st>>>(m, n, A, lda, tau, info, count);
    else
        geqrf_reg_kernel<8, 16, 4, 4><<<persistent_grid(count, 2), 256, 0, st>>>(m, n, A, lda, tau, info, count);
    MAGMA_LAUNCH_CHECK();
    return MAGMA_SUCCESS;
}

}  // namespace magma_amd
