// trsm_vector.h -- reference BLAS dtrsm restricted to one vector: column v of B
// (Left, length m) or row v (Right, length n), each update one fma.
#pragma once

namespace magma_amd {

// x(k): reference to entry k of the vector; alpha != 0.
template <char SIDE, char UPLO, char TRANS, class X>
__device__ __forceinline__ void trsm_vector(int m, int n, double alpha, const double *a, int lda, bool unit, X x)
{
#define AA(i, j) a[(size_t)(i) + (size_t)(j) * lda]
    if (SIDE == 'L') {
        if (TRANS == 'N') {
            if (alpha != 1.0)
                #pragma unroll 4
                for (int i = 0; i < m; ++i) x(i) = alpha * x(i);
            if (UPLO == 'U') {
                for (int k = m - 1; k >= 0; --k) {
                    double bk = x(k);
                    if (bk != 0.0) {
                        if (!unit) bk = bk / AA(k, k);
                        x(k) = bk;
                        #pragma unroll 4
                        for (int i = 0; i < k; ++i) x(i) = fma(-bk, AA(i, k), x(i));
                    }
                }
            } else {
                for (int k = 0; k < m; ++k) {
                    double bk = x(k);
                    if (bk != 0.0) {
                        if (!unit) bk = bk / AA(k, k);
                        x(k) = bk;
                        #pragma unroll 4
                        for (int i = k + 1; i < m; ++i) x(i) = fma(-bk, AA(i, k), x(i));
                    }
                }
            }
        } else if (UPLO == 'U') {
            for (int i = 0; i < m; ++i) {
                double t = alpha * x(i);
                #pragma unroll 4
                for (int k = 0; k < i; ++k) t = fma(-AA(k, i), x(k), t);
                if (!unit) t = t / AA(i, i);
                x(i) = t;
            }
        } else {
            for (int i = m - 1; i >= 0; --i) {
                double t = alpha * x(i);
                #pragma unroll 4
                for (int k = i + 1; k < m; ++k) t = fma(-AA(k, i), x(k), t);
                if (!unit) t = t / AA(i, i);
                x(i) = t;
            }
        }
    } else if (TRANS == 'N') {
        if (UPLO == 'U') {
            for (int j = 0; j < n; ++j) {
                double t = x(j);
                if (alpha != 1.0) t = alpha * t;
                for (int k = 0; k < j; ++k) {
                    const double akj = AA(k, j);
                    if (akj != 0.0) t = fma(-akj, x(k), t);
                }
                if (!unit) t = (1.0 / AA(j, j)) * t;
                x(j) = t;
            }
        } else {
            for (int j = n - 1; j >= 0; --j) {
                double t = x(j);
                if (alpha != 1.0) t = alpha * t;
                for (int k = j + 1; k < n; ++k) {
                    const double akj = AA(k, j);
                    if (akj != 0.0) t = fma(-akj, x(k), t);
                }
                if (!unit) t = (1.0 / AA(j, j)) * t;
                x(j) = t;
            }
        }
    } else if (UPLO == 'U') {
        for (int k = n - 1; k >= 0; --k) {
            double bk = x(k);
            if (!unit) bk = (1.0 / AA(k, k)) * bk;
            for (int j = 0; j < k; ++j) {
                const double ajk = AA(j, k);
                if (ajk != 0.0) x(j) = fma(-ajk, bk, x(j));
            }
            if (alpha != 1.0) bk = alpha * bk;
            x(k) = bk;
        }
    } else {
        for (int k = 0; k < n; ++k) {
            double bk = x(k);
            if (!unit) bk = (1.0 / AA(k, k)) * bk;
            for (int j = k + 1; j < n; ++j) {
                const double ajk = AA(j, k);
                if (ajk != 0.0) x(j) = fma(-ajk, bk, x(j));
            }
            if (alpha != 1.0) bk = alpha * bk;
            x(k) = bk;
        }
    }
#undef AA
}

}  // namespace magma_amd
