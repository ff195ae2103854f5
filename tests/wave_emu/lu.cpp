// getrf's kernel for 64 < max(m, n) <= 128 on matrices without entries (whose
// pointers are null) among ordinary ones that end, or begin, at a page that
// must not be touched; the ordinary ones against the netlib loops.
#include <hip/hip_runtime.h>

#include "lu_kernel.inc"

using namespace magma_amd;

static void reference(int m, int n, double *a, int lda, int *ipiv)
{
    for (int j = 0; j < std::min(m, n); ++j) {
        int p = j;
        for (int i = j + 1; i < m; ++i)
            if (std::fabs(a[i + j * lda]) > std::fabs(a[p + j * lda])) p = i;
        ipiv[j] = p + 1;
        for (int c = 0; c < n; ++c) std::swap(a[j + c * lda], a[p + c * lda]);
        for (int i = j + 1; i < m; ++i) {
            const double l = a[i + j * lda] * (1.0 / a[j + j * lda]);
            a[i + j * lda] = l;
            for (int c = j + 1; c < n; ++c) a[i + c * lda] = std::fma(l, -a[j + c * lda], a[i + c * lda]);
        }
    }
}

int main()
{
    const int count = 7;
    int m[count] = {0, 100, 70, 0, 66, 128, 128}, n[count] = {100, 0, 66, 128, 128, 33, 0}, lda[count], info[count];
    double *A[count] = {}, *B[count] = {};
    int piv[count][128], want[128], *ipiv[count];
    srand(3);
    for (int s = 0; s < count; ++s) {
        lda[s] = std::max(1, m[s]);
        info[s] = -1;
        ipiv[s] = piv[s];
        const size_t e = (size_t)m[s] * n[s];
        if (!e) continue;
        A[s] = emu::guard(e, s & 1);
        B[s] = (double *)malloc(8 * e);
        for (size_t i = 0; i < e; ++i) A[s][i] = B[s][i] = rand() / (double)RAND_MAX - 0.5;
    }
    MatSet set;
    set.m_arr = m; set.n_arr = n; set.lda_arr = lda;
    set.A = A; set.ipiv = ipiv; set.info = info;
    set.count = count;
    emu::run(128, [&] { getrf_mfma_kernel<128>(set); });
    for (int s = 0; s < count; ++s) {
        if (info[s] != 0) return std::printf("matrix %d (%d x %d): info %d\n", s, m[s], n[s], info[s]), 1;
        if (!A[s]) continue;
        reference(m[s], n[s], B[s], lda[s], want);
        if (std::memcmp(want, piv[s], sizeof(int) * std::min(m[s], n[s])))
            return std::printf("matrix %d: pivots\n", s), 1;
        for (int i = 0; i < m[s] * n[s]; ++i)
            if (A[s][i] != B[s][i]) return std::printf("matrix %d: entry %d\n", s, i), 1;
    }
    std::puts("ok");
}
