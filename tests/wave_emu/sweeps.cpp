// tri_sweep of every direction, triangle and scaling against plain loops, the
// operand ending at a page that must not be touched: its loads stay inside the
// matrix ("loads"), and neither what a solve does not read (the other triangle,
// the padding of lda; all NaN here) nor the rows past n that fill the last block
// reach a result ("values").
#include <hip/hip_runtime.h>

#include "tri_mfma.h"

using namespace magma_amd;

static double uniform(double lo, double hi) { return lo + (hi - lo) * (rand() / (RAND_MAX + 1.0)); }

static bool values;

template <int W, int NB, TriDiag DIAG>
static bool one(int n, int lda, bool lower, bool trans, bool large = false)
{
    const size_t elems = (size_t)(n - 1) * lda + n;
    double *a = emu::guard(elems, false), *X = emu::guard((size_t)n * kTriPitch, false);
    std::vector<double> want((size_t)n * 16);
    for (size_t e = 0; e < elems; ++e) {
        const int i = e % lda, j = e / lda;
        const bool read = i < n && (lower ? i > j : i < j), diag = i == j && DIAG != kTriUnit;
        a[e] = read ? uniform(-1, 1) / std::max(1.0, n / 8.0) : diag ? (rand() & 1 ? -1 : 1) * uniform(1, 2) : std::nan("");
    }
    for (int r = 0; r < n; ++r)
        for (int c = 0; c < 16; ++c) X[r * kTriPitch + c] = want[r * 16 + c] = c == 3 ? 0.0 : uniform(-1, 1);
    if (large) {
        // unit lower: the last row's sum is in range, but not without its start
        for (int i = 1; i < n; ++i) a[i] = i == n - 1;
        for (int i = 2; i < n; ++i) a[i + (size_t)lda] = i == n - 1;
        for (int c = 0; c < 16; ++c)
            for (int r : {0, 1, n - 1}) X[r * kTriPitch + c] = want[r * 16 + c] = r == n - 1 ? 1.6e308 : 1e308;
    }
    const bool forward = lower != trans;
    for (int s = 0; s < n; ++s) {
        const int k = forward ? s : n - 1 - s;
        for (int c = 0; c < 16; ++c) {
            double &x = want[k * 16 + c];
            const double d = a[k + (size_t)k * lda];
            if (DIAG == kTriDivide) x = x / d;
            if (DIAG == kTriReciprocal) x = (1.0 / d) * x;
            for (int i = forward ? k + 1 : 0; i < (forward ? n : k); ++i)
                want[i * 16 + c] = std::fma(-x, trans ? a[k + (size_t)i * lda] : a[i + (size_t)k * lda], want[i * 16 + c]);
        }
    }
    emu::outside = 0;
    emu::run(64 * W, [&] { tri_sweep<W, NB, DIAG>(TriView{(GDoublePtr)a, lda, lower, trans}, n, X); });
    if (!values) {
        if (emu::outside) std::printf("%ld loads outside: W=%d n=%d lda=%d lower=%d trans=%d\n", emu::outside, W, n, lda, lower, trans);
        return emu::outside == 0;
    }
    for (int r = 0; r < n; ++r)
        for (int c = 0; c < 16; ++c)
            if (X[r * kTriPitch + c] != want[r * 16 + c]) {
                std::printf("row %d vector %d: %g, not %g: W=%d n=%d lda=%d lower=%d trans=%d\n", r, c, X[r * kTriPitch + c],
                            want[r * 16 + c], W, n, lda, lower, trans);
                return false;
            }
    return true;
}

template <int W, int NB>
static bool all(std::initializer_list<int> orders)
{
    bool ok = true;
    for (int n : orders)
        for (int v = 0; v < 4; ++v) {
            const bool lower = v & 1, trans = v & 2;
            ok &= one<W, NB, kTriDivide>(n, n, lower, trans);
            ok &= one<W, NB, kTriUnit>(n, n + 3, lower, trans);
            if (n > 2 && lower && !trans) ok &= one<W, NB, kTriUnit>(n, n, lower, trans, true);
            if (n % 16 == 1) ok &= one<W, NB, kTriReciprocal>(n, n + 1, lower, trans);
        }
    return ok;
}

int main(int, char **argv)
{
    values = !std::strcmp(argv[1], "values");
    bool ok = all<1, 4>({1, 3, 15, 16, 17, 23, 27, 28, 31, 33, 48, 61, 64});
    ok &= all<4, 2>({49, 65, 72, 96, 113, 127, 128});
    ok &= all<4, 4>({129, 203, 241});
    if (!ok) return 1;
    std::puts("ok");
}
