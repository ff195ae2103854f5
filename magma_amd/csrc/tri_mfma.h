// tri_mfma.h -- triangular sweeps on 16 right-hand sides with the vectors in
// registers: the device code of getrs, potrs, getri and the forward trsm cases.
//
// The 16 vectors are one tile column of v_mfma_f64_16x16x4f64: lane (lk = lane
// / 16, li = lane % 16) holds, of 16-row block t, the rows 16 t + 4 i + lk (i =
// 0..3) of vector li.  That is the MFMA's result layout and, register by
// register, also its B operand for the k slices 4 i .. 4 i + 3, so a solved
// block feeds the updates of the blocks below it as it is.  W wavefronts hold
// the blocks cyclically (block t in wavefront t % W); a solved block reaches
// the other wavefronts through X, the vectors' LDS array, with one barrier per
// 16 columns.  The 16 x 16 diagonal blocks are solved on the vector unit: the
// value of a row reaches the four row groups by permlane swaps, a column of
// the block by DPP row_newbcast from registers.
//
// Why: a sweep with one barrier per column (one row per thread, X in LDS)
// costs a barrier and an LDS round trip per column and right-hand-side pass,
// and reads the factor once per 8 right-hand sides; here the chain of a column
// is in registers, the factor's tiles for the next block column are in flight
// while a diagonal block is solved, and 16 right-hand sides share one read.
//
// Rounding: an entry gets its terms as single fmas in the order of the solved
// rows (the MFMA applies its four k terms as the sequential chain), then the
// division: the reference BLAS order of the forward cases.  The reference's
// skip of a zero x_k (or zero factor entry) can change a result only where the
// other operand is not finite, and then the result here is not finite either:
// callers test that and redo such a matrix with the reference loops.
#pragma once

#include "kernels.h"

namespace magma_amd {

typedef double d4 __attribute__((ext_vector_type(4)));

constexpr int kTriPitch = 17;       // doubles per row of X: 16 vectors and one of padding (banks)

// How a sweep scales a solved row.
enum TriDiag { kTriUnit = 0, kTriDivide = 1, kTriReciprocal = 2 };

// A column-major n x n triangle and the direction in which a sweep takes it:
// lower or upper, transposed or not; forward (ascending rows) when lower !=
// trans.  Logical row s of a sweep is solved s-th: row s forward, row 16
// ceil(n / 16) - 1 - s backward, so a block of 16 is a block of 16 of the
// matrix either way and the rows past n come last or first.
struct TriView {
    GDoublePtr a;
    long lda;
    bool lower, trans;
};

// Offsets into the triangle are 32-bit byte offsets of a buffer resource.
__device__ __forceinline__ bool tri_fits(long lda, int n) { return lda * n < (1l << 28); }

namespace tri_detail {

// x of row group G (lanes 16 G .. 16 G + 15) in all four groups
template <int G>
__device__ __forceinline__ double group_bcast(double x)
{
    const long long b = __double_as_longlong(x);
    unsigned r[2] = {(unsigned)b, (unsigned)(b >> 32)};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        // [x0 x0 x2 x2] and [x1 x1 x3 x3], then one half twice
        const auto p = __builtin_amdgcn_permlane16_swap(r[h], r[h], false, false);
        const unsigned y = (G & 1) ? p[1] : p[0];
        const auto q = __builtin_amdgcn_permlane32_swap(y, y, false, false);
        r[h] = (G & 2) ? q[1] : q[0];
    }
    return __longlong_as_double(((long long)r[1] << 32) | r[0]);
}

__device__ __forceinline__ double lane_value(double x, int lane)
{
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_readlane((int)b, lane), hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// lane S of each row of 16 lanes, in all 16
template <int S>
__device__ __forceinline__ double row_lane(double x)
{
    return __longlong_as_double(
        __builtin_amdgcn_update_dpp(0LL, __double_as_longlong(x), 0x150 + S, 0xF, 0xF, true));
}

// t[i] holds entry (4 i + lk, li); r its reciprocals (kTriReciprocal)
template <int S, TriDiag DIAG>
__device__ __forceinline__ void diag_step(d4 &x, const d4 &t, const d4 &r, int lk)
{
    constexpr int IS = S >> 2, G = S & 3;
    double xs = group_bcast<G>(x[IS]);
    if constexpr (DIAG == kTriDivide) xs = xs / lane_value(t[IS], 16 * G + S);
    if constexpr (DIAG == kTriReciprocal) xs = lane_value(r[IS], 16 * G + S) * xs;
#pragma unroll
    for (int i = IS; i < 4; ++i) {
        const double y = fma(-xs, row_lane<S>(t[i]), x[i]);
        if (i > IS) {
            x[i] = y;
        } else {
            const double z = lk > G ? y : x[i];
            x[i] = lk == G ? xs : z;
        }
    }
}

template <int S, TriDiag DIAG>
__device__ __forceinline__ void diag_steps(d4 &x, const d4 &t, const d4 &r, int lk)
{
    diag_step<S, DIAG>(x, t, r, lk);
    __builtin_amdgcn_sched_barrier(0);          // one column's broadcasts at a time in registers
    if constexpr (S < 15) diag_steps<S + 1, DIAG>(x, t, r, lk);
}

// The 16 x 16 diagonal block.
template <TriDiag DIAG>
__device__ __forceinline__ void diag_solve(d4 &x, const d4 &t, int lk)
{
    d4 r = t;
    if constexpr (DIAG == kTriReciprocal)
#pragma unroll
        for (int i = 0; i < 4; ++i) r[i] = 1.0 / t[i];
    diag_steps<0, DIAG>(x, t, r, lk);
}

}  // namespace tri_detail

// One sweep over X (row r of vector c at X[r * kTriPitch + c]).  All 64 W
// threads; n <= 16 W NB and tri_fits.  X must be complete and visible on entry
// (barrier) and is so on return.
template <int W, int NB, TriDiag DIAG>
__device__ __forceinline__ void tri_sweep(TriView v, int n, double *X)
{
    using namespace tri_detail;
    const int lane = threadIdx.x & 63, w = W == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int li = lane & 15, lk = lane >> 4;
    const bool rev = v.lower == v.trans;
    const int nt = (n + 15) >> 4;
    const int pad = rev ? 16 * nt - n : 0;      // logical rows that are past n come first
    // the matrix pointer is the same in every lane: a scalar resource
    const unsigned long long pa = (unsigned long long)v.a;
    const unsigned plo = __builtin_amdgcn_readfirstlane((int)pa), phi = __builtin_amdgcn_readfirstlane((int)(pa >> 32));
    const auto rs = __builtin_amdgcn_make_buffer_rsrc((void *)(((unsigned long long)phi << 32) | plo), 0,
                                                      8 * (int)((n - 1) * v.lda + n), 0x00020000);
    // byte steps of a logical row and column, forward
    const int ds = 8 * (v.trans ? (int)v.lda : 1), dk = 8 * (v.trans ? 1 : (int)v.lda);
    const int tile = (rev ? 15 - li : li) * ds + (rev ? 3 - lk : lk) * dk;
    const int diag = (rev ? 3 - lk : lk) * ds + (rev ? 15 - li : li) * dk;
    auto ld = [&](int lane_off, int off) {
        return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rs, lane_off, off, 0));
    };
    auto at = [&](int t) { return 16 * (rev ? nt - 1 - t : t); };           // first matrix row of block t
    auto xrow = [&](int s) { return (rev ? 16 * nt - 1 - s : s) * kTriPitch + li; };
    // factor tile below the diagonal: A operand of slice i, entry (row li, column 4 i + lk)
    auto load_tile = [&](int tr, int tc, d4 &a) {
#pragma unroll
        for (int i = 0; i < 4; ++i) a[i] = ld(tile, at(tr) * ds + (at(tc) + 4 * (rev ? 3 - i : i)) * dk);
    };
    auto load_diag = [&](int t, d4 &a) {
#pragma unroll
        for (int i = 0; i < 4; ++i) a[i] = ld(diag, (at(t) + 4 * (rev ? 3 - i : i)) * ds + at(t) * dk);
    };
    d4 x[NB], av[NB], dt;
    load_diag(min(w, nt - 1), dt);
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const int t = w + W * b;
        x[b] = d4{0.0, 0.0, 0.0, 0.0};
        av[b] = x[b];
        if (t < nt) {
            if (t > 0) load_tile(t, 0, av[b]);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int s = 16 * t + 4 * i + lk;
                if (rev ? s >= pad : s < n) x[b][i] = X[xrow(s)];
            }
        }
    }
    if (pad > 0) {
        // rows past n come first: no coupling, unit diagonal
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int s = 4 * i + lk;
            if (w == 0 && (s < pad || li < pad)) dt[i] = s == li ? 1.0 : 0.0;
#pragma unroll
            for (int b = 0; b < NB; ++b)
                if (s < pad) av[b][i] = 0.0;
        }
    }
#pragma unroll 1
    for (int t0 = 0; t0 < nt; t0 += W) {
        // x[0] is block t0 + w here
#pragma unroll 1
        for (int ww = 0; ww < W; ++ww) {
            const int t = t0 + ww;
            if (t >= nt) break;
            if (W == 1 || w == ww) {
                diag_solve<DIAG>(x[0], dt, lk);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int s = 16 * t + 4 * i + lk;
                    if (rev ? s >= pad : s < n) X[xrow(s)] = x[0][i];
                }
                if (t + W < nt) load_diag(t + W, dt);
            }
            if (t + 1 >= nt) break;
            d4 xb;
            if constexpr (W == 1) {
                xb = -x[0];
            } else {
                __syncthreads();
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int s = 16 * t + 4 * i + lk;
                    xb[i] = s >= pad ? -X[xrow(s)] : 0.0;
                }
            }
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                const int tr = t0 + w + W * b;
                if (tr > t && tr < nt) {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        x[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[b][i], xb[i], x[b], 0, 0, 0);
                    if (tr > t + 1) load_tile(tr, t + 1, av[b]);
                }
            }
        }
#pragma unroll
        for (int b = 0; b + 1 < NB; ++b) {
            x[b] = x[b + 1];
            av[b] = av[b + 1];
        }
    }
    __syncthreads();
}

// Row positions after the interchanges ipiv[0..n) (1-based; entries out of
// range are ignored) applied in order: row r ends in row pos[r].  Each
// wavefront tracks the rows 64 (w + W j) + lane against the pivots read 64 at
// a time, so a step costs four VALU instructions and waits on nothing.
template <int W, int NR>
__device__ __forceinline__ void final_positions(const int *ipiv, int n, int *pos)
{
    const int lane = threadIdx.x & 63, w = W == 1 ? 0 : threadIdx.x >> 6;
    const GIntPtr gp = (GIntPtr)ipiv;
    int p[NR];
#pragma unroll
    for (int j = 0; j < NR; ++j) p[j] = 64 * (w + W * j) + lane;
#pragma unroll 1
    for (int k0 = 0; k0 < n; k0 += 64) {
        const int kn = min(64, n - k0);
        int v = lane < kn ? gp[k0 + lane] - 1 : k0 + lane;
        if (v < 0 || v >= n) v = k0 + lane;
#pragma unroll 4
        for (int k = 0; k < kn; ++k) {
            const int q = __builtin_amdgcn_readlane(v, k), kk = k0 + k;
#pragma unroll
            for (int j = 0; j < NR; ++j) p[j] = p[j] == kk ? q : (p[j] == q ? kk : p[j]);
        }
    }
#pragma unroll
    for (int j = 0; j < NR; ++j)
        if (64 * (w + W * j) + lane < n) pos[64 * (w + W * j) + lane] = p[j];
}

// The reference BLAS sweep over X (n x nc, LDS, leading dimension ldx) with
// factor T, one column at a time, with its skip of zero entries.
//   lower/upper: which triangle of T is used; trans: op(T) = T';
//   unit: implicit unit diagonal.  op(T) lower -> forward sweep, upper -> backward.
__device__ inline void reference_sweep(const double *T, int ldt, int n, double *X, int ldx, int nc,
                                       bool lower, bool trans, bool unit)
{
    const int tid = threadIdx.x, nthr = blockDim.x;
    const bool forward = (lower != trans);
    if (n <= nthr) {
        // one row per thread: the next step's entries of T (its column, or row
        // when transposed, and its diagonal) are loaded while the current step
        // runs, so each step does not wait on a global load
        auto entry = [&](int k, int i) { return trans ? T[k + (size_t)i * ldt] : T[i + (size_t)k * ldt]; };
        auto row_of = [&](int k) { return (forward ? k + 1 : 0) + tid; };
        auto row_end = [&](int k) { return forward ? n : k; };
        int k = forward ? 0 : n - 1;
        double tc = 0.0, dc = 1.0;
        if (row_of(k) < row_end(k)) tc = entry(k, row_of(k));
        if (!unit && tid < nc) dc = T[k + (size_t)k * ldt];
        for (int s = 0; s < n; ++s) {
            k = forward ? s : n - 1 - s;
            double tn = 0.0, dn = 1.0;
            if (s + 1 < n) {
                const int k1 = forward ? s + 1 : n - 2 - s;
                if (row_of(k1) < row_end(k1)) tn = entry(k1, row_of(k1));
                if (!unit && tid < nc) dn = T[k1 + (size_t)k1 * ldt];
            }
            if (!unit) {
                if (tid < nc) {
                    double *xk = X + (size_t)tid * ldx + k;
                    // no-transpose sweeps skip a zero entry like reference dtrsm;
                    // its transposed (dot-form) sweeps always divide
                    if (trans || *xk != 0.0) *xk = *xk / dc;
                }
                __syncthreads();
            }
            const int i = row_of(k);
            if (i < row_end(k)) {
                for (int c = 0; c < nc; ++c) {
                    const double xk = X[(size_t)c * ldx + k];
                    if (!trans && xk == 0.0) continue;      // reference dtrsm's skip (x_k stays 0 after division)
                    X[(size_t)c * ldx + i] = fma(-xk, tc, X[(size_t)c * ldx + i]);
                }
            }
            __syncthreads();
            tc = tn;
            dc = dn;
        }
        return;
    }
    for (int s = 0; s < n; ++s) {
        const int k = forward ? s : n - 1 - s;
        if (!unit) {
            if (tid < nc) {
                double *xk = X + (size_t)tid * ldx + k;
                const double d = T[k + (size_t)k * ldt];
                // no-transpose sweeps skip a zero entry like reference dtrsm;
                // its transposed (dot-form) sweeps always divide
                if (trans || *xk != 0.0) *xk = *xk / d;
            }
            __syncthreads();
        }
        // rows still to update: i > k (forward) or i < k (backward)
        const int lo = forward ? k + 1 : 0;
        const int hi = forward ? n : k;
        for (int i = lo + tid; i < hi; i += nthr) {
            // op(T)(i,k): T(i,k) without transpose, T(k,i) with
            const double t = trans ? T[k + (size_t)i * ldt] : T[i + (size_t)k * ldt];
            for (int c = 0; c < nc; ++c) {
                const double xk = X[(size_t)c * ldx + k];
                if (!trans && xk == 0.0) continue;      // reference dtrsm's skip (x_k stays 0 after division)
                X[(size_t)c * ldx + i] = fma(-xk, t, X[(size_t)c * ldx + i]);
            }
        }
        __syncthreads();
    }
}

}  // namespace magma_amd
