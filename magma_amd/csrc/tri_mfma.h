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
// 16 columns.  A 16 x 16 diagonal block is solved four rows at a time: permlane
// swaps give every lane its vector's four rows, each lane solves the 4 x 4
// triangle with the factor's entries as scalars, and one MFMA takes the four
// rows out of the rest of the block.
//
// Why: a sweep with one barrier per column (one row per thread, X in LDS)
// costs a barrier and an LDS round trip per column and right-hand-side pass,
// and reads the factor once per 8 right-hand sides; here the chain of a column
// is in registers, the factor's tiles for the next block column are in flight
// while a diagonal block is solved, and 16 right-hand sides share one read.
//
// Rounding: an entry gets its terms as single fmas in the order of the solved
// rows (the MFMA applies its four k terms as the sequential chain), then the
// division: the reference BLAS order of the forward cases, and its bits up to
// the sign of a zero: the reference skips a zero x_k, which keeps its sign, and
// here it is divided and updated like any other (the inverse of -I has -0 off
// its diagonal).  Beyond that the skip (or that of a zero factor entry) can
// change a result only where the other operand is not finite, and then the
// result here is not finite either: callers test that and redo such a matrix
// with the reference loops.
#pragma once

#include "dpp_fma.h"
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

// the values of x in the four row groups (lanes 16 g .. 16 g + 15), each in all lanes
__device__ __forceinline__ void group_values(double x, double (&y)[4])
{
    const long long b = __double_as_longlong(x);
    unsigned r[2] = {(unsigned)b, (unsigned)(b >> 32)}, z[4][2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        // [x0 x0 x2 x2] and [x1 x1 x3 x3], then each half twice
        const auto p = __builtin_amdgcn_permlane16_swap(r[h], r[h], false, false);
        const auto e = __builtin_amdgcn_permlane32_swap(p[0], p[0], false, false);
        const auto o = __builtin_amdgcn_permlane32_swap(p[1], p[1], false, false);
        z[0][h] = e[0];
        z[1][h] = o[0];
        z[2][h] = e[1];
        z[3][h] = o[1];
    }
#pragma unroll
    for (int g = 0; g < 4; ++g) y[g] = __longlong_as_double(((long long)z[g][1] << 32) | z[g][0]);
}

__device__ __forceinline__ double lane_value(double x, int lane)
{
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_readlane((int)b, lane), hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// Rows 4 S .. 4 S + 3 of the 16 x 16 diagonal block whose A-operand tile is t
// (t[i] holds entry (li, 4 i + lk)): every lane solves the 4 x 4 triangle for
// its vector, then one MFMA takes the four rows out of the rows below.
template <int S, TriDiag DIAG>
__device__ __forceinline__ void diag_slice(d4 &x, const d4 &t, int li, int lk)
{
    double y[4];
    group_values(x[S], y);
    auto entry = [&](int r, int c) { return lane_value(t[S], 16 * c + 4 * S + r); };
#pragma unroll
    for (int r = 0; r < 4; ++r) {
#pragma unroll
        for (int c = 0; c < r; ++c) y[r] = fma(-y[c], entry(r, c), y[r]);
        if constexpr (DIAG == kTriDivide) y[r] = y[r] / entry(r, r);
        if constexpr (DIAG == kTriReciprocal) y[r] = (1.0 / entry(r, r)) * y[r];
    }
    const double lo = (lk & 1) ? y[1] : y[0], hi = (lk & 1) ? y[3] : y[2];
    const double own = (lk & 2) ? hi : lo;
    if constexpr (S < 3) {
        const double a = li > 4 * S + 3 ? t[S] : 0.0;
        x = __builtin_amdgcn_mfma_f64_16x16x4f64(a, -own, x, 0, 0, 0);
    }
    x[S] = own;
}

template <TriDiag DIAG>
__device__ __forceinline__ void diag_solve(d4 &x, const d4 &t, int li, int lk)
{
    diag_slice<0, DIAG>(x, t, li, lk);
    __builtin_amdgcn_sched_barrier(0);          // one slice's scalars at a time in registers
    diag_slice<1, DIAG>(x, t, li, lk);
    __builtin_amdgcn_sched_barrier(0);
    diag_slice<2, DIAG>(x, t, li, lk);
    __builtin_amdgcn_sched_barrier(0);
    diag_slice<3, DIAG>(x, t, li, lk);
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
    auto ld = [&](int lane_off, int off) {
        return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rs, lane_off, off, 0));
    };
    auto at = [&](int t) { return 16 * (rev ? nt - 1 - t : t); };           // first matrix row of block t
    auto xrow = [&](int s, int li) { return (rev ? 16 * nt - 1 - s : s) * kTriPitch + li; };
    // Block eb (-1: none) holds the matrix's last rows and rows past n.  Its tiles
    // repeat row and column n - 1 there, so that every load stays inside the
    // matrix (the resource's range check does not cover the scalar offset); what
    // the repeats bring is cleared or masked where it is used.
    const int last = n - 1 - 16 * (nt - 1), eb = last == 15 ? -1 : rev ? 0 : nt - 1;
    const int tile_e = min(li, last) * ds + lk * dk;        // rows of eb, forward
    // factor tile below the diagonal: A operand of slice i, entry (row li, column 4 i + lk)
    auto load_tile = [&](int tr, int tc, d4 &a) {
        const int lane_off = tr == eb ? tile_e : tile;
#pragma unroll
        for (int i = 0; i < 4; ++i) a[i] = ld(lane_off, at(tr) * ds + (at(tc) + 4 * (rev ? 3 - i : i)) * dk);
    };
    // the same where the tile's columns are those of eb
    auto load_edge = [&](int tr, d4 &a) {
        const int l = opaque(lane);
        const int r = rev ? 15 - (l & 15) : l & 15, k = rev ? 15 - (l >> 4) : l >> 4;
        const int row = (tr == eb ? min(r, last) : r) * ds;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            a[i] = ld(row + min(rev ? k - 4 * i : k + 4 * i, last) * dk, at(tr) * ds + at(eb) * dk);
    };
    auto load_diag = [&](int t, d4 &a) {
        if (t == eb) load_edge(t, a);
        else load_tile(t, t, a);
    };
    d4 x[NB], av[NB], dt;
    load_diag(min(w, nt - 1), dt);
    // With one wavefront the LDS addresses are formed where they are used: kept
    // from block to block they spilled up to 25 of the 128 registers (20,000 of
    // order 64: getri 818 -> 776 us, trsm with 16 vectors 256 -> 252 us).
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const int ln = W == 1 ? opaque(lane) : lane, li = ln & 15, lk = ln >> 4;
        const int t = w + W * b;
        x[b] = d4{0.0, 0.0, 0.0, 0.0};
        av[b] = x[b];
        if (t < nt) {
            if (t > 0) {
                if (eb == 0) load_edge(t, av[b]);
                else load_tile(t, 0, av[b]);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int s = 16 * t + 4 * i + lk;
                if (rev ? s >= pad : s < n) x[b][i] = X[xrow(s, li)];
            }
        }
    }
    if (pad > 0) {
        // rows past n come first: no coupling, unit diagonal
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int s = 4 * i + lk;
            if (w == 0 && (s < pad || li < pad)) dt[i] = s == li ? 1.0 : 0.0;      // (li, s)
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
            const int ln = W == 1 ? opaque(lane) : lane, li = ln & 15, lk = ln >> 4;
            if (W == 1 || w == ww) {
                // Rows past n come last in a forward sweep: no coupling and a unit
                // diagonal there too, and zeros in x, since what the updates left
                // would reach the rows above through the block's MFMAs if it is
                // not finite (0 times Inf).
                const bool edge = !rev && t == eb;
                if (edge) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int k = 4 * i + lk;
                        if (16 * t + max(k, li) >= n) dt[i] = k == li ? 1.0 : 0.0;
                    }
                }
                if (W == 1 || edge) {           // in a branch it costs one wavefront spills
                    const int lim = rev ? 16 * nt : n;
#pragma unroll
                    for (int i = 0; i < 4; ++i) x[0][i] = 16 * t + 4 * i + lk < lim ? x[0][i] : 0.0;
                }
                diag_solve<DIAG>(x[0], dt, li, lk);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int s = 16 * t + 4 * i + lk;
                    if (rev ? s >= pad : s < n) X[xrow(s, li)] = x[0][i];
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
                    xb[i] = s >= pad ? -X[xrow(s, li)] : 0.0;
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
