// lu_mfma.hip -- LU with partial pivoting, FP64, 64 < max(m, n) <= 512: one
// workgroup per matrix, one thread per row, left-looking by block columns of
// 32 columns.
//
// Rows stay where they are for the whole factorization: a pivot is recorded
// (pos[row], the row's current logical position, and prow[step], the physical
// row of a step's pivot) and one last pass puts every column into LAPACK's row
// order.  Block column p (columns 32 p ..):
//
//   load    C = A(:, block) into registers in the MFMA result layout, wavefront
//           w the 16-row tiles w, w + W, ... (issued before the panel of the
//           block column on its left).
//   update  for each factored chunk q < p: the chunk's pivot rows of C go to
//           LDS, two wavefronts solve U = L_qq^-1 C for 16 columns each in
//           registers (tri_mfma.h), then every wavefront takes C -= L_q U on
//           v_mfma_f64_16x16x4f64 with its tiles of L_q already in flight.
//           Rows that are pivots by then are updated too and never looked at.
//   panel   through LDS into one row per thread.  Per column: the arg-max of
//           the wavefront (DPP on the high words), its row's key in an LDS
//           slot, a barrier, the workgroup's pivot from the slots (DPP again),
//           the pivot row and its reciprocal to LDS, a barrier, and the rank-1
//           update with the pivot row's entries as DPP operands.
//   store   the block column, finished U rows included, in physical row order;
//           past the last pivot (wide matrices) in the final one (2441 of
//           32 x 256 401 -> 279 us, 1041 of 64 x 300 426 -> 343 us).
//
// What bounds it: the chain of a panel column (the search, a barrier and an LDS
// round trip, twice) and, with the chip full, the bytes: 8192 of order 256 move
// 35.3 GB at 4.0 TB/s, a wavefront waits 0.49 of its time and waits to issue
// 0.29, and the matrix cores are 19% busy.  Why
// left-looking with fixed rows: a right-looking form reads and writes the
// trailing matrix per panel, moves 64 scattered rows of it, and needs passes of
// its own for the gather, the U solve and the deferred interchanges of L.  The
// rows that are already pivots cost MFMA work instead (n^3 in place of 2/3
// n^3), which has the room.  Why a group of 16 panel columns per loop pass: 32
// columns unrolled are 70 KB of code, more than the instruction cache.  Why two
// barriers per column: every wavefront's candidate row written before the
// first one kept the LDS busy for 450 cycles a column.
// Measured, getrf alone, right-looking form before: 8192 of order 256 12.85 ms
// -> 8.80 ms, 256 of order 500 7.5 -> 1.96 ms; 4096 of order 96 0.94 ms (a
// register-resident kernel for n <= 128) -> 0.68 ms.
//
// Replaces the reference's launch chain for these sizes (panel + laswp + trsm
// + gemm, src/zgetrf_batched.cpp:222-351, src/zgetrf_panel_batched.cpp:127-243,
// magmablas/zgetf2_kernels.cu:353-760) with one persistent launch.
//
// Rounding: every entry receives its updates as single fused multiply-adds in
// increasing k, in the panel (VALU), the solve and the update: the FP64 MFMA
// applies its four k terms of a slice as the sequential fma chain, slices in
// increasing k.  Multipliers are a * (1/pivot) (division below DBL_MIN), the
// pivot is the first maximum of |a| by logical position with NaN taken only in
// the first position.  So factors and pivots are the bits of netlib dgetrf with
// that update order (up to the sign of a zero).  A block column that ends with
// an entry that is not finite, or meets a pivot below DBL_MIN, is done again from
// memory with the reference loops, and so are the ones after it: only then can
// their skip of a zero U entry, or the rule for NaN, change a result.
#include <cfloat>
#include <climits>
#include <type_traits>

#include "dpp_fma.h"
#include "kernels.h"
#include "pivot_select.h"
#include "tri_mfma.h"
#include "tune.h"

namespace magma_amd {
namespace {

constexpr int PW = 32;              // columns of a block column
constexpr int GW = 16;              // columns of a panel group
constexpr int TPW = 4;              // 16-row tiles per wavefront

typedef double d2 __attribute__((ext_vector_type(2)));
typedef d2 __attribute__((address_space(3))) *LDouble2Ptr;

__device__ __forceinline__ int pick(const int *arr, int fixed, int id) { return arr ? arr[id] : fixed; }

template <int MT>
struct LuSmem {
    double P[PW][MT + 1];     // the block column by physical row; the odd pitch spreads
                              // the solve's reads of one row over the banks
    double U[PW][PW + 1];     // -U of the current chunk, [k][column of the block]
    alignas(16) double row[PW + 2];     // the pivot row of a panel column, then 1 / pivot
    int4 slot[MT / 64];       // each wavefront's candidate
    int pos[MT];              // logical position of a physical row
    int prow[MT];             // physical row of step j's pivot
    int swaps[PW];            // logical positions of the panel's pivots
};

// The panel with the reference loops, on P (all threads): columns [0, nc), the
// first jb factored, skipping zero U entries as reference dger does.
template <int MT>
__device__ __forceinline__ void reference_panel(LuSmem<MT> &sm, int m, int j0, int jb, int nc, int &pos,
                                                int &info)
{
    constexpr int W = MT / 64;
    const int tid = threadIdx.x, w = tid >> 6;
#pragma unroll 1
    for (int jj = 0; jj < jb; ++jj) {
        const int j = j0 + jj;
        const bool cand = tid < m && pos >= j;
        const double v = cand ? sm.P[jj][tid] : 0.0;
        // NaN is the largest in the first position and never taken elsewhere (idamax)
        unsigned long long key = 0;
        if (cand && (v == v || pos == j)) key = pivot_key(v == v ? fabs(v) : __builtin_huge_val());
        const bool top = (key >> 32) != 0;
        int p, pr;
        select_pivot<W>(sm.slot, int4{top ? (int)key : 0, cand ? (top ? (int)(key >> 32) + 1 : 1) : 0, pos, tid}, w, p, pr);
        const double piv = sm.P[jj][pr];
        if (piv == 0.0 && info == 0) info = j + 1;
        if (tid == 0) sm.swaps[jj] = p;
        pos = pos == j ? p : (pos == p ? j : pos);
        if (tid < m && pos > j) {
            double l = v;
            if (piv != 0.0) l = fabs(piv) >= DBL_MIN ? (1.0 / piv) * l : l / piv;
            sm.P[jj][tid] = l;
#pragma unroll 1
            for (int c = jj + 1; c < nc; ++c) {
                const double u = sm.P[c][pr];
                if (u != 0.0) sm.P[c][tid] = fma(l, -u, sm.P[c][tid]);
            }
        }
        __syncthreads();
    }
}

// A block column with the reference loops, from memory to memory (all
// threads): the columns' updates by every earlier pivot, then the panel.
template <int MT>
__device__ __forceinline__ void reference_block(LuSmem<MT> &sm, GDoublePtr A, long lda, int m, int j0, int jb, int nc,
                                                int kn, int &pos, int &info)
{
    const int tid = threadIdx.x;
    if (tid < m) {
#pragma unroll 1
        for (int c = 0; c < nc; ++c) sm.P[c][tid] = A[(j0 + c) * lda + tid];
    }
#pragma unroll 1
    for (int k = 0; k < kn; ++k) {
        __syncthreads();
        if (tid < m && pos > k) {
            const double l = A[k * lda + tid];
            const int pr = sm.prow[k];
#pragma unroll 1
            for (int c = 0; c < nc; ++c) {
                const double u = sm.P[c][pr];
                if (u != 0.0) sm.P[c][tid] = fma(l, -u, sm.P[c][tid]);
            }
        }
    }
    __syncthreads();
    reference_panel<MT>(sm, m, j0, jb, nc, pos, info);
    if (tid < m) {
#pragma unroll 1
        for (int c = 0; c < nc; ++c) A[(j0 + c) * lda + tid] = sm.P[c][tid];
    }
}

template <int K = 0, class F>
__device__ __forceinline__ void steps(F f)
{
    if constexpr (K < GW) {
        f(std::integral_constant<int, K>{});
        steps<K + 1>(f);
    }
}

template <int MT>
__global__ void __launch_bounds__(MT) __attribute__((amdgpu_waves_per_eu(2))) getrf_mfma_kernel(MatSet s)
{
    constexpr int W = MT / 64;
    __shared__ LuSmem<MT> sm;

    int tid = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    int li = tid & 15;
    int lk = (tid >> 4) & 3;
    const int cnt = item_count(s);
    const int *idx = item_index(s);
    for (int item = blockIdx.x; item < cnt; item += gridDim.x) {
        const int id = idx ? idx[item] : item;
        const int m = pick(s.m_arr, s.m, id);
        const int n = pick(s.n_arr, s.n, id);
        const long lda = pick(s.lda_arr, s.lda, id);
        const GDoublePtr A = (GDoublePtr)s.A[id];
        int *ipiv = s.ipiv[id];
        const int mn = min(m, n);
        // no entries, and maybe no memory either.  opaque: as a uniform branch
        // the test costs 60 spilled registers (8192 of order 256, with getrs,
        // 12.19 -> 12.49 ms)
        if (opaque(mn) <= 0) {
            if (tid == 0) s.info[id] = 0;
            continue;
        }
        const int npan = (mn + PW - 1) / PW;        // factored chunks
        const int nblk = (n + PW - 1) / PW;
        int info = 0;
        bool exact = false;                         // a multiplier or U entry was not finite
        int pos = tid;
        __syncthreads();
        sm.pos[tid] = tid;
        __syncthreads();

        // 32 columns from c0, a row per thread
        auto store_rows = [&](int c0, const double (&v)[PW]) {
            GDoublePtr pa = opaque(A + c0 * lda + tid);
            if (tid < m) {
#pragma unroll
                for (int k = 0; k < PW; ++k) {
                    if (c0 + k < n) *pa = v[k];
                    pa += lda;
                }
            }
        };
        // this lane's row of tile b, kept inside the matrix for loads
        int rowc[TPW];
#pragma unroll
        for (int b = 0; b < TPW; ++b) rowc[b] = min(16 * (w + W * b) + li, m - 1);
        auto live = [&](int b) { return 16 * (w + W * b) < m; };
        // C: entry (row, column 16 t + lk + 4 i of the block) in c[b][t][i]
        d4 c[TPW][2];
        auto load_c = [&](int c0) {
            GDoublePtr pc = opaque(A + min(c0 + lk, n - 1) * lda);
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
#pragma unroll
                    for (int b = 0; b < TPW; ++b) c[b][t][i] = pc[rowc[b]];
                    pc += c0 + 16 * t + lk + 4 * i + 4 < n ? 4 * lda : 0;
                    __builtin_amdgcn_sched_barrier(0);
                }
        };
        // the rows of C from logical position `from` on to P
        auto tiles_to_p = [&](int from) {
#pragma unroll
            for (int b = 0; b < TPW; ++b) {
                const int row = 16 * (w + W * b) + li;
                if (row < m && sm.pos[row] >= from) {
#pragma unroll
                    for (int t = 0; t < 2; ++t)
#pragma unroll
                        for (int i = 0; i < 4; ++i) sm.P[16 * t + lk + 4 * i][row] = c[b][t][i];
                }
            }
        };
        load_c(0);

        for (int p = 0; p < nblk; ++p) {
            tid = opaque(tid);
            const int j0 = PW * p;
            const int jb = min(PW, max(0, mn - j0));
            const int nc = min(PW, n - j0);
            const int qn = min(p, npan);
            bool bad = exact;

            // ------------------------------------------------ update -------
            // L_q: entry (row, k = 4 s + lk) in lb[b][s]; the 16 x 16 tiles of
            // L_qq in pivot order for the wavefronts that solve
            double lb[TPW][PW / 4];
            d4 t00, t10, t11;
            auto load_l = [&](int q, int b0) {
                GDoublePtr pl = opaque(A + (PW * q + lk) * lda);
#pragma unroll
                for (int k = 0; k < PW / 4; ++k) {
#pragma unroll
                    for (int b = b0; b < b0 + 2; ++b) lb[b][k] = pl[rowc[b]];
                    pl += 4 * lda;
                }
            };
            auto load_t = [&](int q) {
                const int kb = min(PW, mn - PW * q);
                const int r0 = sm.prow[PW * q + min(li, kb - 1)], r1 = sm.prow[PW * q + min(16 + li, kb - 1)];
                const GDoublePtr pt = opaque(A + PW * q * lda);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int k = 4 * i + lk;
                    const GDoublePtr p0 = pt + min(k, kb - 1) * lda;
                    const GDoublePtr p1 = pt + min(16 + k, kb - 1) * lda;
                    const double v0 = p0[r0], v1 = p0[r1], v2 = p1[r1];
                    t00[i] = max(li, k) < kb ? v0 : 0.0;
                    t10[i] = max(16 + li, k) < kb ? v1 : 0.0;
                    t11[i] = 16 + max(li, k) < kb ? v2 : 0.0;
                }
            };
            if (qn > 0) {
                if (w < 2) load_t(0);
                load_l(0, 0);
            }
#pragma unroll 1
            for (int q = 0; q < qn; ++q) {
                const int kb = min(PW, mn - PW * q);
                li = opaque(li);
                lk = opaque(lk);
                // the chunk's pivot rows to P
#pragma unroll
                for (int b = 0; b < TPW; ++b) {
                    const int row = 16 * (w + W * b) + li;
                    if (row < m && (sm.pos[row] >> 5) == q) {
#pragma unroll
                        for (int t = 0; t < 2; ++t)
#pragma unroll
                            for (int i = 0; i < 4; ++i) sm.P[16 * t + lk + 4 * i][row] = c[b][t][i];
                    }
                }
                __syncthreads();
                if (w < 2) {
                    // lane (lk, li): rows 4 i + lk (x0) and 16 + 4 i + lk (x1) of column 16 w + li
                    const double *col = sm.P[16 * w + li];
                    int r0[4], r1[4];
                    d4 x0, x1;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        r0[i] = sm.prow[PW * q + min(4 * i + lk, kb - 1)];
                        r1[i] = sm.prow[PW * q + min(16 + 4 * i + lk, kb - 1)];
                    }
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        x0[i] = 4 * i + lk < kb ? col[r0[i]] : 0.0;
                        x1[i] = 16 + 4 * i + lk < kb ? col[r1[i]] : 0.0;
                    }
                    tri_detail::diag_solve<kTriUnit>(x0, t00, li, lk);
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        x1 = __builtin_amdgcn_mfma_f64_16x16x4f64(t10[i], -x0[i], x1, 0, 0, 0);
                    tri_detail::diag_solve<kTriUnit>(x1, t11, li, lk);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        bad |= !__builtin_isfinite(x0[i]) || !__builtin_isfinite(x1[i]);
                        sm.U[4 * i + lk][16 * w + li] = -x0[i];
                        sm.U[16 + 4 * i + lk][16 * w + li] = -x1[i];
                        if (4 * i + lk < kb) sm.P[16 * w + li][r0[i]] = x0[i];
                        if (16 + 4 * i + lk < kb) sm.P[16 * w + li][r1[i]] = x1[i];
                    }
                    if (q + 1 < qn) load_t(q + 1);
                }
                __syncthreads();
                // a chunk that ends the rows leaves nothing to update
                if (PW * q + PW < m) {
                    load_l(q, 2);
                    double ua[2][PW / 4];
#pragma unroll
                    for (int t = 0; t < 2; ++t)
#pragma unroll
                        for (int k = 0; k < PW / 4; ++k) ua[t][k] = sm.U[4 * k + lk][16 * t + li];
#pragma unroll
                    for (int b = 0; b < TPW; b += 2) {
                        if (live(b)) {
#pragma unroll
                            for (int k = 0; k < PW / 4; ++k)
#pragma unroll
                                for (int d = 0; d < 2; ++d)
#pragma unroll
                                    for (int t = 0; t < 2; ++t)
                                        c[b + d][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(ua[t][k], lb[b + d][k],
                                                                                           c[b + d][t], 0, 0, 0);
                        }
                        if (b == 0 && q + 1 < qn) load_l(q + 1, 0);
                    }
                }
            }

            // ------------------------------------------------ panel --------
            // rows that are no pivots yet to P, then a row per thread
            li = opaque(li);
            lk = opaque(lk);
            tiles_to_p(PW * qn);
            __syncthreads();
            double a[PW];
#pragma unroll
            for (int k = 0; k < PW; ++k) a[k] = sm.P[k][tid];
            if (p + 1 < nblk) load_c(j0 + PW);
            tid = opaque(tid);
            const int pos0 = pos, info0 = info;
            double z = 0.0;                         // NaN when an entry of this row is not finite
            // GW columns at a time; the rest of the row then moves down to the
            // front registers, so that the loop's code stays in the
            // instruction cache (32 columns unrolled: 40 KB)
#pragma unroll 1
            for (int g = 0; g < PW; g += GW) {
                auto step = [&](auto JJ) {
                    constexpr int jj = JJ;
                    if (g + jj >= jb) return;
                    const int j = j0 + g + jj;
                    const double v = a[jj];
                    const bool cand = tid < m && pos >= j;
                    double rv = 1.0 / v;                // beside the search; the pivot's is used
                    asm volatile("" : "+v"(rv));
                    // a NaN ends in the finite test below
                    const long long av = __double_as_longlong(fabs(v));
                    int pp, pr;
                    select_pivot<W>(sm.slot, int4{(int)av, cand ? (int)(av >> 32) + 1 : 0, pos, tid}, w, pp, pr);
                    // Above 128 rows the array lies past what an offset from 0
                    // reaches, and 18 addresses were kept in registers: one address
                    // and offsets (256 of order 500, 7 rhs: 2.45 -> 2.42 ms).
                    constexpr bool far = offsetof(LuSmem<MT>, row) + sizeof(double) * (PW + 2) > 65536;
                    const LDoublePtr row = far ? opaque((LDoublePtr)sm.row) : (LDoublePtr)sm.row;
                    if (tid == pr) {
#pragma unroll
                        for (int k = jj & ~1; k < PW; k += 2) *(LDouble2Ptr)(row + k) = d2{a[k], a[k + 1]};
                        row[PW] = rv;
                        sm.swaps[g + jj] = pp;
                    }
                    __syncthreads();
                    const double piv = row[jj], rc = row[PW];
                    double nu0 = -row[tid & 15], nu1 = -row[16 + (tid & 15)];
                    asm volatile("" : "+v"(nu0), "+v"(nu1));     // both reads here, not one in the branch below
                    if (piv == 0.0 && info == 0) info = j + 1;
                    bad |= piv != 0.0 && !(fabs(piv) >= DBL_MIN);
                    pos = (pos == j) ? pp : ((pos == pp) ? j : pos);
                    const bool below = tid < m && pos > j;
                    double l = piv != 0.0 ? rc * v : v;
                    a[jj] = below ? l : v;
                    l = below ? l : 0.0;                // adds a zero where U is finite
                    fmac_row<jj + 1, PW - GW>(a, nu0, nu1, l);
                    if (g < GW) fmac_row<PW - GW, PW>(a, nu0, nu1, l);
                };
                steps<0>(step);
#pragma unroll
                for (int k = 0; k < GW; ++k) {
                    z = fma(a[k], 0.0, z);
                    sm.P[g + k][tid] = a[k];
                }
#pragma unroll
                for (int k = 0; k + GW < PW; ++k) a[k] = a[k + GW];
            }
            bad |= tid < m && !(z == 0.0);
            if (__syncthreads_or(bad)) {
                // the block column is still in A as it was
                exact = true;
                pos = pos0;
                info = info0;
                reference_block<MT>(sm, A, lda, m, j0, jb, nc, min(j0, mn), pos, info);
            }
            // Past the last pivot (m < n) every row's place is known, and the block
            // column goes there at once.
            if (!exact || jb == 0) {
                const int from = jb > 0 ? tid : sm.prow[min(tid, m - 1)];
#pragma unroll
                for (int k = 0; k < PW; ++k) a[k] = sm.P[k][from];
                store_rows(j0, a);
            }
            if (jb > 0) {
                sm.pos[tid] = pos;
                if (tid < m && pos >= j0 && pos < j0 + jb) sm.prow[pos] = tid;
                if (tid < jb) ipiv[j0 + tid] = sm.swaps[tid] + 1;
            }
            __syncthreads();
        }

        // LAPACK's row order: every other column once through P
        double a[PW];
        auto load_rows = [&](int c0) {
            GDoublePtr pa = opaque(A + c0 * lda + min(tid, m - 1));
#pragma unroll
            for (int k = 0; k < PW; ++k) {
                a[k] = *pa;
                pa += c0 + k + 1 < n ? lda : 0;
            }
        };
        load_rows(0);
#pragma unroll 1
        for (int p = 0; p < npan; ++p) {
            const int c0 = PW * p;
            if (tid < m) {
#pragma unroll
                for (int k = 0; k < PW; ++k) sm.P[k][pos] = a[k];
            }
            __syncthreads();
            if (p + 1 < npan) load_rows(c0 + PW);
            double o[PW];
#pragma unroll
            for (int k = 0; k < PW; ++k) o[k] = sm.P[k][tid];
            store_rows(c0, o);
            __syncthreads();
        }
        if (tid == 0) s.info[id] = info;
    }
}

}  // namespace

template <class K>
static int resident_per_cu(K kernel, int threads)
{
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kernel, threads, 0) != hipSuccess || nb < 1) nb = 1;
    return nb;
}

template <int MT>
static magma_int_t launch_mt(const MatSet &s, int variant, hipStream_t st)
{
    const int grid = persistent_grid(s.count, variant == 1 ? 1 : resident_per_cu(getrf_mfma_kernel<MT>, MT));
    getrf_mfma_kernel<MT><<<grid, MT, 0, st>>>(s);
    MAGMA_LAUNCH_CHECK();
    return MAGMA_SUCCESS;
}

// 64 < max_dim <= 512 (the largest m or n); returns MAGMA_ERR_NOT_SUPPORTED
// above.  The kernel goes by the rows, which are what a workgroup's threads and
// LDS hold; by the larger side, wide matrices left most of both idle (us:
// 100 x 512 x 390 1003 -> 519, 64 x 300 x 1041 981 -> 343).
magma_int_t launch_getrf_mfma(const MatSet &s, int max_dim, int max_m, hipStream_t st)
{
    if (s.count <= 0) return MAGMA_SUCCESS;
    if (max_dim > 512) return MAGMA_ERR_NOT_SUPPORTED;
    const int v = tuned_variant(kTuneGetrf, size_class_of(max_dim));
    if (max_m <= 128) return launch_mt<128>(s, v, st);
    if (max_m <= 256) return launch_mt<256>(s, v, st);
    return launch_mt<512>(s, v, st);
}

}  // namespace magma_amd
