// pivot_select.h -- the pivot of a panel column over a workgroup's threads.
#pragma once

#include "kernels.h"
#include "wave_reduce.h"

namespace magma_amd {

// A candidate is an int4: the low and high word of its key, its logical
// position, its physical row.  The larger key wins, ties go to the smaller
// logical position; high word 0 marks a row that is no candidate.
__device__ __forceinline__ bool pivot_before(const int4 &a, const int4 &b)
{
    if (a.y != b.y) return (unsigned)a.y > (unsigned)b.y;
    if (a.x != b.x) return (unsigned)a.x > (unsigned)b.x;
    return a.z < b.z;
}

// The workgroup's pivot from each thread's candidate: logical position p and
// physical row pr.  The high words decide it but for ties, which take the
// longer comparison.  Two barriers with the caller's next one: slot is read
// after the first and written again after the second.
template <int W>
__device__ __forceinline__ void select_pivot(int4 *slot, int4 cand, int w, int &p, int &pr)
{
    const int lane = threadIdx.x & 63;
    const unsigned hk = cand.y;
    const unsigned mh = wave_max_u32(hk);
    bool win = hk == mh;
    if (mh == 0) {
        win = lane == 0;
    } else if (__builtin_expect(__builtin_popcountll(__builtin_amdgcn_ballot_w64(win)) != 1, 0)) {
        const unsigned ml = wave_max_u32(win ? cand.x : 0);
        win &= (unsigned)cand.x == ml;
        win &= cand.z == wave_min_i32(win ? cand.z : INT_MAX);
    }
    if (win) slot[w] = cand;
    __syncthreads();
    const int4 h = slot[lane & (W - 1)];
    unsigned m = h.y;
    m = max(m, (unsigned)__builtin_amdgcn_update_dpp(0, (int)m, 0xB1, 0xF, 0xF, false));                // xor 1
    if (W > 2) m = max(m, (unsigned)__builtin_amdgcn_update_dpp(0, (int)m, 0x4E, 0xF, 0xF, false));     // xor 2
    if (W > 4) m = max(m, (unsigned)__builtin_amdgcn_update_dpp(0, (int)m, 0x141, 0xF, 0xF, false));    // half-row mirror
    const unsigned tie = (unsigned)__builtin_amdgcn_ballot_w64((unsigned)h.y == m) & ((1u << W) - 1);
    int src = __builtin_ctz(tie);
    if (__builtin_expect((tie & (tie - 1)) != 0, 0)) {
        int4 best = slot[src];
#pragma unroll 1
        for (int q = src + 1; q < W; ++q) {
            const int4 o = slot[q];
            if (pivot_before(o, best)) {
                best = o;
                src = q;
            }
        }
        src = __builtin_amdgcn_readfirstlane(src);
    }
    p = __builtin_amdgcn_readlane(h.z, src);
    pr = __builtin_amdgcn_readlane(h.w, src);
}

}  // namespace magma_amd
