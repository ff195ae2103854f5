// A workgroup of 64-lane wavefronts on the CPU, for kernels' device code built
// by the host compiler: every thread is a fiber that runs until it meets a
// cross-lane operation or a barrier.  Control flow around those has to be
// uniform over a wavefront (or the workgroup), as the kernels have it.  Buffer
// loads check the whole offset against the descriptor; other accesses are
// checked by what surrounds the operands (guard()).
#pragma once

#include <sys/mman.h>
#include <ucontext.h>

#include <bit>
#include <climits>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <vector>

#define __HIPCC__ 1
#define __device__
#define __global__
#define __shared__ static
#define __forceinline__ inline
#define __launch_bounds__(...)
#define amdgpu_waves_per_eu(...) unused

typedef int hipError_t;
typedef struct ihipStream_t *hipStream_t;
constexpr int hipSuccess = 0;
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }

using std::max;
using std::min;
struct int4 { int x, y, z, w; };
struct double2 { double x, y; };
inline double2 make_double2(double x, double y) { return {x, y}; }
inline long long __double_as_longlong(double x) { return std::bit_cast<long long>(x); }
inline double __longlong_as_double(long long x) { return std::bit_cast<double>(x); }
inline int __float_as_int(float x) { return std::bit_cast<int>(x); }

namespace emu {

struct Fiber {
    ucontext_t ctx;
    std::vector<char> stack;
    bool done;
};
struct Slot { alignas(16) char b[32]; };

inline std::vector<Fiber> fibers;
inline ucontext_t scheduler;
inline std::function<void()> body;
inline unsigned cur, threads;
inline long moves, outside;             // progress; buffer loads past the descriptor
struct Wave { long gen = 0; int arrived = 0; Slot slot[2][64]; };
inline std::vector<Wave> waves;
inline long block_gen;
inline unsigned block_arrived, block_or[2];

inline void yield() { swapcontext(&fibers[cur].ctx, &scheduler); }

// the wavefront's values of v, one a lane
template <class T>
const Slot *exchange(T v)
{
    static_assert(sizeof(T) <= sizeof(Slot));
    Wave &w = waves[cur / 64];
    const long g = w.gen;
    Slot *s = w.slot[g & 1];
    std::memcpy(s[cur & 63].b, &v, sizeof(T));
    ++moves;
    if (++w.arrived == 64) {
        w.arrived = 0;
        ++w.gen;
    }
    while (w.gen == g) yield();
    return s;
}
template <class T>
T lane(const Slot *s, int l)
{
    T v;
    std::memcpy(&v, s[l & 63].b, sizeof(T));
    return v;
}

inline bool barrier(bool x)
{
    const long g = block_gen;
    if (block_arrived == 0) block_or[g & 1] = 0;
    block_or[g & 1] |= x;
    ++moves;
    if (++block_arrived == threads) {
        block_arrived = 0;
        ++block_gen;
    }
    while (block_gen == g) yield();
    return block_or[g & 1] != 0;
}

inline void enter()
{
    body();
    fibers[cur].done = true;
    ++moves;
    yield();
}

// one workgroup of nthr threads
inline void run(unsigned nthr, std::function<void()> f)
{
    body = f;
    threads = nthr;
    waves.assign(nthr / 64, Wave());
    fibers.resize(nthr);
    block_arrived = 0;
    for (Fiber &t : fibers) {
        t.stack.resize(1 << 17);
        t.done = false;
        getcontext(&t.ctx);
        t.ctx.uc_stack.ss_sp = t.stack.data();
        t.ctx.uc_stack.ss_size = t.stack.size();
        t.ctx.uc_link = nullptr;
        makecontext(&t.ctx, enter, 0);
    }
    for (bool live = true; live;) {
        live = false;
        const long before = moves;
        for (cur = 0; cur < nthr; ++cur)
            if (!fibers[cur].done) {
                live = true;
                swapcontext(&scheduler, &fibers[cur].ctx);
            }
        if (live && moves == before) {
            std::puts("a cross-lane operation or barrier that not every thread reaches");
            std::exit(1);
        }
    }
}

// Memory for n doubles that ends at (or, front, begins after) an inaccessible page.
inline double *guard(size_t n, bool front)
{
    const size_t page = 4096, bytes = n * sizeof(double), body_bytes = (bytes + page - 1) / page * page;
    char *p = (char *)mmap(nullptr, body_bytes + 2 * page, PROT_NONE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
    if (p == MAP_FAILED || mprotect(p + page, body_bytes, PROT_READ | PROT_WRITE) != 0) std::abort();
    return (double *)(p + page + (front ? 0 : body_bytes - bytes));
}

struct Index {
    unsigned x;
};

// lanes that a DPP control word reads, -1: none (the old value stays)
inline int dpp_source(int ctrl, int l)
{
    const int row = l & ~15, i = l & 15;
    if (ctrl < 0x100) return (l & ~3) | ((ctrl >> (2 * (l & 3))) & 3);         // quad_perm
    if (ctrl >= 0x111 && ctrl <= 0x11F) return i - (ctrl & 15) >= 0 ? l - (ctrl & 15) : -1;     // row_shr
    if (ctrl == 0x140) return row + 15 - i;                                     // row_mirror
    if (ctrl == 0x141) return (l & ~7) + 7 - (l & 7);                           // row_half_mirror
    if (ctrl >= 0x150 && ctrl <= 0x15F) return row + (ctrl & 15);               // row_newbcast
    std::abort();
}

inline int update_dpp(int old, int v, int ctrl)
{
    const Slot *s = exchange(v);
    const int from = dpp_source(ctrl, cur & 63);
    return from < 0 ? old : lane<int>(s, from);
}

inline unsigned long long ballot(bool x)
{
    const Slot *s = exchange(x);
    unsigned long long m = 0;
    for (int l = 0; l < 64; ++l) m |= (unsigned long long)lane<bool>(s, l) << l;
    return m;
}

struct Pair {
    unsigned v[2];
    unsigned operator[](int i) const { return v[i]; }
};

// the odd rows (of 16, or 32, lanes) of a against the even rows of b
inline Pair permlane_swap(unsigned a, unsigned b, int rows)
{
    const Slot *s = exchange(Pair{{a, b}});
    const int l = cur & 63;
    const bool odd = (l / rows) & 1;
    return {{odd ? lane<Pair>(s, l - rows).v[1] : a, odd ? b : lane<Pair>(s, l + rows).v[0]}};
}

typedef double d4 __attribute__((ext_vector_type(4)));

inline d4 mfma_f64(double a, double b, d4 c)
{
    const Slot *s = exchange(double2{a, b});
    const int l = cur & 63, col = l & 15;
    for (int i = 0; i < 4; ++i)
        for (int k = 0; k < 4; ++k)
            c[i] = std::fma(lane<double2>(s, 16 * k + l / 16 + 4 * i).x, lane<double2>(s, 16 * k + col).y, c[i]);
    return c;
}

struct Buffer {
    const char *p;
    int bytes;
};

inline double buffer_load(Buffer r, int lane_off, int off)
{
    const long at = (long)lane_off + off;
    if (at < 0 || at + 8 > r.bytes) {
        ++outside;
        return std::nan("");
    }
    double v;
    std::memcpy(&v, r.p + at, 8);
    return v;
}

}  // namespace emu

#define threadIdx (emu::Index{emu::cur})
#define blockDim (emu::Index{emu::threads})
#define blockIdx (emu::Index{0})
#define gridDim (emu::Index{1})
#define __syncthreads() ((void)emu::barrier(false))
#define __syncthreads_or(x) (emu::barrier(x))
#define __builtin_amdgcn_readlane(v, l) (emu::lane<int>(emu::exchange((int)(v)), l))
#define __builtin_amdgcn_readfirstlane(v) (emu::lane<int>(emu::exchange((int)(v)), 0))
#define __builtin_amdgcn_update_dpp(old, v, ctrl, rows, banks, bound) (emu::update_dpp(old, v, ctrl))
#define __builtin_amdgcn_ballot_w64(x) (emu::ballot(x))
#define __builtin_amdgcn_permlane16_swap(a, b, f, c) (emu::permlane_swap(a, b, 16))
#define __builtin_amdgcn_permlane32_swap(a, b, f, c) (emu::permlane_swap(a, b, 32))
#define __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, x, y, z) (emu::mfma_f64(a, b, c))
#define __builtin_amdgcn_make_buffer_rsrc(p, stride, n, flags) (emu::Buffer{(const char *)(p), n})
#define __builtin_amdgcn_raw_buffer_load_b64(r, v, s, aux) (emu::buffer_load(r, v, s))
#define __builtin_amdgcn_sched_barrier(x) ((void)0)
