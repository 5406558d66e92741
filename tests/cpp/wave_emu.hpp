// wave_emu.hpp -- runs the source of a HIP kernel on the CPU, one workgroup at
// a time: a fiber per thread, wavefronts of 64 whose cross-lane operations are
// rendezvous of their lanes, and __syncthreads() a rendezvous of the workgroup.
// Between two of these the wavefronts' order is free, and `policy` chooses it:
// one that is right on the device under every order must be right here under
// each.  Inside a wavefront the highest lane goes first, so that what lane 0
// stores is seen by no lane of its own wavefront early (they run in lockstep on
// the device).
//
// The kernel's text is included after this header with `__shared__` objects made
// static and `extern __shared__ T x[]` turned into pointers to dynamic_lds.
#pragma once

#include <setjmp.h>
#include <ucontext.h>

#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <functional>
#include <random>
#include <vector>

namespace wave_emu
{

enum policy : int {
    kFirstAhead, // wavefront 0 runs as far as it can, then 1, ...
    kLastAhead,  // the last one first
    kShuffled    // a random order after every rendezvous
};

struct dim3_ {
    uint32_t x = 0, y = 0, z = 0;
};

enum state : int { kReady, kAtWave, kAtBlock, kDone };

// (ucontext starts a fiber; the switches after that are jumps, without system calls)
struct fiber {
    ucontext_t ctx;
    jmp_buf at;
    bool started = false;
    state st = kReady;
    uint32_t tid = 0, ops = 0;
    std::vector<char> stack;
};

struct block {
    uint32_t threads = 0;
    std::vector<fiber> f;
    std::vector<uint64_t> val[2]; // a lane's operand, by the parity of its operation
    jmp_buf main;
    uint32_t cur = 0;
    std::function<void()> body;
};

inline block *g = nullptr;
inline dim3_ block_idx, block_dim, grid_dim;
alignas(16) inline unsigned char dynamic_lds[163840];

struct thread_index {
    struct lane_x {
        operator uint32_t() const
        {
            return g->cur;
        }
    } x;
};
inline thread_index thread_idx;

inline void entry()
{
    g->body();
    g->f[g->cur].st = kDone;
    _longjmp(g->main, 1);
}

inline void wait(state s)
{
    fiber &me = g->f[g->cur];
    me.st = s;
    if (_setjmp(me.at) == 0) _longjmp(g->main, 1);
}

__attribute__((noinline)) inline void resume(uint32_t tid)
{
    fiber &x = g->f[tid];
    g->cur = tid;
    if (_setjmp(g->main) != 0) return;
    if (x.started) _longjmp(x.at, 1);
    x.started = true;
    setcontext(&x.ctx);
}

// Deposits v and waits for the wavefront's 64 lanes; afterwards operand(lane).
struct wave_op {
    uint32_t par, first;
    explicit wave_op(uint64_t v)
    {
        fiber &me = g->f[g->cur];
        par = me.ops++ & 1u;
        first = g->cur & ~63u;
        g->val[par][g->cur] = v;
        wait(kAtWave);
    }
    uint64_t operand(uint32_t lane) const
    {
        return g->val[par][first + lane];
    }
};

inline void fatal(const char *what)
{
    std::printf("emulator: %s\n", what);
    std::exit(3);
}

// One workgroup of `threads` threads runs body().
inline void run(uint32_t threads, int how, uint32_t seed, std::function<void()> body)
{
    static block b;
    g = &b;
    b.threads = threads;
    b.body = std::move(body);
    if (b.f.size() < threads) b.f.resize(threads);
    for (auto &v : b.val) v.assign(threads, 0u);
    block_dim.x = threads;
    for (uint32_t t = 0; t < threads; ++t) {
        fiber &x = b.f[t];
        if (x.stack.empty()) x.stack.resize(65536u);
        x.st = kReady;
        x.started = false;
        x.tid = t;
        x.ops = 0u;
        getcontext(&x.ctx);
        x.ctx.uc_stack.ss_sp = x.stack.data();
        x.ctx.uc_stack.ss_size = x.stack.size();
        x.ctx.uc_link = nullptr;
        makecontext(&x.ctx, entry, 0);
    }
    std::mt19937 rng(seed);
    const uint32_t waves = threads / 64u;
    std::vector<uint32_t> order(waves);
    for (uint32_t w = 0; w < waves; ++w) order[w] = how == kLastAhead ? waves - 1u - w : w;
    for (;;) {
        if (how == kShuffled) std::shuffle(order.begin(), order.end(), rng);
        uint32_t at_block = 0u, done = 0u;
        for (uint32_t w : order) {
            // this wavefront as far as it can go
            for (;;) {
                uint32_t here[4] = {0u, 0u, 0u, 0u};
                for (uint32_t l = 64u; l-- > 0u;) {
                    fiber &x = b.f[64u * w + l];
                    if (x.st == kReady) resume(64u * w + l);
                    ++here[x.st];
                }
                if (here[kAtWave] == 0u) {
                    at_block += here[kAtBlock];
                    done += here[kDone];
                    break;
                }
                if (here[kAtWave] != 64u) fatal("a cross-lane operation that not every lane reaches");
                for (uint32_t l = 0; l < 64u; ++l) b.f[64u * w + l].st = kReady;
            }
        }
        if (done == threads) return;
        if (at_block + done != threads) fatal("no thread can go on");
        for (uint32_t t = 0; t < threads; ++t) {
            if (b.f[t].st == kAtBlock) b.f[t].st = kReady;
        }
    }
}

} // namespace wave_emu

// ---- the names that a kernel uses -------------------------------------------------
#define __global__
#define __device__
#define __host__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __align__(n) alignas(n)
#define threadIdx wave_emu::thread_idx
#define blockIdx wave_emu::block_idx
#define blockDim wave_emu::block_dim
#define gridDim wave_emu::grid_dim

using std::max;
using std::min;

struct uint2 {
    uint32_t x, y;
};
inline uint2 make_uint2(uint32_t x, uint32_t y)
{
    return {x, y};
}

inline void __syncthreads()
{
    wave_emu::wait(wave_emu::kAtBlock);
}
inline uint64_t __ballot(bool p)
{
    const wave_emu::wave_op op(p ? 1u : 0u);
    uint64_t r = 0u;
    for (uint32_t l = 0; l < 64u; ++l) r |= op.operand(l) << l;
    return r;
}
inline uint32_t __shfl_up(uint32_t v, uint32_t d)
{
    const uint32_t lane = wave_emu::g->cur & 63u;
    const wave_emu::wave_op op(v);
    return static_cast<uint32_t>(op.operand(lane >= d ? lane - d : lane));
}
inline uint32_t __builtin_amdgcn_readlane(uint32_t v, uint32_t from)
{
    return static_cast<uint32_t>(wave_emu::wave_op(v).operand(from & 63u));
}
inline uint32_t __builtin_amdgcn_readfirstlane(uint32_t v)
{
    return static_cast<uint32_t>(wave_emu::wave_op(v).operand(0u));
}
// row_shr:1/2/4/8 and row_bcast:15/31, no lane masked, out-of-range lanes keep `old`
inline uint32_t __builtin_amdgcn_update_dpp(uint32_t old, uint32_t v, uint32_t ctrl, uint32_t, uint32_t, bool)
{
    const uint32_t lane = wave_emu::g->cur & 63u;
    const wave_emu::wave_op op(v);
    if (ctrl > 0x110u && ctrl < 0x120u) {
        const uint32_t d = ctrl - 0x110u;
        return (lane & 15u) >= d ? static_cast<uint32_t>(op.operand(lane - d)) : old;
    }
    if (ctrl == 0x142u) return lane >= 16u ? static_cast<uint32_t>(op.operand((lane & ~15u) - 1u)) : old;
    if (ctrl == 0x143u) return lane >= 32u ? static_cast<uint32_t>(op.operand(31u)) : old;
    wave_emu::fatal("a data-parallel move that is not written here");
    return old;
}
inline int __popcll(uint64_t v)
{
    return __builtin_popcountll(v);
}
inline int __clz(int v)
{
    return v ? __builtin_clz(static_cast<unsigned>(v)) : 32;
}
inline int __clzll(long long v)
{
    return v ? __builtin_clzll(static_cast<unsigned long long>(v)) : 64;
}
inline uint32_t __brev(uint32_t v)
{
    uint32_t r = 0u;
    for (uint32_t b = 0; b < 32u; ++b) r |= ((v >> b) & 1u) << (31u - b);
    return r;
}
template <class T>
inline T atomicAdd(T *p, T v)
{
    const T o = *p;
    *p = o + v;
    return o;
}
inline uint32_t atomicMax(uint32_t *p, uint32_t v)
{
    const uint32_t o = *p;
    *p = std::max(o, v);
    return o;
}
inline uint32_t atomicMin(uint32_t *p, uint32_t v)
{
    const uint32_t o = *p;
    *p = std::min(o, v);
    return o;
}
