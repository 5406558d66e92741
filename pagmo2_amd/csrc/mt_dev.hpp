// mt_dev.hpp -- std::mt19937 (include/pagmo/rng.hpp:43) and libstdc++'s
// uniform_real_distribution<double> mapping, on the device.
//
// The generator is written from the MT19937 definition (Matsumoto & Nishimura
// 1998) as the linear recurrence over the word sequence x:
//   x[0..623]   = the seeded state (libstdc++ mersenne_twister_engine::seed)
//   x[k+624]    = x[k+397] ^ (((x[k] & 0x80000000) | (x[k+1] & 0x7fffffff)) >> 1)
//                 ^ (x[k+1] & 1 ? 0x9908b0df : 0)
//   output j    = temper(x[624+j])
// The words are made a block at a time, x[624 q .. 624 q + 623] from the block
// before it, by one workgroup: y[k] (k < 227) needs the old block only,
// y[k + 227] also y[k] and y[k + 454] also y[k + 227], so thread k makes those
// three words in registers and a block costs one workgroup barrier.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace pgh
{
namespace dev
{

constexpr uint32_t kMtN = 624u, kMtM = 397u, kMtStep = kMtN - kMtM;

// Generator state in device memory: a block of the word sequence and how many
// of its words have been handed out (the seeded block counts as handed out).
struct mt_state {
    uint32_t x[kMtN];
    uint32_t pos;
    uint32_t pad[15];
};

// a ^ (b & c), one three-input instruction
__device__ __forceinline__ uint32_t mt_xor_and(uint32_t a, uint32_t b, uint32_t c)
{
    return __builtin_amdgcn_bitop3_b32(a, b, c, 0x78);
}

__device__ __forceinline__ uint32_t mt_temper(uint32_t y)
{
    y ^= y >> 11;
    y = mt_xor_and(y, y << 7, 0x9d2c5680u);
    y = mt_xor_and(y, y << 15, 0xefc60000u);
    y ^= y >> 18;
    return y;
}

__device__ __forceinline__ uint32_t mt_next_word(uint32_t a, uint32_t b, uint32_t c)
{
    const uint32_t y = (a & 0x80000000u) | (b & 0x7fffffffu);
    return c ^ (y >> 1) ^ ((b & 1u) ? 0x9908b0dfu : 0u);
}

// libstdc++ mersenne_twister_engine::seed(sd): x[i] = 1812433253 *
// (x[i-1] ^ (x[i-1] >> 30)) + i.  Host side: the state is built once per seed
// (623 dependent multiplications, 12 us on one lane of the device).
inline void mt_seed_host(uint32_t seed, mt_state &st)
{
    st = mt_state{};
    st.x[0] = seed;
    for (uint32_t i = 1; i < kMtN; ++i) {
        const uint32_t p = st.x[i - 1];
        st.x[i] = 1812433253u * (p ^ (p >> 30)) + i;
    }
    st.pos = kMtN;
}

// libstdc++ generate_canonical<double, 53> over two 32-bit draws
// (bits/random.tcc): sum = u0 + u1 * 2^32 (one rounding; the product is exact,
// so the fma's rounding is the sum's), ret = sum / 2^64, and a result of 1
// becomes nextafter(1, 0) = 1 - 2^-53.  mt_sum is sum with that last case.
__device__ __forceinline__ double mt_sum(uint32_t u0, uint32_t u1)
{
    return fmin(fma(static_cast<double>(u1), 4294967296.0, static_cast<double>(u0)), 0x1.fffffffffffffp63);
}

__device__ __forceinline__ double mt_canonical(uint32_t u0, uint32_t u1)
{
    return mt_sum(u0, u1) * 0x1p-64; // exact scaling
}

// uniform_real_distribution<double>(a, b): canonical * (b - a) + a
// (bits/random.h, operator()), multiply and add rounded separately.  w is
// mt_width(a, b): for |b - a| above 2^-958 the scaling by 2^-64 is exact on
// either factor (a sum is 0 or at least 1), so the product rounds alike.  For a
// problem's bounds, which are units apart or more; an island's velocity limits
// can lie at any value and scale the sum (pso.hip, velocity_sink).
__host__ __device__ __forceinline__ double mt_width(double a, double b)
{
    return (b - a) * 0x1p-64;
}
__device__ __forceinline__ double mt_uniform(uint32_t u0, uint32_t u1, double a, double w)
{
    return mt_sum(u0, u1) * w + a;
}

// ---- a generator held in LDS by one workgroup ----------------------------------
// buf has kMtBuf words, two phases of four blocks.  Between calls the current
// block is at kMtCur and `pos` of its words have been handed out.
constexpr uint32_t kMtBlock = 512u;      // the generator kernels' workgroup
constexpr uint32_t kMtPhase = 4u * kMtN; // words per phase
constexpr uint32_t kMtCur = 3u * kMtN;
constexpr uint32_t kMtBuf = 5056u; // two phases, and the parts of a jump

// The block after A into B (disjoint).  A barrier must follow.
__device__ __forceinline__ void mt_block(const uint32_t *__restrict__ A, uint32_t *__restrict__ B)
{
    const uint32_t t = threadIdx.x;
    if (t < kMtStep) {
        const uint32_t l = min(t + 2u * kMtStep, kMtN - 2u); // the third word's first operand, t < 170
        const uint32_t a0 = A[t], a1 = A[t + 1u], c = A[t + kMtM], b0 = A[t + kMtStep], b1 = A[t + kMtStep + 1u];
        // x[623] and y[0] for the block's last word
        const uint32_t d0 = t == 169u ? A[kMtN - 1u] : A[l];
        uint32_t d1 = A[l + 1u];
        if ((t & ~63u) == 128u) {
            const uint32_t y0 = mt_next_word(A[0], A[1], A[kMtM]);
            if (t == 169u) d1 = y0;
        }
        const uint32_t w0 = mt_next_word(a0, a1, c), w1 = mt_next_word(b0, b1, w0);
        B[t] = w0;
        B[t + kMtStep] = w1;
        if (t < kMtN - 2u * kMtStep) B[t + 2u * kMtStep] = mt_next_word(d0, d1, w1);
    }
}

__device__ __forceinline__ void mt_load(const mt_state &st, uint32_t *__restrict__ buf, uint32_t &pos)
{
    for (uint32_t i = threadIdx.x; i < kMtN; i += kMtBlock) buf[kMtCur + i] = st.x[i];
    pos = st.pos;
    __syncthreads();
}

// The state after the last call, whose barrier orders buf's words.
__device__ __forceinline__ void mt_store(mt_state &st, const uint32_t *__restrict__ buf, uint32_t pos)
{
    for (uint32_t i = threadIdx.x; i < kMtN; i += kMtBlock) st.x[i] = buf[kMtCur + i];
    if (threadIdx.x == 0) st.pos = pos;
}

// Hands out the next `count` words: sink(at, words, n, tid, nthr), n words in
// LDS, untempered, from position `at` of the hand-out on (an even one after
// the first run), by threads tid of nthr, which must not synchronise.  The
// first four wavefronts make a phase of four blocks while the others hand out
// the phase before it, with a barrier per block: making a block is a chain of LDS
// reads, about 30 instructions for a thread's three words and LDS writes, which the
// hand-out's tempering and mapping (about 28 instructions per two words) overlaps.
// Measured: one workgroup alone makes 2.6 words/ns with the mapping to doubles
// (1.3 with a barrier per 227 words and the hand-out in the same threads, and
// the mapping in a pass of its own), two on a CU 3.4 together, which keeps its
// SIMDs about 60% busy; four on a CU make 4.0 but need twice the jumps.
template <class Sink>
__device__ __forceinline__ void mt_hand_out(uint32_t *__restrict__ buf, uint32_t &pos, uint64_t count, Sink sink)
{
    static_assert(kMtBlock == 512u, "four wavefronts make blocks, four hand out");
    const uint32_t t = threadIdx.x;
    uint64_t done = 0u, prev_at = 0u;
    const uint32_t have = static_cast<uint32_t>(min(static_cast<uint64_t>(kMtN - pos), count));
    if (have) {
        sink(static_cast<uint64_t>(0), buf + kMtCur + pos, have, t, kMtBlock);
        pos += have;
        done = have;
    }
    // the block to continue from, the phase before (prev_n words) and the one
    // being made, by offsets into buf
    uint32_t cur = kMtCur, prev = 0u, prev_n = 0u, ph = kMtPhase;
    while (done < count) {
        const uint32_t n = static_cast<uint32_t>(min(static_cast<uint64_t>(kMtPhase), count - done));
        const uint32_t blocks = (n + kMtN - 1u) / kMtN; // 1 .. 4
        for (uint32_t b = 0; b < 4u; ++b) {
            if (b < blocks) {
                mt_block(buf + cur, buf + ph + b * kMtN);
                cur = ph + b * kMtN;
            }
            // the phase before, 256 pairs of words at a time: two, one, one and
            // the last 224
            if (t >= 256u) {
                const uint32_t lo = b ? 512u * (b + 1u) : 0u, hi = min(prev_n, b < 3u ? 512u * (b + 2u) : kMtPhase);
                if (lo < hi) sink(prev_at + lo, buf + prev + lo, hi - lo, t - 256u, 256u);
            }
            __syncthreads();
        }
        prev = ph;
        prev_n = n;
        prev_at = done;
        ph = ph ? 0u : kMtPhase;
        done += n;
        pos = n - (blocks - 1u) * kMtN;
    }
    if (prev_n) sink(prev_at, buf + prev, prev_n, t, kMtBlock);
    // (the phase at kMtCur, unless it is the one just handed out and then cur
    // is kMtCur, was handed out before the last barrier)
    if (cur != kMtCur) {
        for (uint32_t i = t; i < kMtN; i += kMtBlock) buf[kMtCur + i] = buf[cur + i];
    }
    __syncthreads();
}

// mt_hand_out to memory, tempered.
struct mt_word_sink {
    uint32_t *out;
    __device__ __forceinline__ void operator()(uint64_t at, const uint32_t *__restrict__ w, uint32_t n, uint32_t tid,
                                               uint32_t nthr) const
    {
        uint32_t *o = out + at;
        // pairs of words when both sides are 8-byte aligned
        if (((reinterpret_cast<uintptr_t>(o) | reinterpret_cast<uintptr_t>(w)) & 7u) == 0u) {
            for (uint32_t i = tid; i < n / 2u; i += nthr) {
                const uint2 v = reinterpret_cast<const uint2 *>(w)[i];
                reinterpret_cast<uint2 *>(o)[i] = make_uint2(mt_temper(v.x), mt_temper(v.y));
            }
            if ((n & 1u) && tid == 0u) o[n - 1u] = mt_temper(w[n - 1u]);
        } else {
            for (uint32_t i = tid; i < n; i += nthr) o[i] = mt_temper(w[i]);
        }
    }
};

// Nothing handed to anyone: a generator that skips words.
struct mt_no_sink {
    __device__ __forceinline__ void operator()(uint64_t, const uint32_t *, uint32_t, uint32_t, uint32_t) const {}
};

// a[j] ^= c0 w[j] ^ c1 w[j + 1] (j < 10) for bits b and b + 1, c0 and c1, of the
// wavefront-uniform word pw: nothing, ten XORs or ten three-input XORs.
// Written out with its branches: from the C++ the compiler copied the ten
// accumulators on every path, as many moves as XORs.  Every lane is active.
__device__ __forceinline__ void mt_xor_pair(uint32_t (&a)[10], const uint32_t *w, uint32_t pw, uint32_t b)
{
    asm("s_bitcmp1_b32 %21, %22\n"
        "s_cbranch_scc0 .Lmt_first_off%=\n"
        "s_bitcmp1_b32 %21, %23\n"
        "s_cbranch_scc0 .Lmt_first_only%=\n"
        "v_bitop3_b32 %0, %0, %10, %11 bitop3:0x96\n"
        "v_bitop3_b32 %1, %1, %11, %12 bitop3:0x96\n"
        "v_bitop3_b32 %2, %2, %12, %13 bitop3:0x96\n"
        "v_bitop3_b32 %3, %3, %13, %14 bitop3:0x96\n"
        "v_bitop3_b32 %4, %4, %14, %15 bitop3:0x96\n"
        "v_bitop3_b32 %5, %5, %15, %16 bitop3:0x96\n"
        "v_bitop3_b32 %6, %6, %16, %17 bitop3:0x96\n"
        "v_bitop3_b32 %7, %7, %17, %18 bitop3:0x96\n"
        "v_bitop3_b32 %8, %8, %18, %19 bitop3:0x96\n"
        "v_bitop3_b32 %9, %9, %19, %20 bitop3:0x96\n"
        "s_branch .Lmt_done%=\n"
        ".Lmt_first_only%=:\n"
        "v_xor_b32 %0, %0, %10\n"
        "v_xor_b32 %1, %1, %11\n"
        "v_xor_b32 %2, %2, %12\n"
        "v_xor_b32 %3, %3, %13\n"
        "v_xor_b32 %4, %4, %14\n"
        "v_xor_b32 %5, %5, %15\n"
        "v_xor_b32 %6, %6, %16\n"
        "v_xor_b32 %7, %7, %17\n"
        "v_xor_b32 %8, %8, %18\n"
        "v_xor_b32 %9, %9, %19\n"
        "s_branch .Lmt_done%=\n"
        ".Lmt_first_off%=:\n"
        "s_bitcmp1_b32 %21, %23\n"
        "s_cbranch_scc0 .Lmt_done%=\n"
        "v_xor_b32 %0, %0, %11\n"
        "v_xor_b32 %1, %1, %12\n"
        "v_xor_b32 %2, %2, %13\n"
        "v_xor_b32 %3, %3, %14\n"
        "v_xor_b32 %4, %4, %15\n"
        "v_xor_b32 %5, %5, %16\n"
        "v_xor_b32 %6, %6, %17\n"
        "v_xor_b32 %7, %7, %18\n"
        "v_xor_b32 %8, %8, %19\n"
        "v_xor_b32 %9, %9, %20\n"
        ".Lmt_done%=:\n"
        : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(a[4]),
          "+v"(a[5]), "+v"(a[6]), "+v"(a[7]), "+v"(a[8]), "+v"(a[9])
        : "v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]), "v"(w[4]), "v"(w[5]),
          "v"(w[6]), "v"(w[7]), "v"(w[8]), "v"(w[9]), "v"(w[10]), "s"(pw), "n"(b), "n"(b + 1u)
        : "scc");
}

// ---- jumps -------------------------------------------------------------------
// A jump polynomial p = z^J mod phi on the device: its 19937 coefficients as
// kMtN 32-bit words (bit i of word c is coefficient 32 c + i), the last bits
// zero.
// Moves the generator J words ahead: word k of the block J words further on
// is the XOR of x[i + k] over the set coefficients i of p, x from the current
// block on (Haramoto et al. 2008; the low 31 bits of word 0 reach no later
// word).  pos stays: it counts within the block.
//
// A wavefront covers all 624 words, lane l the ten from 10 l on, and the eight
// wavefronts share the coefficients, 32 (one word of p) at a time: a lane
// loads the 42 words x[32 c + 10 l ..] once, for 320 (coefficient, word)
// pairs, and XORs ten of them per set coefficient; p's bits are uniform, so an
// unset coefficient costs a branch and two set ones in a row one three-input
// XOR per word.  The wavefronts' partial results are XORed in the end.  Bound
// by the VALU: 19937 x 10 x 3/8 instructions, 31 us of a CU.  Measured: 70 us
// for one jump on a CU, 47 us each for two or more at once (about 500 us for
// one before, when a thread kept one state word and walked the list of set
// coefficients with one LDS read per coefficient).
__device__ __forceinline__ void mt_jump(uint32_t *__restrict__ buf, const uint32_t *__restrict__ p)
{
    constexpr uint32_t kPer = 10u, kChunks = kMtPhase / 32u; // 78 chunks of 32 coefficients per phase
    constexpr uint32_t kPhases = 8u;                         // 8 x 2496 >= 19937 coefficients
    constexpr uint32_t kWaves = kMtBlock / 64u;
    const uint32_t t = threadIdx.x, lane = t & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(t >> 6);
    for (uint32_t i = t; i < kMtN; i += kMtBlock) buf[i] = buf[kMtCur + i];
    __syncthreads();
    uint32_t acc[kPer];
#pragma unroll
    for (uint32_t j = 0; j < kPer; ++j) acc[j] = 0u;
    const uint32_t *mine = buf + kPer * lane;
    for (uint32_t ph = 0;; ++ph) {
        // this wavefront's words of p: chunk wave + kWaves l in lane l
        const uint32_t ci = wave + kWaves * lane;
        const uint32_t pv = ci < kChunks ? p[ph * kChunks + ci] : 0u;
#pragma unroll
        for (uint32_t b = 0; b < 4u; ++b) {
            mt_block(buf + b * kMtN, buf + (b + 1u) * kMtN);
            __syncthreads();
        }
        for (uint32_t c = wave, q = 0; c < kChunks; c += kWaves, ++q) {
            const uint32_t pw = __builtin_amdgcn_readlane(pv, q);
            uint32_t w[42];
#pragma unroll
            for (uint32_t i = 0; i < 21u; ++i) {
                const uint2 v = reinterpret_cast<const uint2 *>(mine + 32u * c)[i];
                w[2u * i] = v.x;
                w[2u * i + 1u] = v.y;
            }
#pragma unroll
            for (uint32_t b = 0; b < 32u; b += 2u) {
                mt_xor_pair(acc, w + b, pw, b);
            }
        }
        __syncthreads();
        if (ph + 1u == kPhases) break;
        for (uint32_t i = t; i < kMtN; i += kMtBlock) buf[i] = buf[kMtPhase + i];
        __syncthreads();
    }
    // the wavefronts' parts, 630 words each (5040 of buf's)
    constexpr uint32_t kPart = 63u * kPer;
    static_assert(kWaves * kPart <= kMtBuf && kMtPhase + kMtN + 64u <= kMtBuf, "parts and over-read windows");
    if (lane < 63u) {
#pragma unroll
        for (uint32_t j = 0; j < kPer; ++j) buf[wave * kPart + kPer * lane + j] = acc[j];
    }
    __syncthreads();
    uint32_t y[2];
#pragma unroll
    for (uint32_t r = 0; r < 2u; ++r) {
        const uint32_t k = min(t + r * kMtBlock, kMtN - 1u);
        y[r] = 0u;
#pragma unroll
        for (uint32_t v = 0; v < kWaves; ++v) y[r] ^= buf[v * kPart + k];
    }
    __syncthreads();
#pragma unroll
    for (uint32_t r = 0; r < 2u; ++r) {
        if (t + r * kMtBlock < kMtN) buf[kMtCur + t + r * kMtBlock] = y[r];
    }
    __syncthreads();
}

} // namespace dev
} // namespace pgh
