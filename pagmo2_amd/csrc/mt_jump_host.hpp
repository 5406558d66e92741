// mt_jump_host.hpp -- jump-ahead of std::mt19937 (host part): the polynomials
// that move a generator's state forward by J words.
//
// Method (Haramoto, Matsumoto, Nishimura, Panneton, L'Ecuyer, "Efficient jump
// ahead for F2-linear random number generators", INFORMS J. Computing 20,
// 2008).  With T the one-word transition of the state S_j = (x[j], ...,
// x[j+623]) of the recurrence in mt_dev.hpp and phi the characteristic
// polynomial of T, T^J = p(T) for p = z^J mod phi, so that
//   S_J = p(T) S_0,   word k of S_J = XOR over the set coefficients i of p of x[i+k].
// T never reads the 31 low bits of x[j], so the identity holds on every bit
// that a later word depends on.  phi has degree 19937 and the closed form that
// Matsumoto and Nishimura give ("Mersenne Twister", ACM TOMACS 8, 1998,
// appendix), so it costs nothing to set up (Berlekamp-Massey over 2 x 19937
// output bits took 28 ms of a process's first jump).
//
// Polynomials over GF(2) are bit vectors (bit i = coefficient of z^i), 312
// 64-bit words below degree 19937.  Products use carry-less multiplication
// (PCLMULQDQ when the CPU has it, a shift-and-add loop otherwise).  A product
// is reduced from its highest words down by phi itself, which has 134 terms
// below z^19937, the highest of them 623 below: nine words at a time, XORed in
// at 134 places.  (Through a table of z^(64 w) mod phi, a carry-less product per
// word of the table's 312 x 312, a multiplication took 155 us; so it takes 100,
// and one by a power of z below the degree 20.)
#pragma once

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <map>
#include <mutex>
#include <random>
#include <thread>
#include <vector>

#if defined(__x86_64__)
#include <immintrin.h>
#endif

namespace pgh
{
namespace mtj
{

constexpr uint32_t kDeg = 19937;
constexpr uint32_t kWords = (kDeg + 63u) / 64u; // 312

using poly = std::vector<uint64_t>;

inline bool bit(const poly &p, uint64_t i)
{
    return i / 64u < p.size() && ((p[i >> 6] >> (i & 63u)) & 1u);
}

// 64 bits of p from bit `at` (zeros past the end).
inline uint64_t bits64(const poly &p, uint64_t at)
{
    const uint64_t w = at >> 6, s = at & 63u;
    const uint64_t lo = w < p.size() ? p[w] : 0u;
    if (s == 0u) return lo;
    const uint64_t hi = w + 1u < p.size() ? p[w + 1u] : 0u;
    return (lo >> s) | (hi << (64u - s));
}

// ---- carry-less 64 x 64 -> 128 -------------------------------------------------
inline void clmul_soft(uint64_t a, uint64_t b, uint64_t &lo, uint64_t &hi)
{
    lo = hi = 0u;
    for (uint32_t i = 0; i < 64u; ++i) {
        if ((b >> i) & 1u) {
            lo ^= a << i;
            if (i) hi ^= a >> (64u - i);
        }
    }
}

#if defined(__x86_64__)
__attribute__((target("pclmul,sse2"))) inline void clmul_hw(uint64_t a, uint64_t b, uint64_t &lo, uint64_t &hi)
{
    const __m128i r = _mm_clmulepi64_si128(_mm_cvtsi64_si128(static_cast<long long>(a)),
                                           _mm_cvtsi64_si128(static_cast<long long>(b)), 0x00);
    lo = static_cast<uint64_t>(_mm_cvtsi128_si64(r));
    hi = static_cast<uint64_t>(_mm_cvtsi128_si64(_mm_unpackhi_epi64(r, r)));
}

// acc[0 .. n] ^= a[0 .. n) * c (a word vector times one word)
__attribute__((target("pclmul,sse2"))) inline void mul_word_acc_hw(const uint64_t *a, uint64_t n, uint64_t c,
                                                                   uint64_t *acc)
{
    const __m128i cv = _mm_cvtsi64_si128(static_cast<long long>(c));
    __m128i carry = _mm_setzero_si128();
    for (uint64_t i = 0; i < n; ++i) {
        const __m128i r = _mm_clmulepi64_si128(_mm_cvtsi64_si128(static_cast<long long>(a[i])), cv, 0x00);
        // r = lo | hi << 64: lo goes to word i, hi to word i + 1
        const __m128i cur = _mm_xor_si128(r, carry);
        acc[i] ^= static_cast<uint64_t>(_mm_cvtsi128_si64(cur));
        carry = _mm_srli_si128(r, 8);
    }
    acc[n] ^= static_cast<uint64_t>(_mm_cvtsi128_si64(carry));
}

inline bool have_pclmul()
{
    static const bool yes = __builtin_cpu_supports("pclmul");
    return yes;
}
#endif

inline void mul_word_acc(const uint64_t *a, uint64_t n, uint64_t c, uint64_t *acc)
{
#if defined(__x86_64__)
    if (have_pclmul()) {
        mul_word_acc_hw(a, n, c, acc);
        return;
    }
#endif
    uint64_t carry = 0u;
    for (uint64_t i = 0; i < n; ++i) {
        uint64_t lo, hi;
        clmul_soft(a[i], c, lo, hi);
        acc[i] ^= lo ^ carry;
        carry = hi;
    }
    acc[n] ^= carry;
}

// ---- arithmetic modulo phi ------------------------------------------------------
class field
{
  public:
    bool ok = false;
    poly phi; // kWords + 1 words, degree kDeg

    field()
    {
        // phi = A (B^31 + a_0 B^30 + ... + a_30) + a_31 with A = z^624 + z^397,
        // B = z^623 + z^396 and a_i bit i of 0x9908b0df, by Horner's rule
        constexpr uint32_t a = 0x9908b0dfu;
        phi.assign(kWords + 1u, 0u);
        phi[0] = 1u;
        const auto times = [&](uint32_t hi, uint32_t lo, uint32_t c) {
            poly r(kWords + 1u, 0u);
            for (uint32_t s : {hi, lo}) {
                for (uint64_t w = 0; w <= kWords; ++w) {
                    const uint64_t at = 64u * w + s, q = at >> 6, b = at & 63u;
                    if (q <= kWords) r[q] ^= phi[w] << b;
                    if (b && q < kWords) r[q + 1u] ^= phi[w] >> (64u - b);
                }
            }
            r[0] ^= c;
            phi = r;
        };
        for (uint32_t i = 0; i < 31u; ++i) times(623u, 396u, (a >> i) & 1u);
        times(624u, 397u, (a >> 31) & 1u);
        if (!bit(phi, kDeg) || bits64(phi, kDeg + 1u)) return;
        for (uint32_t e = 0; e < kDeg; ++e) {
            if (bit(phi, e)) low.push_back(e);
        }
        ok = low.back() + 64u * kRun <= kDeg; // reduce() folds onto lower words only
    }

    // a * b mod phi (a, b reduced)
    poly mul(const poly &a, const poly &b) const
    {
        poly prod(2u * kWords + 1u, 0u);
        for (uint32_t j = 0; j < kWords; ++j) {
            if (b[j]) mul_word_acc(a.data(), kWords, b[j], prod.data() + j);
        }
        return reduce(std::move(prod));
    }

    poly sqr(const poly &a) const
    {
        return mul(a, a);
    }

    // z^J mod phi: left to right over J's bits, squaring and shifting by z
    poly zpow(uint64_t J) const
    {
        poly r(kWords, 0u);
        if (J < kDeg) {
            r[J >> 6] = uint64_t(1) << (J & 63u);
            return r;
        }
        r[0] = 1u;
        for (int b = 63; b >= 0; --b) {
            r = sqr(r);
            if ((J >> b) & 1u) r = times_z(r);
        }
        return r;
    }

  private:
    static constexpr uint32_t kRun = 9u; // words folded at a time
    std::vector<uint32_t> low;           // phi's exponents below kDeg, ascending

    // r ^= v z^at (z^kDeg mod phi), v of N words
    template <uint32_t N>
    void fold(uint64_t *__restrict__ r, const uint64_t *__restrict__ v, uint64_t at) const
    {
        for (const uint32_t e : low) {
            uint64_t *__restrict__ o = r + ((at + e) >> 6);
            const uint32_t b = (at + e) & 63u;
            uint64_t t[N + 1u];
            t[0] = v[0] << b;
            // (two shifts: by 64 - b, also for b = 0)
            for (uint32_t i = 1; i < N; ++i) t[i] = (v[i] << b) | ((v[i - 1u] >> 1) >> (63u - b));
            t[N] = (v[N - 1u] >> 1) >> (63u - b);
            for (uint32_t i = 0; i <= N; ++i) o[i] ^= t[i]; // (at + e lies over 600 below the words taken)
        }
    }

    poly times_z(const poly &a) const
    {
        poly r(kWords + 1u, 0u);
        uint64_t carry = 0u;
        for (uint32_t w = 0; w < kWords; ++w) {
            r[w] = (a[w] << 1) | carry;
            carry = a[w] >> 63;
        }
        r[kWords] = carry;
        return reduce(std::move(r));
    }

    // r mod phi, r of any length from kWords words on
    poly reduce(poly r) const
    {
        uint64_t top = r.size();
        for (; top >= kWords + kRun; top -= kRun) fold_top<kRun>(r, top);
        for (; top > kWords; --top) fold_top<1u>(r, top);
        // the last word's bits from kDeg on
        const uint64_t v = r[kWords - 1u] >> (kDeg & 63u);
        r[kWords - 1u] &= (uint64_t(1) << (kDeg & 63u)) - 1u;
        fold<1u>(r.data(), &v, 0u);
        r.resize(kWords);
        return r;
    }
    template <uint32_t N>
    void fold_top(poly &r, uint64_t top) const
    {
        uint64_t v[N], some = 0u;
        for (uint32_t i = 0; i < N; ++i) {
            v[i] = r[top - N + i];
            r[top - N + i] = 0u;
            some |= v[i];
        }
        if (some) fold<N>(r.data(), v, 64u * (top - N) - kDeg);
    }
};

inline const field &the_field()
{
    static const field f;
    return f;
}

struct poly_cache {
    std::mutex mu;
    std::map<uint64_t, poly> map; // references stay valid as entries are added
    std::map<uint64_t, uint64_t> runs; // S -> c: z^S, z^(2 S), ..., z^(c S) are all in map
};

inline poly_cache &the_cache()
{
    static poly_cache c;
    return c;
}

// z^J mod phi, memoised (the same few distances recur).
inline const poly &jump_poly(uint64_t J)
{
    poly_cache &c = the_cache();
    std::lock_guard<std::mutex> lk(c.mu);
    auto it = c.map.find(J);
    if (it != c.map.end()) return it->second;
    return c.map.emplace(J, the_field().zpow(J)).first->second;
}

// Computes the polynomials of the distances not yet memoised on up to
// `threads` host threads (each z^J is independent), so that the jump_poly
// calls that follow find them.
inline void prefetch_jump_polys(const std::vector<uint64_t> &Js, unsigned threads)
{
    const field &f = the_field();
    poly_cache &c = the_cache();
    std::vector<uint64_t> todo;
    {
        std::lock_guard<std::mutex> lk(c.mu);
        for (uint64_t J : Js) {
            if (!c.map.count(J) && std::find(todo.begin(), todo.end(), J) == todo.end()) todo.push_back(J);
        }
    }
    if (todo.size() < 2u || threads < 2u) return; // jump_poly computes them as they come
    std::vector<poly> res(todo.size());
    std::atomic<size_t> next{0};
    auto work = [&] {
        for (size_t i = next++; i < todo.size(); i = next++) res[i] = f.zpow(todo[i]);
    };
    std::vector<std::thread> pool;
    const size_t n = std::min<size_t>(threads, todo.size());
    try {
        pool.reserve(n);
        for (size_t t = 1; t < n; ++t) pool.emplace_back(work);
    } catch (...) {
        // fewer helper threads: the work queue is shared, so this thread and
        // those started finish it
    }
    work();
    for (auto &th : pool) th.join();
    std::lock_guard<std::mutex> lk(c.mu);
    for (size_t i = 0; i < todo.size(); ++i) c.map.emplace(todo[i], std::move(res[i]));
}

// z^(k S) mod phi for k = 1 .. count, memoised: one multiplication each
// rather than one exponentiation each.  With m of them known, the next
// (up to m) are those times z^(m S), shared among the host's threads.
inline void prefetch_multiples(uint64_t S, uint64_t count)
{
    if (count == 0u || S == 0u) return;
    poly_cache &c = the_cache();
    const field &f = the_field();
    std::vector<poly> res(count + 1u); // res[k]: z^(k S)
    uint64_t have = 0u;
    {
        // (count S alone says nothing: it may be there as a multiple of another distance)
        std::lock_guard<std::mutex> lk(c.mu);
        const auto run = c.runs.find(S);
        if (run != c.runs.end()) have = run->second;
        if (have >= count) return;
        for (uint64_t k = 1; k <= have; ++k) res[k] = c.map.at(k * S);
    }
    if (have == 0u) res[1] = jump_poly(S);
    uint64_t known = std::max<uint64_t>(have, 1u);
    // z^S is one term below the degree: its products are cheap, and the first few are
    // sooner made one after another than by threads
    for (; S < kDeg && known < std::min<uint64_t>(count, 32u); ++known) res[known + 1u] = f.mul(res[known], res[1]);
    const unsigned threads = std::min(8u, std::max(1u, std::thread::hardware_concurrency()));
    for (uint64_t m = known; m < count;) {
        const uint64_t n = std::min(m, count - m);
        std::atomic<uint64_t> next{1};
        const auto work = [&] {
            for (uint64_t k = next++; k <= n; k = next++) res[m + k] = f.mul(res[k], res[m]);
        };
        std::vector<std::thread> pool;
        try {
            if (n >= 8u) {
                pool.reserve(threads);
                for (unsigned t = 1; t < threads; ++t) pool.emplace_back(work);
            }
        } catch (...) {
            // fewer helper threads: the work queue is shared, so this thread
            // and those started finish it
        }
        work();
        for (auto &th : pool) th.join();
        m += n;
    }
    std::lock_guard<std::mutex> lk(c.mu);
    for (uint64_t k = have + 1u; k <= count; ++k) c.map.emplace(k * S, std::move(res[k]));
    uint64_t &run = c.runs[S];
    run = std::max(run, count);
}

// ---- shares of an archipelago's velocity draws -------------------------------------
// Words per share, where all islands together draw `total` on a device of `cus` CUs:
// 2^15, or the power of two that leaves two to four shares per CU.  A share costs a
// jump, as much as making 1.5 10^5 words, and its polynomial's place in the
// archipelago's table: 10^8 words in shares of 2^15 would be 3052 of them.
inline uint64_t velocity_share(uint64_t total, uint32_t cus)
{
    const uint64_t want = total / (2u * std::max(cus, 1u));
    uint64_t share = uint64_t(1) << 15;
    while (share * 2u <= want) share *= 2u;
    return share;
}

// ---- when a device table of multiples is worth making ----------------------------
// Making one costs a process 1 to 3 ms once (31 to 127 multiples, an allocation and
// an upload), as long as one workgroup takes for 2^21 to 2^23 words.  So calls of up
// to kRentWords words do without, as one segment, until those of the table's size
// class have come to that many words between them: a program that draws one
// population never pays for the table, one that draws many soon has it.
constexpr uint64_t kRentWords = uint64_t(1) << 21;

// A call of `words` words finds no table, and those before it made `spent`: true if
// it does without, which is entered.
inline bool without_table(uint64_t &spent, uint64_t words)
{
    if (words > kRentWords || spent + words > kRentWords) return false;
    spent += words;
    return true;
}

} // namespace mtj
} // namespace pgh
