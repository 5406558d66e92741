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
// of degree < 2 x 19968 is reduced through a table of z^(64 w) mod phi for the
// words w >= 312 it has: each such word c contributes c * (z^(64 w) mod phi),
// so the reduction is 312 x 312 independent word products; the bits 19937 ..
// 19967 left over are reduced one by one.
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
        // tab[w - kWords] = z^(64 w) mod phi, w = kWords .. 2 kWords - 1
        poly t = shift_reduce_bits(unit_at(64u * kWords));
        tab.push_back(t);
        for (uint32_t w = kWords + 1u; w < 2u * kWords; ++w) {
            t = times_z64(t);
            tab.push_back(t);
        }
        ok = true;
    }

    // a * b mod phi (a, b reduced)
    poly mul(const poly &a, const poly &b) const
    {
        poly prod(2u * kWords + 1u, 0u);
        for (uint32_t j = 0; j < kWords; ++j) {
            if (b[j]) mul_word_acc(a.data(), kWords, b[j], prod.data() + j);
        }
        return reduce(prod);
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
    std::vector<poly> tab;

    static poly unit_at(uint64_t i)
    {
        poly r(i / 64u + 1u, 0u);
        r[i / 64u] = uint64_t(1) << (i & 63u);
        return r;
    }

    // XOR of phi << s into r at bit position `at` (phi's leading bit lands on at + kDeg)
    void add_phi_at(poly &r, uint64_t at) const
    {
        const uint64_t ws = at >> 6, bs = at & 63u;
        for (uint64_t w = 0; w <= kWords; ++w) {
            const uint64_t lo = phi[w] << bs;
            const uint64_t hi = bs ? (phi[w] >> (64u - bs)) : 0u;
            if (ws + w < r.size()) r[ws + w] ^= lo;
            if (bs && ws + w + 1u < r.size()) r[ws + w + 1u] ^= hi;
        }
    }

    // bit-by-bit reduction (used for the table and the last 31 bits)
    poly shift_reduce_bits(poly r) const
    {
        for (uint64_t k = static_cast<uint64_t>(r.size()) * 64u; k-- > kDeg;) {
            if (bit(r, k)) add_phi_at(r, k - kDeg);
        }
        r.resize(kWords);
        return r;
    }

    poly times_z64(const poly &a) const
    {
        poly r(kWords + 1u, 0u);
        for (uint32_t w = 0; w < kWords; ++w) r[w + 1u] = a[w];
        return shift_reduce_bits(r);
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
        return shift_reduce_bits(r);
    }

    // prod has up to 2 kWords + 1 words: words w >= kWords fold through the
    // table (word 2 kWords is zero for products of reduced operands: their
    // degree is below 2 x 19937 - 1 < 64 x 2 kWords)
    poly reduce(const poly &prod) const
    {
        poly r(kWords + 1u, 0u);
        for (uint32_t w = 0; w < kWords; ++w) r[w] = prod[w];
        for (uint32_t w = kWords; w < 2u * kWords; ++w) {
            if (prod[w]) mul_word_acc(tab[w - kWords].data(), kWords, prod[w], r.data());
        }
        return shift_reduce_bits(r);
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
    const unsigned threads = std::min(8u, std::max(1u, std::thread::hardware_concurrency()));
    for (uint64_t m = std::max<uint64_t>(have, 1u); m < count;) {
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

} // namespace mtj
} // namespace pgh
