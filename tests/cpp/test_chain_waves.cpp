// test_chain_waves.cpp -- k_chain of pagmo2_amd/csrc/fnds_chain.hip on the CPU under
// several orders of its wavefronts (wave_emu.hpp): the members' positions inside
// their fronts must be those of the reference's loop
// (src/utils/multi_objective.cpp:210-254), whichever wavefront is ahead.
// The kernels' text comes from the source file by way of tests/test_chain_waves_cpu.py.
#include <cstdio>
#include <cstring>
#include <numeric>
#include <string>
#include <vector>

#include "wave_emu.hpp"

namespace pgh
{
constexpr uint32_t kChainMaxN = 16384, kChainMaxM = 3;
inline void wave_lds_fence()
{
    wave_emu::wave_op(0u);
}
#include "bin/fnds_chain_kernels.inc"
} // namespace pgh

using namespace pgh;

struct problem {
    std::string name;
    std::vector<double> x, y;
};

static problem layers(const std::string &name, const std::vector<uint32_t> &sizes, double delta, uint32_t seed)
{
    std::mt19937 rng(seed);
    std::uniform_real_distribution<double> u(0., 1.);
    std::vector<std::pair<double, double>> p;
    for (size_t L = 0; L < sizes.size(); ++L) {
        for (uint32_t k = 0; k < sizes[L]; ++k) {
            const double a = u(rng);
            p.emplace_back(a + delta * static_cast<double>(L), 1. - a + delta * static_cast<double>(L));
        }
    }
    std::shuffle(p.begin(), p.end(), rng);
    problem r;
    r.name = name;
    for (auto &q : p) {
        r.x.push_back(q.first);
        r.y.push_back(q.second);
    }
    return r;
}

static int check(const problem &pr, int how, uint32_t seed)
{
    const uint32_t n = static_cast<uint32_t>(pr.x.size());
    const auto dom = [&](uint32_t a, uint32_t b) {
        return pr.x[a] <= pr.x[b] && pr.y[a] <= pr.y[b] && (pr.x[a] < pr.x[b] || pr.y[a] < pr.y[b]);
    };
    // the reference's loop
    std::vector<uint32_t> cnt(n, 0u);
    for (uint32_t i = 0; i < n; ++i) {
        for (uint32_t j = 0; j < n; ++j) cnt[j] += dom(i, j) ? 1u : 0u;
    }
    std::vector<std::vector<uint32_t>> fronts(1);
    for (uint32_t i = 0; i < n; ++i) {
        if (!cnt[i]) fronts[0].push_back(i);
    }
    while (!fronts.back().empty()) {
        std::vector<uint32_t> next;
        for (uint32_t p : fronts.back()) {
            for (uint32_t q = 0; q < n; ++q) {
                if (dom(p, q) && --cnt[q] == 0u) next.push_back(q);
            }
        }
        fronts.push_back(next);
    }
    fronts.pop_back();
    // the kernel's inputs: offsets, members by index, and their dominators' bits
    std::vector<uint32_t> fo(n + 1u, 0u), want(n);
    std::vector<uint64_t> masks;
    std::vector<uint32_t> before, first(n, 0u); // first: the second front's last dominators' places
    for (size_t f = 0; f < fronts.size(); ++f) {
        std::vector<uint32_t> by = fronts[f];
        std::sort(by.begin(), by.end());
        const uint32_t at = fo[f], size = static_cast<uint32_t>(by.size());
        fo[f + 1u] = at + size;
        for (uint32_t k = 0; k < size; ++k) {
            const auto it = std::find(fronts[f].begin(), fronts[f].end(), by[k]);
            want[at + k] = static_cast<uint32_t>(it - fronts[f].begin());
        }
        if (f) {
            const uint32_t words = (static_cast<uint32_t>(before.size()) + 63u) / 64u;
            for (uint32_t w = 0; w < words; ++w) {
                for (uint32_t c = 0; c < size; ++c) {
                    uint64_t bits = 0u;
                    for (uint32_t q = 64u * w; q < std::min<size_t>(64u * w + 64u, before.size()); ++q) {
                        if (dom(before[q], by[c])) bits |= uint64_t(1) << (q - 64u * w);
                    }
                    if (f == 1u && bits) first[at + c] = 64u * w + 63u - static_cast<uint32_t>(__builtin_clzll(bits));
                    // (a large second front's words are not there on the device)
                    masks.push_back(f == 1u && size > kWide && n > 2u * kWide ? 0xababababababababull : bits);
                }
            }
        }
        before = by;
    }
    const uint64_t used = masks.size(), mask_words = n + static_cast<uint64_t>(n) * n / 256u + 64u;
    masks.resize(mask_words + 8192u, 0xabababababababababull); // a guard past the end
    uint32_t P = 1u;
    while (P < n) P <<= 1;
    const uint64_t scalars[4] = {fronts.size(), 0u, 0u, 0u};
    std::vector<uint32_t> got(n, 0xffffffffu);
    std::memset(wave_emu::dynamic_lds, 0xcd, sizeof wave_emu::dynamic_lds);
    wave_emu::run(kWide, how, seed, [&] {
        k_chain(fo.data(), masks.data(), mask_words, n, scalars, n, P, first.data(), got.data());
    });
    for (uint32_t i = 0; i < n; ++i) {
        if (got[i] != want[i]) {
            std::printf("%s, order %d, seed %u: n %u, %zu fronts, %llu words: place %u is %u, not %u\n", pr.name.c_str(),
                        how, seed, n, fronts.size(), static_cast<unsigned long long>(used), i, got[i], want[i]);
            return 1;
        }
    }
    return 0;
}

int main()
{
    std::vector<problem> ps;
    // runs of small fronts longer than what is staged at a time, one behind another
    ps.push_back(layers("small fronts", std::vector<uint32_t>(70, 40u), 0.03, 1u));
    ps.push_back(layers("fronts of two words", std::vector<uint32_t>(24, 110u), 2.0, 2u));
    // a run, then a front for the whole workgroup, then runs again
    {
        std::vector<uint32_t> s(40, 60u);
        s[20] = 1300u;
        ps.push_back(layers("a large front between", s, 2.0, 3u));
        s[20] = 500u;
        ps.push_back(layers("a middle front between", s, 2.0, 4u));
    }
    ps.push_back(layers("one large front after a small one", {90u, 1200u, 100u, 100u}, 2.0, 5u));
    // a large second front, and one behind it
    ps.push_back(layers("two large fronts", {300u, 1500u, 1100u, 60u}, 2.0, 6u));
    ps.push_back(layers("two large fronts of few dominators", {1500u, 1400u, 1200u}, 0.002, 7u));
    int bad = 0;
    for (const problem &p : ps) {
        bad += check(p, wave_emu::kFirstAhead, 0u);
        bad += check(p, wave_emu::kLastAhead, 0u);
        for (uint32_t s = 1; s <= 2u; ++s) bad += check(p, wave_emu::kShuffled, s);
    }
    if (bad) return 1;
    std::puts("ok");
    return 0;
}
