// test_rank_waves.cpp -- k_order, k_rank, k_far, k_fronts, k_slots and k_masks of
// pagmo2_amd/csrc/fnds_chain.hip on the CPU under several orders of their wavefronts
// (wave_emu.hpp): the ranks must be those of the definition, whatever share of the
// points has no dominator.  Tiles that the kernels may not read hold garbage.
#include <cstdio>
#include <cstring>
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

enum kind : int { kUniform, kLong, kChainOnly, kOneFront, kThreeFronts, kOneDominated, kSeventh, kKinds };

static int check(uint32_t n, int which, int how)
{
    std::mt19937 rng(n + static_cast<uint32_t>(which));
    std::uniform_real_distribution<double> u(0., 1.);
    std::vector<double> x(n), y(n);
    for (uint32_t i = 0; i < n; ++i) {
        x[i] = u(rng);
        switch (which) {
            case kUniform: y[i] = u(rng); break;
            case kLong: y[i] = x[i] + 0.05 * u(rng); break;
            case kChainOnly: y[i] = x[i]; break;
            case kOneFront: y[i] = -x[i]; break;
            case kThreeFronts: y[i] = -x[i] + (i % 3u) * 3.; break;
            case kOneDominated: y[i] = -x[i] + (i == n / 2u ? 3. : 0.); break;
            default: y[i] = -x[i] + (i % 7u == 0u ? 3. : 0.); break;
        }
    }
    const auto dom = [&](uint32_t a, uint32_t b) {
        return x[a] <= x[b] && y[a] <= y[b] && (x[a] < x[b] || y[a] < y[b]);
    };
    std::vector<uint32_t> cnt(n, 0u), place(n), perm(n);
    for (uint32_t i = 0; i < n; ++i) {
        for (uint32_t j = 0; j < n; ++j) cnt[j] += dom(i, j) ? 1u : 0u;
    }
    uint64_t n_free = ~uint64_t(0);
    wave_emu::run(kWide, how, 1u, [&] { k_order(cnt.data(), n, place.data(), &n_free); });
    bool ok = n_free == static_cast<uint64_t>(std::count(cnt.begin(), cnt.end(), 0u));
    for (uint32_t i = 0; i < n; ++i) {
        perm[place[i]] = i;
    }
    const uint32_t nb = (n + 63u) / 64u;
    std::vector<uint64_t> tiles(static_cast<size_t>(nb) * (nb + 1u) / 2u * 64u, 0xabababababababab);
    for (uint32_t J = 0; J < nb; ++J) {
        if (block_is_free(n_free, n, J)) continue;
        for (uint32_t I = 0; I <= J; ++I) {
            for (uint32_t c = 0; c < 64u; ++c) {
                uint64_t w = 0u;
                for (uint32_t k = 0; 64u * J + c < n && k < 64u && 64u * I + k < n; ++k) {
                    if (dom(perm[64u * I + k], perm[64u * J + c])) w |= uint64_t(1) << k;
                }
                tiles[tile_at(J, I) + c] = w;
            }
        }
    }
    std::vector<uint32_t> base(n, 0xdeadu), ranks(n, 777u), top(nb, 0u), want(n, 0u);
    std::vector<uint64_t> planes(static_cast<size_t>(nb) * kPlanes, 0u);
    uint32_t fronts = 1u;
    for (uint32_t e = 0; e < n; ++e) {
        for (uint32_t d = 0; d < e; ++d) {
            if (dom(perm[d], perm[e])) want[e] = std::max(want[e], want[d] + 1u);
        }
        fronts = std::max(fronts, want[e] + 1u);
    }
    for (uint32_t J0 = 0; J0 < nb; J0 += kSpan) {
        const uint32_t J1 = std::min(J0 + kSpan, nb);
        wave_emu::run(kWide, how, 2u, [&] {
            k_rank(tiles.data(), n, J0, J1, J0 ? base.data() : nullptr, ranks.data(), planes.data(), top.data(),
                   &n_free);
        });
        for (uint32_t b = 0; b < nb - J1; ++b) {
            wave_emu::block_idx.x = b;
            wave_emu::run(kFarBlock, how, 3u, [&] {
                k_far(tiles.data(), n, J0, J1, planes.data(), top.data(), base.data(), J0 == 0u ? 1u : 0u, &n_free);
            });
        }
        wave_emu::block_idx.x = 0u;
    }
    std::vector<uint32_t> fo(n + 1u), rank(n), any(n);
    std::vector<uint64_t> fo64(n + 1u), wbase(n + 1u);
    uint64_t scalars[4] = {0u, 0u, 0u, 0u};
    wave_emu::run(kWide, how, 4u, [&] {
        k_fronts(ranks.data(), perm.data(), n, fo.data(), fo64.data(), wbase.data(), rank.data(), any.data(), scalars);
    });
    ok = ok && scalars[0] == fronts;
    std::vector<uint32_t> seen(n, 0u);
    for (uint32_t e = 0; e < n; ++e) {
        ok = ok && ranks[e] == want[e] && rank[perm[e]] == want[e] && any[e] < n && rank[any[e]] < fronts &&
             fo[rank[any[e]]] <= e && e < fo[rank[any[e]] + 1u];
        if (any[e] < n) ++seen[any[e]];
    }
    for (uint32_t i = 0; i < n; ++i) ok = ok && seen[i] == 1u;
    // every front's members by index
    std::vector<uint32_t> members(n, 0xffffffffu);
    const uint32_t per = kBlock / 64u, groups = (n + per - 1u) / per, extra = n > kBigFront ? (nb + per - 1u) / per : 0u;
    for (uint32_t b = 0; ok && b < groups + extra; ++b) {
        wave_emu::block_idx.x = b;
        wave_emu::run(kBlock, how, 5u, [&] { k_slots(any.data(), rank.data(), fo.data(), n, extra, members.data()); });
    }
    wave_emu::block_idx.x = 0u;
    for (uint32_t f = 0; ok && f < fronts; ++f) {
        for (uint32_t q = fo[f]; q < fo[f + 1u]; ++q) {
            ok = ok && members[q] < n && rank[members[q]] == f && (q == fo[f] || members[q - 1u] < members[q]);
        }
    }
    // the dominators' bits in the front before
    std::vector<int64_t> keys(2u * n);
    for (uint32_t i = 0; i < n; ++i) {
        // (positive once shifted: a double's bits then order as the double does)
        const double v[2] = {x[i] + 8., y[i] + 8.};
        std::memcpy(&keys[2u * i], v, sizeof v);
    }
    uint64_t words = 0u;
    for (uint32_t f = 1; ok && f < fronts; ++f) {
        ok = wbase[f] == words;
        words += static_cast<uint64_t>(fo[f + 1u] - fo[f]) * ((fo[f] - fo[f - 1u] + 63u) / 64u);
    }
    std::vector<uint64_t> masks(words + 1u, 0xcdcdcdcdcdcdcdcd);
    std::vector<uint32_t> first(n, 0u);
    const uint32_t large_x = (nb + per - 1u) / per, large_y = n > 2u * kWide ? std::min((nb + kTileWords - 1u) / kTileWords, 7u) : 0u;
    for (uint32_t b = 0; ok && b < large_x * large_y + groups; ++b) {
        wave_emu::block_idx.x = b;
        wave_emu::run(kBlock, how, 6u, [&] {
            k_masks<2>(keys.data(), cnt.data(), members.data(), rank.data(), fo.data(), wbase.data(), n, large_x, large_y,
                       masks.data(), first.data());
        });
    }
    wave_emu::block_idx.x = 0u;
    const auto shifted_dom = [&](uint32_t a, uint32_t b) {
        return keys[2u * a] <= keys[2u * b] && keys[2u * a + 1u] <= keys[2u * b + 1u] && cnt[a] < cnt[b];
    };
    for (uint32_t f = 1; ok && f < fronts; ++f) {
        const uint32_t a = fo[f], size = fo[f + 1u] - a, pa = fo[f - 1u], sw = (a - pa + 63u) / 64u;
        for (uint32_t c = 0; ok && c < size; ++c) {
            if (f == 1u && size > kWide && large_y) { // the last dominator's place instead
                uint32_t last = 0u;
                for (uint32_t q = 0; q < a - pa; ++q) last = shifted_dom(members[pa + q], members[a + c]) ? q : last;
                ok = first[a + c] == last;
                continue;
            }
            for (uint32_t w = 0; ok && w < sw; ++w) {
                uint64_t bits = 0u;
                for (uint32_t q = 64u * w; q < std::min(64u * w + 64u, a - pa); ++q) {
                    if (shifted_dom(members[pa + q], members[a + c])) bits |= uint64_t(1) << (q - 64u * w);
                }
                ok = masks[wbase[f] + static_cast<uint64_t>(w) * size + c] == bits;
            }
        }
    }
    ok = ok && masks[words] == 0xcdcdcdcdcdcdcdcd;
    if (!ok) std::printf("%u points of kind %d, order %d\n", n, which, how);
    return ok ? 0 : 1;
}

int main()
{
    int bad = 0;
    for (uint32_t n : {2u, 65u, 700u}) {
        for (int which = 0; which < kKinds; ++which) {
            for (int how : {wave_emu::kFirstAhead, wave_emu::kLastAhead, wave_emu::kShuffled}) bad += check(n, which, how);
        }
    }
    // beyond a span of blocks
    bad += check(2300u, kOneFront, wave_emu::kFirstAhead);
    bad += check(2300u, kOneDominated, wave_emu::kShuffled);
    bad += check(2300u, kThreeFronts, wave_emu::kFirstAhead);
    // a front beyond kBigFront, alone and beside another
    bad += check(4161u, kOneFront, wave_emu::kShuffled);
    bad += check(4900u, kSeventh, wave_emu::kFirstAhead);
    // a second front beyond kWide behind one and before another
    bad += check(3300u, kThreeFronts, wave_emu::kLastAhead);
    if (bad) return 1;
    std::puts("ok");
    return 0;
}
