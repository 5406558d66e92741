// fnds_route.hpp -- which way fast_non_dominated_sorting takes to the fronts: from
// ranks (fnds_chain.hip) or by a peel (fnds.hip).  Host code without the runtime.
#pragma once

#include <cstdint>

namespace pgh
{

// fnds_chain.hip takes up to kChainMaxN points (its sort keys, positions and bit
// planes fit one workgroup's LDS) of one to kChainMaxM objectives.  With more
// objectives the fronts are few and large, and the grid-wide peel, whose cost is
// an exchange per front, is faster: ranks and order inside the fronts of 16384 x 3
// (54 fronts) took 0.70 ms against 0.90 for the peel with what leads up to it, of
// 16384 x 5 (15 fronts) 1.30 against 0.67; with two objectives (8192: 176-213 fronts)
// 0.40 against 1.2-1.4.  (Since then a large front costs the ranks a fraction of
// that; a whole call of 16384 x 3 takes 1.03 against 1.3 ms.)
constexpr uint32_t kChainMaxN = 16384, kChainMaxM = 3;

// A workspace's choice of peel.
struct peel_choice {
    uint32_t blocks = 0; // the peel's workgroups; 0: the default rule
    bool always = false; // also where the fronts would come from ranks
    // the caller's own count: every run is peeled by so many; 0: the default
    void set(uint32_t b)
    {
        blocks = b;
        always = b != 0u;
    }
    // A tuner's fastest count for n points of m objectives.  It stands for runs that
    // are peeled anyway; where the fronts could come from ranks only if it was faster
    // than those too.
    void tuned(uint64_t n, uint64_t m, uint32_t b, bool beats_ranks)
    {
        always = by_ranks(n, m) && beats_ranks;
        blocks = by_ranks(n, m) && !beats_ranks ? 0u : b;
    }
    static bool by_ranks(uint64_t n, uint64_t m)
    {
        return n <= kChainMaxN && m >= 1u && m <= kChainMaxM;
    }
    bool ranks(uint64_t n, uint64_t m) const
    {
        return by_ranks(n, m) && !always;
    }
};

} // namespace pgh
