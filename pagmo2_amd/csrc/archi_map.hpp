// archi_map.hpp -- the launch mappings of an archipelago's generation: the default
// and those that pgh_archi_tune times (pso.hip; no result depends on them).
#pragma once

#include <cstdint>
#include <vector>

#include "pagmo_hip/pgh.h"

namespace pgh
{

// Default LDS for the individuals of a Lennard-Jones item: with it (and a
// rosenbrock item's) three workgroups fit a CU (two: 101 against 88 us a
// generation of the 32-island workload, 133 against 114 us of the 64-island one;
// four, with 36 KiB: 90 and 111; 16 KiB cuts the items of 12 islands too small,
// 56 against 51 us).
constexpr uint32_t kStepLjLds = 49152;

// The default (the 64-island workload's fastest form): its lj_lds of 0 means
// kStepLjLds.
constexpr pgh_archi_mapping kArchiDefault{PGH_ARCHI_STEP_ONE, 0u, 0u, 0u};

// What the tuner times, the default's like among them.
inline std::vector<pgh_archi_mapping> archi_candidates()
{
    std::vector<pgh_archi_mapping> cand;
    for (uint32_t form : {static_cast<uint32_t>(PGH_ARCHI_STEP_SPLIT), static_cast<uint32_t>(PGH_ARCHI_STEP_ONE)}) {
        for (uint32_t lds : {uint32_t(65536), kStepLjLds, uint32_t(32768), uint32_t(16384)}) {
            for (uint32_t bpc : {0u, 2u}) cand.push_back(pgh_archi_mapping{form, lds, bpc, 0u});
        }
    }
    return cand;
}

} // namespace pgh
