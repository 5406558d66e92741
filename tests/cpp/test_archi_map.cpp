// CPU check of pagmo2_amd/csrc/archi_map.hpp: the mapping that an archipelago has by
// default is among those that the tuner times, and each is one that may be set.
#include <cstdio>

#include "archi_map.hpp"

int main()
{
    int failures = 0;
    bool found = false;
    const pgh_archi_mapping d = pgh::kArchiDefault;
    const uint32_t lds = d.lj_lds ? d.lj_lds : pgh::kStepLjLds;
    for (const pgh_archi_mapping &m : pgh::archi_candidates()) {
        found |= m.form == d.form && (m.lj_lds ? m.lj_lds : pgh::kStepLjLds) == lds && m.blocks_per_cu == d.blocks_per_cu;
        if (m.form > 1u || m.lj_lds > 65536u || m.blocks_per_cu > 64u) ++failures;
    }
    if (!found) {
        std::puts("the tuner does not time the default mapping");
        ++failures;
    }
    if (failures) return 1;
    std::puts("ok");
    return 0;
}
