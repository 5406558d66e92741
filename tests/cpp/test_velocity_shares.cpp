// CPU check of an archipelago's velocity shares (pagmo2_amd/csrc/mt_jump_host.hpp,
// velocity_share): 2^15 words up to two shares per CU of them, beyond a power of two
// of which there are at most four per CU.
#include <cstdio>

#include "mt_jump_host.hpp"

int main()
{
    int failures = 0;
    for (uint32_t cus : {1u, 80u, 256u}) {
        for (uint64_t total = 1; total < (uint64_t(1) << 42); total = total * 3u + 7u) {
            const uint64_t s = pgh::mtj::velocity_share(total, cus), n = (total + s - 1u) / s;
            const bool pow2 = (s & (s - 1u)) == 0u;
            const bool least = s == uint64_t(1) << 15;
            if (!pow2 || s < (uint64_t(1) << 15) || n > 4u * cus || (!least && n < 2u * cus) ||
                (total <= 2u * cus * (uint64_t(1) << 15) && !least)) {
                std::printf("%llu words, %u CUs: shares of %llu, %llu of them\n", static_cast<unsigned long long>(total),
                            cus, static_cast<unsigned long long>(s), static_cast<unsigned long long>(n));
                ++failures;
            }
        }
    }
    if (failures) return 1;
    std::puts("ok");
    return 0;
}
