// CPU check of prefetch_multiples (pagmo2_amd/csrc/mt_jump_host.hpp): afterwards every
// multiple asked for is memoised, also where the last one was there before as a
// multiple of another distance, and each is z^(k S) mod phi.
#include <cstdio>

#include "mt_jump_host.hpp"

using namespace pgh::mtj;

static int failures = 0;

static void check(uint64_t S, uint64_t count)
{
    prefetch_multiples(S, count);
    const poly step = the_field().zpow(S);
    poly want = step;
    for (uint64_t k = 1; k <= count; ++k) {
        const auto it = the_cache().map.find(k * S);
        if (it == the_cache().map.end()) {
            std::printf("z^(%llu x %llu) is not memoised\n", static_cast<unsigned long long>(k),
                        static_cast<unsigned long long>(S));
            ++failures;
            return;
        }
        if (it->second != want) {
            std::printf("z^(%llu x %llu) is wrong\n", static_cast<unsigned long long>(k),
                        static_cast<unsigned long long>(S));
            ++failures;
            return;
        }
        want = the_field().mul(want, step);
    }
}

int main()
{
    check(uint64_t(1) << 18, 15);
    check(uint64_t(1) << 15, 120); // 120 x 2^15 = 15 x 2^18
    check(uint64_t(1) << 15, 40);  // fewer: all there
    check(uint64_t(1) << 15, 131); // more of them
    check(uint64_t(1) << 14, 1);
    check(uint64_t(1) << 14, 37);
    check(624u * 41u + 7u, 20); // a distance of no particular form
    if (failures) return 1;
    std::puts("ok");
    return 0;
}
