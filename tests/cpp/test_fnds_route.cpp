// CPU check of pagmo2_amd/csrc/fnds_route.hpp: what setting and tuning a workspace's peel
// do to the runs after it.
#include <cstdio>

#include "fnds_route.hpp"

static int failures = 0;

static void expect(bool ok, const char *what)
{
    if (!ok) {
        std::puts(what);
        ++failures;
    }
}

int main()
{
    pgh::peel_choice p;
    expect(p.ranks(200, 2) && p.ranks(16384, 3) && p.ranks(2, 1), "the default: ranks");
    expect(!p.ranks(16385, 2) && !p.ranks(200, 4) && !p.ranks(200, 0), "the default: peels");
    p.tuned(12000, 5, 47, true);
    expect(p.blocks == 47u, "the tuned count");
    expect(p.ranks(200, 2), "tuning an input that is always peeled takes the ranks from later small runs");
    p.tuned(20000, 2, 79, true);
    expect(p.ranks(16384, 3) && p.blocks == 79u, "tuning many points takes the ranks from later runs");
    p.tuned(8192, 2, 32, false);
    expect(p.ranks(8192, 2) && p.blocks == 0u, "the ranks were faster");
    p.tuned(8192, 2, 32, true);
    expect(!p.ranks(8192, 2) && p.blocks == 32u, "the peel was faster");
    p.set(20);
    expect(!p.ranks(8192, 2) && p.blocks == 20u, "a count that is set peels");
    p.set(0);
    expect(p.ranks(8192, 2) && p.blocks == 0u, "back to the default");
    if (failures) return 1;
    std::puts("ok");
    return 0;
}
