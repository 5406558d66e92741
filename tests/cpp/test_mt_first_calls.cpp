// CPU check of when a table of jumps is made (pagmo2_amd/csrc/mt_jump_host.hpp,
// without_table): not for one call of up to 2^21 words nor for a few small ones, at
// once for a larger one, and for many small ones in the end.
#include <cstdio>

#include "mt_jump_host.hpp"

using pgh::mtj::without_table;

static int failures = 0;

static void expect(bool ok, const char *what)
{
    if (!ok) {
        std::printf("%s\n", what);
        ++failures;
    }
}

int main()
{
    for (uint64_t n : {uint64_t(131074), uint64_t(1) << 18, uint64_t(1) << 20, uint64_t(1) << 21}) {
        uint64_t spent = 0u, calls = 0u;
        expect(without_table(spent, n), "the first call makes a table");
        for (calls = 1; without_table(spent, n); ++calls) {
        }
        expect(calls == (uint64_t(1) << 21) / n, "calls without a table");
        expect(!without_table(spent, n), "one that is due is put off");
    }
    uint64_t spent = 0u;
    expect(!without_table(spent, (uint64_t(1) << 21) + 1u), "a large call does without");
    expect(spent == 0u, "a large call is entered");
    if (failures) return 1;
    std::puts("ok");
    return 0;
}
