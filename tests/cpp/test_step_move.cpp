// test_step_move.cpp -- step_move of pagmo2_amd/csrc/pso.hip on the CPU (wave_emu.hpp):
// several elements in flight per thread read and write the item's own elements, their
// words and their neighbours' memory only, whatever the row length, and each element
// as the launch-per-element form does.  Every array lies between two pages that may
// not be touched, flush with one of them; the kernel's text comes from the source
// file by way of tests/test_step_move_cpu.py.
#include <sys/mman.h>
#include <unistd.h>

#include <cmath>
#include <cstdio>
#include <cstring>
#include <vector>

#include "wave_emu.hpp"

struct uint4 {
    uint32_t x, y, z, w;
};

namespace pgh
{
constexpr uint32_t kBlock = 256, kGenBatch = 32;
inline void bounds_of(int, uint32_t j, double &lb, double &ub)
{
    lb = -5. - 0.01 * j;
    ub = 10. + 0.02 * j;
}
inline double mt_canonical(uint32_t u0, uint32_t u1)
{
    return std::fmin(std::fma(static_cast<double>(u1), 4294967296.0, static_cast<double>(u0)), 0x1.fffffffffffffp63) *
           0x1p-64;
}
#include "bin/step_move.inc"
} // namespace pgh

using namespace pgh;

// n values between two pages without access, flush with the one behind or before.
template <class T>
struct guarded {
    T *p = nullptr;
    char *map = nullptr;
    size_t bytes = 0;
    guarded(size_t n, bool at_end)
    {
        const size_t page = static_cast<size_t>(sysconf(_SC_PAGESIZE));
        const size_t body = (n * sizeof(T) + page - 1u) / page * page;
        bytes = body + 2u * page;
        map = static_cast<char *>(mmap(nullptr, bytes, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0));
        mprotect(map, page, PROT_NONE);
        mprotect(map + page + body, page, PROT_NONE);
        p = reinterpret_cast<T *>(map + page + (at_end ? body - n * sizeof(T) : 0u));
    }
    ~guarded()
    {
        munmap(map, bytes);
    }
};

template <uint32_t U>
static int check(uint32_t pop, uint32_t nx, uint32_t first, uint32_t count, bool at_end)
{
    std::mt19937 rng(pop * 131u + nx);
    std::uniform_real_distribution<double> u(-4., 9.);
    const size_t elems = static_cast<size_t>(pop) * nx;
    // the island's own part of each array, at its offset in it: nothing before or
    // behind is to be read
    guarded<double> X(elems, at_end), V(elems, at_end), L0(elems, at_end), L1(elems, at_end), lbf(pop, at_end);
    guarded<uint32_t> sel(pop, at_end), words(4u * elems, at_end);
    for (size_t m = 0; m < elems; ++m) {
        X.p[m] = u(rng);
        V.p[m] = 0.1 * u(rng);
        L0.p[m] = u(rng);
        L1.p[m] = u(rng);
        for (uint32_t q = 0; q < 4u; ++q) words.p[4u * m + q] = static_cast<uint32_t>(rng());
    }
    for (uint32_t p = 0; p < pop; ++p) {
        lbf.p[p] = u(rng);
        sel.p[p] = rng() & 1u;
    }
    island_desc di{};
    di.kind = 0;
    di.dim = di.nx = nx;
    di.pop = pop;
    di.gens = 1u;
    di.radius = 2u;
    di.omega = 0.7298;
    di.eta1 = di.eta2 = 2.05;
    di.max_vel = 0.5;
    di.xoff = 7777u;
    di.foff = 333u;
    di.woff = 4096u;
    di.variant = 5u;
    di.topo = 2u;
    tile tl{0u, first, count, 0u};
    step_args a{};
    a.words = words.p - di.woff;
    a.X = X.p - di.xoff;
    a.V = V.p - di.xoff;
    a.lbX0 = L0.p - di.xoff;
    a.lbX1 = L1.p - di.xoff;
    a.lbf_cur = lbf.p - di.foff;
    a.sel_cur = sel.p - di.foff;
    // element by element
    std::vector<double> wx(X.p, X.p + elems), wv(V.p, V.p + elems);
    for (uint32_t p = first; p < first + count; ++p) {
        const uint32_t bn = best_neighbour(p, pop, di.radius, lbf.p);
        for (uint32_t d = 0; d < nx; ++d) {
            const size_t m = static_cast<size_t>(p) * nx + d;
            const uint32_t *w = words.p + 4u * m;
            const double own = (sel.p[p] ? L1 : L0).p[m], best = (sel.p[bn] ? L1 : L0).p[static_cast<size_t>(bn) * nx + d];
            double v;
            const double x = pso_move(di, d, wx[m], wv[m], own, best, mt_canonical(w[0], w[1]), mt_canonical(w[2], w[3]), v);
            wx[m] = x;
            wv[m] = v;
        }
    }
    std::vector<double> put(static_cast<size_t>(count) * nx, -777.);
    static step_rows rw;
    bool went = true;
    wave_emu::run(kBlock, wave_emu::kShuffled, nx, [&] {
        if (!step_move<false, U>(di, tl, a, rw, [&](uint32_t t, uint32_t dd, double x) {
                if (t >= count || dd >= nx) went = false;
                else put[static_cast<size_t>(t) * nx + dd] = x;
            })) {
            went = false;
        }
    });
    bool ok = went && std::memcmp(wx.data(), X.p, elems * 8u) == 0 && std::memcmp(wv.data(), V.p, elems * 8u) == 0;
    ok = ok && std::memcmp(put.data(), wx.data() + static_cast<size_t>(first) * nx, put.size() * 8u) == 0;
    if (!ok) std::printf("pop %u, nx %u, rows %u + %u, %u in flight\n", pop, nx, first, count, U);
    return ok ? 0 : 1;
}

int main()
{
    int bad = 0;
    for (uint32_t nx : {1u, 2u, 3u, 7u, 15u, 16u, 17u, 63u, 64u, 65u, 100u, 127u, 129u, 255u, 256u, 257u, 300u, 511u, 512u,
                        513u, 777u, 1023u, 1025u}) {
        for (uint32_t count : {1u, 2u, 5u, 8u, 16u, 31u, 32u}) {
            if (count * nx > 9000u) continue;
            const uint32_t pop = count + 5u;
            bad += check<4>(pop, nx, 0u, count, false); // flush with the page before
            bad += check<4>(pop, nx, pop - count, count, true); // ... behind
            bad += check<2>(pop, nx, pop - count, count, true);
        }
    }
    bad += check<4>(261u, 3u, 5u, 256u, true);
    bad += check<2>(256u, 9u, 0u, 256u, false);
    if (bad) return 1;
    std::puts("ok");
    return 0;
}
