// fnds_ws.hpp -- the fast_non_dominated_sorting workspace (fnds.hip) and the
// multi-objective orderings that reuse it (mo_sort.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <vector>

#include "fnds_route.hpp"
#include "pgh_internal.hpp"

namespace pgh
{
// Order-preserving int64 key of a double under pagmo's comparisons
// (include/pagmo/detail/custom_comparisons.hpp:54-100): NaN sorts after +inf
// and equals every NaN, -0 equals +0.
__device__ __forceinline__ int64_t order_key(double x)
{
    if (x != x) return INT64_MAX;
    if (x == 0.0) return 0; // -0 == +0
    const int64_t b = __double_as_longlong(x);
    return b >= 0 ? b : (b ^ INT64_MAX);
}

// Orders a wavefront's LDS writes before its following reads (its LDS accesses
// execute in order; the compiler must keep them so).
__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A buffer inside one of the workspace's allocations.
struct ws_view {
    void *ptr = nullptr;
};
struct ws_part {
    ws_view *view;
    uint64_t bytes;
};
// Lays the parts out in `mem`, grown if needed, each on a 256-byte boundary.
inline pgh_status ws_carve(dev_buf &mem, const std::vector<ws_part> &parts)
{
    const auto padded = [](uint64_t b) { return (std::max<uint64_t>(b, 8u) + 255u) & ~uint64_t(255); };
    uint64_t total = 0;
    for (const ws_part &p : parts) total += padded(p.bytes);
    PGH_TRY(mem.reserve(total));
    auto *at = static_cast<char *>(mem.ptr);
    for (const ws_part &p : parts) {
        p.view->ptr = at;
        at += padded(p.bytes);
    }
    return PGH_OK;
}
} // namespace pgh

struct pgh_fnds_ws {
    hipStream_t stream = nullptr;
    hipStream_t own = nullptr; // created by the host-buffer entry points
    pgh::dev_buf staged;
    uint64_t n = 0, m = 0, words = 0;
    // every call's buffers, and those of the domination lists, in one device
    // allocation each (a new workspace's first call took 26, 1.7 ms)
    pgh::dev_buf main, lists_mem;
    pgh::ws_view keys, cnt32, ndom32, key32, rank, front_items, front_offsets, scalars;
    pgh::ws_view D, dom_count, dom_offsets;
    pgh::dev_buf dom_items;
    pgh::dev_buf comp, ctl; // the grid peel's sort-key lists and flags (two halves each)
    // fnds_chain.hip: the order by dominator count with the keys, counts and
    // ranks in it, the dominance bits, what far blocks give a rank, the ranks'
    // bit planes; ranks by index, front offsets, offsets of the fronts' words
    // of `masks`, the members in any order and by index, their positions, and the last
    // dominators of a large second front
    pgh::ws_view perm, skeys, scnt, srank, tiles, base, planes, rank32, fo32, wbase, any, members, masks, pos32, first;
    uint64_t h_sizes[3] = {0, 0, 0}; // n_fronts, n_dom_items, peel barrier timeout
    bool sized = false;
    bool emitted = false; // dom_items holds the result's lists
    bool lists = false; // D, dom_offsets and dom_count hold this result's
    bool items = false; // front_items holds every front's
    bool by_ranks = false; // the result's fronts come from ranks (fnds_chain.hip)
    // workgroups of the grid-wide front peel, set or found by pgh_fnds_tune (any
    // count gives the same result, and so do ranks)
    pgh::peel_choice peel;
    // mo_sort.hip: sort keys and values (two of each), crowding, radix-sort
    // scratch, and a staged output
    pgh::dev_buf sk0, sk1, sv0, sv1, crowd, sort_tmp, out_staged;
    // a host thread's own workspace (pgh_fnds_thread_workspace): released
    // with its thread, never by pgh_fnds_destroy
    bool thread_owned = false;
};

namespace pgh
{
// The buffers of fnds_chain.hip for n points.
void chain_parts(pgh_fnds_ws *ws, uint32_t n, uint32_t m, std::vector<ws_part> &parts);
// Front offsets, items, ranks and the number of fronts of the n <= kChainMaxN
// points whose keys and dominator counts the workspace holds (fnds_chain.hip);
// the items of the fronts that start at or before `upto` only (n: all).
pgh_status launch_chain_fronts(pgh_fnds_ws *ws, hipStream_t s, uint32_t n, uint32_t m, uint32_t upto);
// The items again, for another `upto`.
pgh_status launch_chain_items(pgh_fnds_ws *ws, hipStream_t s, uint32_t n, uint32_t upto);
// Dominator counts (cnt32, zeroed before) from the keys and, with `lists`, D
// and its rows' bit counts (ndom32, zeroed before).
pgh_status launch_pairs(pgh_fnds_ws *ws, hipStream_t s, uint32_t n, uint32_t m, bool lists);
// dom_offsets, dom_count and scalars[1] from those counts, n <= kChainMaxN.
pgh_status launch_offsets(pgh_fnds_ws *ws, hipStream_t s, uint32_t n);
// pgh_fnds_run, where they cost extra without the domination lists (D,
// dom_offsets, dom_count) and the items of fronts that start after `upto`;
// pgh_fnds_sizes makes what is missing when asked.
pgh_status fnds_run(pgh_fnds_ws *ws, const double *objs, uint64_t n, uint64_t m, hipStream_t s, bool lists,
                    uint64_t upto);
// Makes the items that a run with a smaller `upto` left out.
pgh_status fnds_all_items(pgh_fnds_ws *ws);
} // namespace pgh
