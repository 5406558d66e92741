// fnds_chain.hip -- the fronts of fast_non_dominated_sorting
// (src/utils/multi_objective.cpp:228-254) for up to kChainMaxN points, without a
// grid-wide exchange per front.
//
// The reference peels front after front; the order inside front L + 1 is that
// in which its nested loop completes the elements: by the position in front L
// of an element's last dominator there, then by index.  Here the two halves of
// that are separated:
//
//   k_order    permutation by the number of dominators.  A dominator of an
//              element has strictly fewer dominators, so this order is
//              topological, and a point that is nowhere worse dominates exactly
//              when it has fewer dominators (equal points have equally many)
//   k_tiles    the dominance bits in that order, one 64-bit word per element
//              and block of 64 earlier elements
//   k_rank     rank = 1 + the largest rank of a dominator, block by block in one
//              workgroup
//   k_fronts,  the members of every front by index, and for every element the
//   k_slots,   bits of its dominators among the members of the front before
//   k_masks    its own
//   k_chain    front after front in one workgroup: the position of each
//              element's last dominator and the members' order by it
//   k_items    the fronts' elements in that order
//
// What stays serial is a few hundred instructions per 64 elements (k_rank) and
// per front (k_chain), on bits: the largest of a set of small numbers is found
// from their bit planes, a 64-bit AND per bit, with no loop over the set.
// Measured (8192 x 2 with 213 fronts; 16384 x 3 with 54): the peel's kernel took
// 1.16 and 0.75 ms, here k_rank takes 0.18 and 0.26 ms, k_chain 0.12 and 0.27 and
// the rest 0.08 and 0.15.  Both serial kernels are bound by the latency of one
// wavefront's dependent instructions.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <iterator>
#include <vector>

#include "fnds_ws.hpp"
#include "pgh_internal.hpp"

namespace pgh
{
namespace
{

constexpr uint32_t kBlock = 256, kWide = 1024;
constexpr uint32_t kRankBits = 14; // ranks and positions below kChainMaxN = 2^14
constexpr uint32_t kPlanes = 16;   // bit planes' stride: kRankBits, padded

// Exclusive scan over one workgroup of kWide threads; sh holds kWide / 64.
__device__ __forceinline__ uint32_t wide_exclusive_scan(uint32_t v, uint32_t *sh, uint32_t &total)
{
    const uint32_t lane = threadIdx.x & 63u, wid = threadIdx.x >> 6;
    uint32_t x = v;
#pragma unroll
    for (uint32_t d = 1; d < 64u; d <<= 1) {
        const uint32_t y = __shfl_up(x, d);
        if (lane >= d) x += y;
    }
    if (lane == 63u) sh[wid] = x;
    __syncthreads();
    if (wid == 0u) {
        uint32_t t = lane < kWide / 64u ? sh[lane] : 0u;
#pragma unroll
        for (uint32_t d = 1; d < kWide / 64u; d <<= 1) {
            const uint32_t y = __shfl_up(t, d);
            if (lane >= d) t += y;
        }
        if (lane < kWide / 64u) sh[lane] = t;
    }
    __syncthreads();
    total = sh[kWide / 64u - 1u];
    const uint32_t excl = (wid ? sh[wid - 1u] : 0u) + x - v;
    __syncthreads();
    return excl;
}

// bins[0 .. n) of counts -> their exclusive prefix, by one workgroup.
__device__ __forceinline__ void scan_bins(uint32_t *bins, uint32_t n, uint32_t *sh)
{
    const uint32_t per = (n + kWide - 1u) / kWide;
    const uint32_t b = min(threadIdx.x * per, n), e = min(b + per, n);
    uint32_t sum = 0u, total;
    for (uint32_t i = b; i < e; ++i) sum += bins[i];
    uint32_t o = wide_exclusive_scan(sum, sh, total);
    for (uint32_t i = b; i < e; ++i) {
        const uint32_t c = bins[i];
        bins[i] = o;
        o += c;
    }
    __syncthreads();
}

// use(i, load(i), true) for the workgroup's elements, kAtOnce loads in flight (one
// after another their latency is most of these kernels); every lane calls use, those
// past the end with false.
template <class Load, class Use>
__device__ __forceinline__ void in_batches(uint32_t n, Load load, Use use)
{
    constexpr uint32_t kAtOnce = 8;
    for (uint32_t b = 0; b < n; b += kAtOnce * kWide) {
        const uint32_t i0 = b + threadIdx.x;
        decltype(load(i0)) v[kAtOnce];
#pragma unroll
        for (uint32_t u = 0; u < kAtOnce; ++u) v[u] = load(min(i0 + u * kWide, n - 1u));
#pragma unroll
        for (uint32_t u = 0; u < kAtOnce; ++u) {
            if (b + u * kWide >= n) break; // uniform
            use(i0 + u * kWide, v[u], i0 + u * kWide < n);
        }
    }
}

// bins[k] += 1 for every lane that is `in`, and what was there.  One addition for the
// wavefront where all lanes have bin 0 (or, ANY, any one bin): 64 to one address take
// 64 turns (one front of 16384, whose counts are all zero: k_order 41 us).
template <bool ANY>
__device__ __forceinline__ uint32_t bin_add(uint32_t *bins, uint32_t k, bool in)
{
    uint32_t same = 0u;
    if constexpr (ANY) same = __builtin_amdgcn_readfirstlane(k); // (lanes past the end repeat the last element)
    if (__ballot(k != same) != 0u) return in ? atomicAdd(&bins[k], 1u) : 0u;
    const uint64_t who = __ballot(in);
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t old = 0u;
    if (lane == 0u && who) old = atomicAdd(&bins[same], static_cast<uint32_t>(__popcll(who)));
    return __builtin_amdgcn_readfirstlane(old) + static_cast<uint32_t>(__popcll(who & ((uint64_t(1) << lane) - 1u)));
}

// Every element's place in the order by dominator count (equal counts in any
// order; no result depends on it), and the number of those without dominators.
__global__ __launch_bounds__(kWide) void k_order(const uint32_t *__restrict__ cnt, uint32_t n,
                                                 uint32_t *__restrict__ place, uint64_t *__restrict__ n_free)
{
    extern __shared__ uint32_t bins[]; // n
    __shared__ uint32_t sh[kWide / 64u];
    for (uint32_t i = threadIdx.x; i < n; i += kWide) bins[i] = 0u;
    __syncthreads();
    in_batches(n, [&](uint32_t i) { return cnt[i]; },
               [&](uint32_t, uint32_t c, bool in) { bin_add<false>(bins, min(c, n - 1u), in); });
    __syncthreads();
    if (threadIdx.x == 0) *n_free = bins[0]; // (its next store is this thread's)
    scan_bins(bins, n, sh);
    in_batches(n, [&](uint32_t i) { return cnt[i]; },
               [&](uint32_t i, uint32_t c, bool in) {
                   const uint32_t at = bin_add<false>(bins, min(c, n - 1u), in);
                   if (in) place[i] = min(at, n - 1u);
               });
}

// The elements, their counts and their keys in that order (scattered here: one
// workgroup stores 64 scattered words no faster than one a cycle), and `first` cleared.
__global__ __launch_bounds__(kBlock) void k_scatter(const int64_t *__restrict__ keys,
                                                    const uint32_t *__restrict__ cnt,
                                                    const uint32_t *__restrict__ place, uint32_t n, uint32_t m,
                                                    uint32_t *__restrict__ perm, uint32_t *__restrict__ scnt,
                                                    int64_t *__restrict__ skeys, uint32_t *__restrict__ first)
{
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const uint32_t e = place[i];
    first[i] = 0u;
    perm[e] = i;
    scnt[e] = cnt[i];
    for (uint32_t q = 0; q < m; ++q) {
        skeys[static_cast<uint64_t>(e) * m + q] = keys[static_cast<uint64_t>(i) * m + q];
    }
}

// dom_offsets (n + 1) = exclusive prefix of ndom, dom_count widened, and
// scalars[1] = the total (below 2^27 for n <= kChainMaxN).
__global__ __launch_bounds__(kWide) void k_offsets(const uint32_t *__restrict__ ndom,
                                                   const uint32_t *__restrict__ cnt, uint32_t n,
                                                   uint64_t *__restrict__ offsets, uint64_t *__restrict__ dom_count,
                                                   uint64_t *__restrict__ scalars)
{
    extern __shared__ uint32_t bins[]; // n + 1
    __shared__ uint32_t sh[kWide / 64u];
    for (uint32_t i = threadIdx.x; i <= n; i += kWide) bins[i] = i < n ? ndom[i] : 0u;
    __syncthreads();
    scan_bins(bins, n + 1u, sh);
    for (uint32_t i = threadIdx.x; i <= n; i += kWide) {
        offsets[i] = bins[i];
        if (i < n) dom_count[i] = cnt[i];
    }
    if (threadIdx.x == 0) scalars[1] = bins[n];
}

// A point's keys and dominator count.
template <int MT>
struct point {
    int64_t k[MT];
    uint32_t cnt;
    __device__ __forceinline__ void load(const int64_t *__restrict__ keys, const uint32_t *__restrict__ counts,
                                         uint32_t i)
    {
        cnt = counts[i];
#pragma unroll
        for (int q = 0; q < MT; ++q) k[q] = keys[static_cast<uint64_t>(i) * MT + q];
    }
};

// a dominates b (pareto_dominance, multi_objective.cpp:97-113): nowhere worse,
// and not equal, which the counts tell.
template <int MT>
__device__ __forceinline__ bool dominates(const point<MT> &a, const point<MT> &b)
{
    bool le = a.cnt < b.cnt;
#pragma unroll
    for (int q = 0; q < MT; ++q) le &= a.k[q] <= b.k[q];
    return le;
}

// Lane `from`'s value, uniform.
__device__ __forceinline__ int64_t lane_i64(int64_t v, uint32_t from)
{
    const uint32_t lo = __builtin_amdgcn_readlane(static_cast<uint32_t>(v), from);
    const uint32_t hi = __builtin_amdgcn_readlane(static_cast<uint32_t>(static_cast<uint64_t>(v) >> 32), from);
    return static_cast<int64_t>((static_cast<uint64_t>(hi) << 32) | lo);
}

// Every unordered pair of 64-element blocks (I, J), I <= J, once, in the
// elements' own order: the dominator count of every element (cnt) and, with
// LISTS, the row-major bits D (bit j of row i: i dominates j) and their number
// per row (ndom).  A wavefront holds the rows of ROWS blocks I, one
// per lane and block, and takes J's elements one after another, whose keys are
// scalars: two 64-lane comparisons per objective give both directions.  Bound
// by the comparisons (64-bit, 2 m per 64 pairs).
template <int MT, bool LISTS, uint32_t ROWS>
__global__ __launch_bounds__(kBlock) void k_pairs(const int64_t *__restrict__ keys, uint32_t n, uint32_t m,
                                                  uint64_t *__restrict__ D, uint32_t words,
                                                  uint32_t *__restrict__ cnt, uint32_t *__restrict__ ndom)
{
    const uint32_t J = blockIdx.x, lane = threadIdx.x & 63u;
    const uint32_t I0 =
        (blockIdx.y * (kBlock / 64u) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * ROWS;
    if (I0 > J) return; // wavefront-uniform, no barrier below
    const uint32_t c0 = 64u * J, cols = min(64u, n - c0);
    int64_t row[ROWS][MT > 0 ? MT : 1];
    uint32_t by[ROWS];                      // dominators of the lane's rows
    uint64_t bits[ROWS], back[ROWS];   // the rows' words of block J; J's words of block I (lane c: c's)
    uint32_t col_by = 0u;                        // dominators of column `lane`
    bool there[ROWS], below[ROWS];
#pragma unroll
    for (uint32_t k = 0; k < ROWS; ++k) {
        const uint32_t r = min(64u * (I0 + k) + lane, n - 1u);
        if constexpr (MT > 0) {
#pragma unroll
            for (int q = 0; q < MT; ++q) row[k][q] = keys[static_cast<uint64_t>(r) * MT + q];
        }
        by[k] = 0u;
        bits[k] = back[k] = 0u;
        // rows past n (J's own block only) repeat row n - 1 and are left out
        there[k] = I0 + k < J || (I0 + k == J && lane < cols);
        below[k] = I0 + k < J;
    }
    int64_t mine[MT > 0 ? MT : 1]; // column `lane`
    if constexpr (MT > 0) {
#pragma unroll
        for (int q = 0; q < MT; ++q) mine[q] = keys[static_cast<uint64_t>(min(c0 + lane, n - 1u)) * MT + q];
    }
    // bit c of a row's word, from the top down: two halves of 32 columns
    uint32_t half[2][ROWS] = {};
#pragma unroll
    for (uint32_t h = 0; h < 2u; ++h) {
        for (uint32_t c = 32u * h; c < 32u * h + 32u; ++c) {
            if (c >= cols) { // uniform: J is the last, short block
#pragma unroll
                for (uint32_t k = 0; k < ROWS; ++k) half[h][k] *= 2u;
                continue;
            }
            int64_t col[MT > 0 ? MT : 1];
            if constexpr (MT > 0) {
#pragma unroll
                for (int q = 0; q < MT; ++q) col[q] = lane_i64(mine[q], c);
            }
            uint32_t dominators = 0u;
#pragma unroll
            for (uint32_t k = 0; k < ROWS; ++k) {
                // blocks past J (uniform) are computed and left out
                bool le = true, ge = true;
                if constexpr (MT > 0) {
#pragma unroll
                    for (int q = 0; q < MT; ++q) {
                        le &= row[k][q] <= col[q];
                        ge &= row[k][q] >= col[q];
                    }
                } else {
                    const uint32_t r = min(64u * (I0 + k) + lane, n - 1u);
                    const int64_t *a = keys + static_cast<uint64_t>(r) * m, *b = keys + static_cast<uint64_t>(c0 + c) * m;
                    for (uint32_t q = 0; q < m && (le || ge); ++q) {
                        le &= a[q] <= b[q];
                        ge &= a[q] >= b[q];
                    }
                }
                // row dominates column; the diagonal block holds both
                // directions, so there only this one counts
                const bool down = le && !ge && there[k];
                dominators += static_cast<uint32_t>(__popcll(__ballot(down)));
                if constexpr (LISTS) half[h][k] = 2u * half[h][k] + (down ? 1u : 0u);
                const bool up = ge && !le && below[k];
                by[k] += up ? 1u : 0u;
                if constexpr (LISTS) {
                    const uint64_t v = __ballot(up);
                    if (lane == c) back[k] = v;
                }
            }
            if (lane == c) col_by = dominators;
        }
    }
    if constexpr (LISTS) {
#pragma unroll
        for (uint32_t k = 0; k < ROWS; ++k) {
            bits[k] = __brev(half[0][k]) | (static_cast<uint64_t>(__brev(half[1][k])) << 32);
        }
    }
    uint32_t col_nd = 0u;
#pragma unroll
    for (uint32_t k = 0; k < ROWS; ++k) {
        const uint32_t I = I0 + k, r = 64u * I + lane;
        if (I > J) break;
        if constexpr (LISTS) {
            if (r < n) {
                D[static_cast<uint64_t>(r) * words + J] = bits[k];
                const uint32_t nd = static_cast<uint32_t>(__popcll(bits[k]));
                if (nd) atomicAdd(&ndom[r], nd);
            }
            if (I < J && lane < cols) {
                D[static_cast<uint64_t>(c0 + lane) * words + I] = back[k];
                col_nd += static_cast<uint32_t>(__popcll(back[k]));
            }
        }
        if (by[k]) atomicAdd(&cnt[r], by[k]); // I < J: r < n
    }
    if (lane < cols) {
        if (col_by) atomicAdd(&cnt[c0 + lane], col_by);
        if (LISTS && col_nd) atomicAdd(&ndom[c0 + lane], col_nd);
    }
}

__device__ __forceinline__ uint64_t tile_at(uint32_t J, uint32_t I)
{
    return (static_cast<uint64_t>(J) * (J + 1u) / 2u + I) * 64u;
}

// Block J has no element with a dominator (the first n_free have none).  Such blocks, a
// front's worth of them, are not worth a tile nor a step of k_rank: one front of 16384
// points took k_rank 235 us, and k_tiles 51.
__device__ __forceinline__ bool block_is_free(uint64_t n_free, uint32_t n, uint32_t J)
{
    return min(64u * J + 63u, n - 1u) < n_free;
}

// Word c of tile (J, I), I <= J: the dominators of element 64 J + c (in perm's
// order) among elements 64 I .. 64 I + 63.  A wavefront holds a block of rows,
// one per lane and block, and takes the columns of J one after another, whose keys
// are scalars: the word is the ballot of the comparison.
template <int MT, uint32_t ROWS>
__global__ __launch_bounds__(kBlock) void k_tiles(const int64_t *__restrict__ skeys,
                                                  const uint32_t *__restrict__ scnt, uint32_t n,
                                                  const uint64_t *__restrict__ n_free,
                                                  uint64_t *__restrict__ tiles)
{
    const uint32_t J = blockIdx.x, lane = threadIdx.x & 63u;
    const uint32_t I0 = (blockIdx.y * (kBlock / 64u) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * ROWS;
    if (I0 > J) return; // wavefront-uniform, no barrier below
    const uint32_t c0 = 64u * J, cols = min(64u, n - c0);
    if (block_is_free(*n_free, n, J)) return; // no word of it is read
    uint64_t out[ROWS];
    point<MT> row[ROWS];
#pragma unroll
    for (uint32_t k = 0; k < ROWS; ++k) {
        const uint32_t r = 64u * (I0 + k) + lane;
        row[k].load(skeys, scnt, min(r, n - 1u));
        if (r >= n) row[k].cnt = 0xffffffffu; // dominates nothing
        out[k] = 0u;
    }
    constexpr uint32_t kBatch = ROWS > 1u ? 4u : 8u; // columns whose scalars are loaded together
    for (uint32_t cb = 0; cb < cols; cb += kBatch) {
        point<MT> col[kBatch];
#pragma unroll
        for (uint32_t u = 0; u < kBatch; ++u) col[u].load(skeys, scnt, c0 + min(cb + u, cols - 1u));
#pragma unroll
        for (uint32_t u = 0; u < kBatch; ++u) {
#pragma unroll
            for (uint32_t k = 0; k < ROWS; ++k) {
                const uint64_t w = __ballot(dominates<MT>(row[k], col[u]));
                if (lane == cb + u) out[k] = w; // (past cols: the last column's word again, in lanes not read)
            }
        }
    }
#pragma unroll
    for (uint32_t k = 0; k < ROWS; ++k) {
        if (I0 + k <= J) tiles[tile_at(J, I0 + k) + lane] = lane < cols ? out[k] : 0u;
    }
}

// The largest number whose bit is set in `word` (0 for none), numbers given by
// their bit planes: number q has bit b when bit q of planes[b] is set.  BITS
// planes from the highest down, each an AND and a selection.
template <uint32_t BITS>
__device__ __forceinline__ uint32_t plane_max_n(uint64_t word, const uint64_t *__restrict__ planes)
{
    uint64_t p[BITS];
#pragma unroll
    for (uint32_t b = 0; b < BITS; ++b) p[b] = planes[b];
    uint32_t v = 0u;
#pragma unroll
    for (uint32_t b = BITS; b-- > 0u;) {
        const uint64_t t = word & p[b];
        const bool some = t != 0u;
        word = some ? t : word;
        v = 2u * v + (some ? 1u : 0u);
    }
    return v;
}
// planes of numbers below 2^bits (uniform), zero from there on
__device__ __forceinline__ uint32_t plane_max(uint64_t word, const uint64_t *__restrict__ planes, uint32_t bits)
{
    if (bits <= 6u) return plane_max_n<6u>(word, planes);
    if (bits <= 8u) return plane_max_n<8u>(word, planes);
    if (bits <= 10u) return plane_max_n<10u>(word, planes);
    return plane_max_n<kRankBits>(word, planes);
}

__device__ __forceinline__ uint32_t bits_of(uint32_t v) // bits needed for values up to v
{
    return 32u - static_cast<uint32_t>(__clz(static_cast<int>(v)));
}

// The maximum over the wavefront, uniform (data-parallel moves: no LDS).
__device__ __forceinline__ uint32_t wave_max(uint32_t v)
{
#define PGH_DPP_MAX(ctrl) v = max(v, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, v, ctrl, 0xf, 0xf, false)))
    PGH_DPP_MAX(0x111); // row_shr:1
    PGH_DPP_MAX(0x112); // row_shr:2
    PGH_DPP_MAX(0x114); // row_shr:4
    PGH_DPP_MAX(0x118); // row_shr:8
    PGH_DPP_MAX(0x142); // row_bcast:15
    PGH_DPP_MAX(0x143); // row_bcast:31
#undef PGH_DPP_MAX
    return __builtin_amdgcn_readlane(v, 63);
}

// Lane b < kPlanes gets the ballot of bit b of r (b < BITS; zero above).
template <uint32_t BITS>
__device__ __forceinline__ uint64_t planes_by_lane(uint32_t r, uint32_t lane)
{
    uint64_t mine = 0u;
#pragma unroll
    for (uint32_t b = 0; b < BITS; ++b) {
        const uint64_t p = __ballot((r >> b) & 1u);
        if (lane == b) mine = p;
    }
    return mine;
}

// r = max(r, 1 + r of every dominator in the block's own tile), to a fixed
// point: as many rounds as the longest chain inside the block (a few: blocks
// hold points of like dominator counts).  For ranks below 2^BITS at the end
// (a larger one is returned as such).  Returns the planes (planes_by_lane).
template <uint32_t BITS>
__device__ __forceinline__ uint64_t settle_block(uint32_t &r, uint64_t own, uint32_t lane)
{
    for (;;) {
        uint64_t word = own, mine = 0u;
        uint32_t v = 0u;
#pragma unroll
        for (uint32_t b = BITS; b-- > 0u;) {
            const uint64_t p = __ballot((r >> b) & 1u);
            const uint64_t t = word & p;
            const bool some = t != 0u;
            word = some ? t : word;
            v = 2u * v + (some ? 1u : 0u);
            if (lane == b) mine = p;
        }
        const bool up = own != 0u && v >= r;
        if (__ballot(up) == 0u) return mine;
        if (up) r = v + 1u;
        if (__ballot(r >> BITS) != 0u) return 0u;
    }
}

// Ranks of blocks J0 .. J1 - 1 of 64 elements (in perm's order), block after
// block in one workgroup; `base` holds what the blocks before J0 give (k_far).
// Wavefront 0 finishes block J: from base, what the others collected (rr) from
// blocks J0 .. J - 2 while it finished J - 1, the tile (J, J - 1) and the
// block's own tile.  Meanwhile the others collect for block J + 1; a tile whose
// block has no rank that could raise any of the 64 is skipped.  Tiles are loaded
// two blocks ahead.  Blocks without dominators, which come first, are of rank 0
// and only entered; the others then collect for the first block that is none before
// wavefront 0 begins with it.
constexpr uint32_t kSpan = 32; // blocks per launch at most
__global__ __launch_bounds__(kWide) void k_rank(const uint64_t *__restrict__ tiles, uint32_t n, uint32_t J0,
                                                uint32_t J1, const uint32_t *__restrict__ base,
                                                uint32_t *__restrict__ rank, uint64_t *__restrict__ planes_out,
                                                uint32_t *__restrict__ top_out, const uint64_t *__restrict__ n_free)
{
    __shared__ __align__(16) uint64_t planes[kSpan * kPlanes];
    __shared__ uint32_t top[kSpan];
    __shared__ uint32_t rr[2][64];
    const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (threadIdx.x < 128u) (&rr[0][0])[threadIdx.x] = 0u;
    __syncthreads();
    constexpr uint32_t kCollect = kWide / 64u - 1u, kTilesEach = (kSpan + kCollect - 1u) / kCollect;
    // wavefront 0: own tile, the one before it and base of blocks J and J + 1;
    // the others: their tiles of blocks J + 1 and J + 2, block J' - 1 - wave and
    // kCollect steps further back
    uint64_t w[2][kTilesEach];
    uint32_t bs[2] = {0u, 0u};
    static_assert(kTilesEach >= 2u, "wavefront 0 uses two slots");
    // (inlined everywhere, so that the slots stay registers)
    const auto fetch = [&](uint32_t J, uint32_t slot) __attribute__((always_inline)) {
        if (wave == 0u) {
            w[slot][0] = J < J1 ? tiles[tile_at(J, J) + lane] : 0u;
            w[slot][1] = J < J1 && J > J0 ? tiles[tile_at(J, J - 1u) + lane] : 0u;
            bs[slot] = base && J < J1 ? base[min(64u * J + lane, n - 1u)] : 0u;
        } else {
#pragma unroll
            for (uint32_t g = 0; g < kTilesEach; ++g) {
                const uint32_t back = wave + 1u + kCollect * g;
                w[slot][g] = J < J1 && J0 + back <= J ? tiles[tile_at(J, J - back) + lane] : 0u;
            }
        }
    };
    // what blocks J0 .. T - 2 give block T, by the wavefronts but the first; the slot
    // then takes block T + 2
    const auto collect = [&](uint32_t T, uint32_t slot) __attribute__((always_inline)) {
        uint32_t r = 0u;
#pragma unroll
        for (uint32_t g = 0; g < kTilesEach; ++g) {
            const uint32_t back = wave + 1u + kCollect * g;
            if (J0 + back > T) continue;
            const uint32_t k = T - back - J0, tk = top[k];
            const uint64_t word = w[slot][g];
            if (__ballot(word != 0u && tk >= r) == 0u) continue;
            const uint32_t v = plane_max(word, planes + k * kPlanes, bits_of(tk)) + 1u;
            if (word) r = max(r, v);
        }
        fetch(T + 2u, slot);
        if (r) atomicMax(&rr[T & 1u][lane], r);
    };
    const auto step = [&](uint32_t J, uint32_t slot) __attribute__((always_inline)) {
        if (wave == 0u) {
            const uint64_t own = w[slot][0], before = w[slot][1];
            const uint32_t e = 64u * J + lane;
            uint32_t r = max(rr[J & 1u][lane], bs[slot]);
            rr[J & 1u][lane] = 0u;
            fetch(J + 2u, slot);
            if (J > J0) {
                const uint32_t k = J - 1u - J0;
                const uint32_t v = plane_max(before, planes + k * kPlanes, bits_of(top[k])) + 1u;
                if (before) r = max(r, v);
            }
            if (e >= n) r = 0u;
            // a rank rises by the longest chain inside the block, a few: bits
            // for 8 more first, for 63 more if that was not enough
            const uint32_t r0 = r, m0 = wave_max(r);
            uint64_t p = 0u;
            for (uint32_t more = 8u;; more = 63u) {
                r = r0;
                const uint32_t most = m0 + more;
                if (most < 64u) p = settle_block<6u>(r, own, lane);
                else if (most < 256u) p = settle_block<8u>(r, own, lane);
                else if (most < 1024u) p = settle_block<10u>(r, own, lane);
                else p = settle_block<kRankBits>(r, own, lane);
                if (more == 63u || __ballot(r > most) == 0u) break;
            }
            const uint32_t big = wave_max(r);
            if (lane < kPlanes) {
                planes[(J - J0) * kPlanes + lane] = p;
                planes_out[static_cast<uint64_t>(J) * kPlanes + lane] = p;
            }
            if (lane == 0u) {
                top[J - J0] = big;
                top_out[J] = big;
            }
            if (e < n) rank[e] = r;
        } else if (J + 1u < J1) {
            collect(J + 1u, slot);
        }
        __syncthreads();
    };
    // wavefront 0 holds blocks J and J + 1, the others J + 1 and J + 2
    fetch(wave == 0u ? J0 : J0 + 1u, 0u);
    fetch(wave == 0u ? J0 + 1u : J0 + 2u, 1u);
    // the first block with a dominator, or J1 (looked at while those are in flight)
    const uint64_t free_now = *n_free;
    const uint32_t Js = free_now >= n ? J1 : min(max(static_cast<uint32_t>(free_now) / 64u, J0), J1);
    if (Js > J0) { // uniform
        for (uint32_t x = threadIdx.x; x < (Js - J0) * kPlanes; x += kWide) {
            planes[x] = 0u;
            planes_out[static_cast<uint64_t>(J0) * kPlanes + x] = 0u;
        }
        if (threadIdx.x < Js - J0) top[threadIdx.x] = top_out[J0 + threadIdx.x] = 0u;
        for (uint32_t e = 64u * J0 + threadIdx.x; e < min(64u * Js, n); e += kWide) rank[e] = 0u;
        __syncthreads();
        if (Js >= J1) return;
        if (wave == 0u) {
            fetch(Js, 0u);
            fetch(Js + 1u, 1u);
        } else {
            fetch(Js, 1u);
            fetch(Js + 1u, 0u);
            collect(Js, 1u);
        }
        __syncthreads();
    }
    for (uint32_t J = Js; J < J1; J += 2u) {
        step(J, 0u);
        if (J + 1u < J1) step(J + 1u, 1u);
    }
}

// base[e] = max(base[e], 1 + the largest rank of e's dominators in blocks
// I0 .. I1 - 1), for the elements of blocks J1 + blockIdx.x: a workgroup per
// block, its eight wavefronts sharing the (at most kSpan) tiles.
constexpr uint32_t kFarBlock = 512;
__global__ __launch_bounds__(kFarBlock) void k_far(const uint64_t *__restrict__ tiles, uint32_t n, uint32_t I0,
                                                   uint32_t I1, const uint64_t *__restrict__ planes,
                                                   const uint32_t *__restrict__ top, uint32_t *__restrict__ base,
                                                   uint32_t first, const uint64_t *__restrict__ n_free)
{
    __shared__ uint32_t rr[64];
    const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t J = I1 + blockIdx.x, e = 64u * J + lane;
    if (block_is_free(*n_free, n, J)) return; // uniform; its base is not read
    if (threadIdx.x < 64u) rr[lane] = 0u;
    __syncthreads();
    uint32_t r = 0u;
    for (uint32_t k = I1 - I0; k-- > 0u;) { // the nearest blocks hold the larger ranks
        if (k % (kFarBlock / 64u) != wave) continue;
        const uint32_t I = I0 + k, tI = top[I];
        const uint64_t word = tiles[tile_at(J, I) + lane];
        if (__ballot(word != 0u && tI >= r) == 0u) continue;
        const uint32_t v = plane_max(word, planes + static_cast<uint64_t>(I) * kPlanes, bits_of(tI)) + 1u;
        if (word) r = max(r, v);
    }
    if (r) atomicMax(&rr[lane], r);
    __syncthreads();
    if (threadIdx.x < 64u && e < n) base[e] = first ? rr[lane] : max(base[e], rr[lane]);
}

// Front offsets (32 and 64 bits), the offset of each front's words of k_masks (and at n
// the most members of a front but the first), the number of fronts, the elements' ranks by index and the members of every
// front in any order.
__global__ __launch_bounds__(kWide) void k_fronts(const uint32_t *__restrict__ srank,
                                                  const uint32_t *__restrict__ perm, uint32_t n,
                                                  uint32_t *__restrict__ fo, uint64_t *__restrict__ front_offsets,
                                                  uint64_t *__restrict__ wbase, uint32_t *__restrict__ rank,
                                                  uint32_t *__restrict__ any, uint64_t *__restrict__ scalars)
{
    extern __shared__ uint32_t bins[]; // n + 1
    __shared__ uint32_t sh[kWide / 64u], s_fronts, s_large;
    const uint32_t t = threadIdx.x;
    for (uint32_t i = t; i <= n; i += kWide) bins[i] = 0u;
    if (t == 0) s_fronts = s_large = 0u;
    __syncthreads();
    uint32_t big = 0u;
    in_batches(n, [&](uint32_t e) { return min(srank[e], n - 1u); },
               [&](uint32_t, uint32_t r, bool in) {
                   big = in ? max(big, r + 1u) : big;
                   bin_add<true>(bins, r, in);
               });
    atomicMax(&s_fronts, big);
    __syncthreads();
    const uint32_t F = s_fronts; // no front below F is empty
    scan_bins(bins, F + 1u, sh);
    for (uint32_t f = t; f <= F; f += kWide) {
        fo[f] = bins[f];
        front_offsets[f] = bins[f];
    }
    // words of front f: its size times the words of the front before it
    {
        const uint32_t per = (F + kWide - 1u) / kWide;
        const uint32_t b = min(t * per, F), e = min(b + per, F);
        const auto words = [&](uint32_t f) {
            return f ? (bins[f + 1u] - bins[f]) * ((bins[f] - bins[f - 1u] + 63u) / 64u) : 0u;
        };
        uint32_t sum = 0u, total; // at most n + n^2 / 256
        for (uint32_t f = b; f < e; ++f) sum += words(f);
        uint32_t o = wide_exclusive_scan(sum, sh, total), most = 0u;
        for (uint32_t f = b; f < e; ++f) {
            wbase[f] = o;
            o += words(f);
            if (f) most = max(most, bins[f + 1u] - bins[f]);
        }
        most = wave_max(most);
        if ((t & 63u) == 0u && most) atomicMax(&s_large, most);
    }
    if (t == 0) scalars[0] = F;
    __syncthreads();
    if (t == 0) wbase[n] = s_large; // (a place of no front's)
    in_batches(n, [&](uint32_t e) { return make_uint2(min(srank[e], n - 1u), perm[e]); },
               [&](uint32_t, uint2 v, bool in) {
                   const uint32_t at = bin_add<true>(bins, v.x, in);
                   if (in) {
                       rank[v.y] = v.x;
                       any[min(at, n - 1u)] = v.y;
                   }
               });
}

// members: every front's elements by index.  A wavefront per element counts the
// smaller ones, in a front of up to kBigFront.  In a larger one (at most three) a
// wavefront per 64 indices counts them in the ranks of all smaller indices, once for
// all its elements of that front: one front of 16384 took 126 us element by element.
constexpr uint32_t kBigFront = 4096;
__global__ __launch_bounds__(kBlock) void k_slots(const uint32_t *__restrict__ any, const uint32_t *__restrict__ rank,
                                                  const uint32_t *__restrict__ fo, uint32_t n, uint32_t big_groups,
                                                  uint32_t *__restrict__ members)
{
    const uint32_t lane = threadIdx.x & 63u;
    if (blockIdx.x >= big_groups) {
        const uint32_t x = (blockIdx.x - big_groups) * (kBlock / 64u) + (threadIdx.x >> 6);
        if (x >= n) return;
        const uint32_t i = any[x], f = rank[i], a = fo[f], b = fo[f + 1u];
        if (b - a > kBigFront) return;
        uint32_t slot = 0u;
        for (uint32_t q = a; q < b; q += 64u) {
            const uint32_t o = q + lane;
            slot += static_cast<uint32_t>(__popcll(__ballot(o < b && any[min(o, b - 1u)] < i)));
        }
        if (lane == 0u) members[a + slot] = i;
        return;
    }
    // (these workgroups first: theirs is the longer chain)
    const uint32_t x = blockIdx.x * (kBlock / 64u) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (64u * x >= n) return;
    const uint32_t i = 64u * x + lane, r = rank[min(i, n - 1u)];
    uint64_t todo = __ballot(i < n && fo[r + 1u] - fo[r] > kBigFront);
    while (todo) { // uniform
        const uint32_t f = __builtin_amdgcn_readlane(r, static_cast<uint32_t>(__builtin_ctzll(todo)));
        const uint64_t mine = __ballot(i < n && r == f);
        uint32_t before = 0u;
        constexpr uint32_t kAtOnce = 16;
        for (uint32_t q0 = 0; q0 < x; q0 += kAtOnce) {
            uint32_t v[kAtOnce];
#pragma unroll
            for (uint32_t u = 0; u < kAtOnce; ++u) v[u] = rank[64u * min(q0 + u, x - 1u) + lane];
#pragma unroll
            for (uint32_t u = 0; u < kAtOnce; ++u) {
                before += static_cast<uint32_t>(__popcll(__ballot(q0 + u < x && v[u] == f)));
            }
        }
        if (i < n && r == f) {
            members[fo[f] + before + static_cast<uint32_t>(__popcll(mine & ((uint64_t(1) << lane) - 1u)))] = i;
        }
        todo &= ~mine;
    }
}

// k_masks for a front of more than kWide members: a wavefront takes 64 of them, one per
// lane, and kTileWords words of the front before, whose members it loads 64 at a time
// and broadcasts.  Of the second front the words are not kept: the first front's
// positions are its members' places, so the position of a member's last dominator
// there, all that k_chain wants of them, is its highest bit (`first`, by place).
constexpr uint32_t kTileWords = 2;
template <int MT>
__device__ __forceinline__ void masks_of_large(const int64_t *__restrict__ keys, const uint32_t *__restrict__ cnt,
                                               const uint32_t *__restrict__ members,
                                               const uint32_t *__restrict__ rank, const uint32_t *__restrict__ fo,
                                               const uint64_t *__restrict__ wbase, uint32_t n, uint32_t b, uint32_t w0,
                                               uint64_t *__restrict__ masks, uint32_t *__restrict__ first)
{
    const uint32_t lane = threadIdx.x & 63u, x = 64u * b + lane;
    if (64u * b >= n) return;
    const uint32_t i = members[min(x, n - 1u)], f = rank[i], a = fo[f], size = fo[f + 1u] - a;
    const uint32_t pa = f ? fo[f - 1u] : a; // the front before: pa .. a - 1
    uint64_t todo = __ballot(x < n && f > 0u && size > kWide && 64u * w0 < a - pa);
    if (todo == 0u) return;
    point<MT> mine;
    mine.load(keys, cnt, i);
    const uint64_t base = wbase[f];
    while (todo) { // the 64 members' fronts in turn, uniform
        const uint32_t lead = static_cast<uint32_t>(__builtin_ctzll(todo));
        const uint32_t ff = __builtin_amdgcn_readlane(f, lead), fa = __builtin_amdgcn_readlane(a, lead);
        const uint32_t fp = __builtin_amdgcn_readlane(pa, lead);
        const bool on = ((todo >> lane) & 1u) && f == ff;
        todo &= ~__ballot(on);
        const uint32_t words = min((fa - fp + 63u) / 64u, w0 + kTileWords);
        uint32_t last = 0u;
        for (uint32_t w = w0; w < words; ++w) {
            const uint32_t q = fp + 64u * w, there = min(64u, fa - q);
            point<MT> other;
            other.load(keys, cnt, members[min(q + lane, fa - 1u)]);
            uint32_t half[2] = {0u, 0u}; // bit u from the top down
#pragma unroll
            for (uint32_t h = 0; h < 2u; ++h) {
#pragma unroll 4
                for (uint32_t u = 32u * h; u < 32u * h + 32u; ++u) {
                    point<MT> one;
                    one.cnt = __builtin_amdgcn_readlane(other.cnt, u);
#pragma unroll
                    for (int k = 0; k < MT; ++k) one.k[k] = lane_i64(other.k[k], u);
                    half[h] = 2u * half[h] + (u < there && dominates<MT>(one, mine) ? 1u : 0u);
                }
            }
            const uint64_t bits = __brev(half[0]) | (static_cast<uint64_t>(__brev(half[1])) << 32);
            if (ff == 1u) {
                last = bits ? 64u * w + 63u - static_cast<uint32_t>(__clzll(static_cast<long long>(bits))) : last;
            } else if (on) {
                masks[base + static_cast<uint64_t>(w) * size + (x - a)] = bits;
            }
        }
        if (on && last) atomicMax(&first[x], last);
    }
}

// For every element of a front but the first: the bits of its dominators among
// the members of the front before, word w of member c of front f at
// wbase[f] + w * size + c.  A wavefront per element, which reads the front before;
// for fronts of more than kWide members (n > 2 kWide) the first large_x * large_y
// workgroups, which read it once per 64 elements (fronts of 5701, 3636, 2603, ...
// element by element: 124 us).
template <int MT>
__global__ __launch_bounds__(kBlock) void k_masks(const int64_t *__restrict__ keys, const uint32_t *__restrict__ cnt,
                                                  const uint32_t *__restrict__ members,
                                                  const uint32_t *__restrict__ rank, const uint32_t *__restrict__ fo,
                                                  const uint64_t *__restrict__ wbase, uint32_t n, uint32_t large_x,
                                                  uint32_t large_y, uint64_t *__restrict__ masks,
                                                  uint32_t *__restrict__ first)
{
    const uint32_t lane = threadIdx.x & 63u;
    if (blockIdx.x < large_x * large_y) {
        if (wbase[n] <= kWide) return; // no such front
        const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        for (uint32_t w0 = blockIdx.x / large_x * kTileWords; 64u * w0 < n; w0 += large_y * kTileWords) {
            masks_of_large<MT>(keys, cnt, members, rank, fo, wbase, n, blockIdx.x % large_x * (kBlock / 64u) + wave, w0,
                               masks, first);
        }
        return;
    }
    const uint32_t x = (blockIdx.x - large_x * large_y) * (kBlock / 64u) + (threadIdx.x >> 6);
    if (x >= n) return;
    const uint32_t i = members[x], f = rank[i];
    if (f == 0u) return;
    const uint32_t a = fo[f], size = fo[f + 1u] - a, pa = fo[f - 1u];
    if (large_y && size > kWide) return;
    point<MT> mine, other;
    mine.load(keys, cnt, i);
    for (uint32_t q = pa, w = 0u; q < a; q += 64u, ++w) {
        const uint32_t o = q + lane;
        other.load(keys, cnt, members[min(o, a - 1u)]);
        const uint64_t bits = __ballot(o < a && dominates<MT>(other, mine));
        if (lane == 0u) masks[wbase[f] + static_cast<uint64_t>(w) * size + (x - a)] = bits;
    }
}

// Bitonic sort of sh[0 .. P), P a power of two, by one workgroup.  Exchanges
// over at most 64 places stay within a wavefront's own 128.
__device__ __forceinline__ void wide_bitonic_sort(uint32_t *sh, uint32_t P)
{
    for (uint32_t k = 2; k <= P; k <<= 1) {
        for (uint32_t j = k >> 1; j > 0; j >>= 1) {
            for (uint32_t i = threadIdx.x; i < P / 2u; i += kWide) {
                const uint32_t x = 2u * i - (i & (j - 1u)), y = x + j;
                const uint32_t a = sh[x], b = sh[y];
                if ((a > b) == ((x & k) == 0u)) {
                    sh[x] = b;
                    sh[y] = a;
                }
            }
            if (j > 64u || (j == 1u && k >= 128u)) __syncthreads(); // (then the next exchange is over k > 64)
            else wave_lds_fence();
        }
    }
    __syncthreads();
}

// A member's place (value v) among 64 members whose values have the planes q,
// `same` at first those that exist: the members with a smaller value, and those
// of `below` (the smaller slots) with the same, bit by bit.
template <uint32_t BITS>
__device__ __forceinline__ uint32_t place_in_word(uint32_t v, const uint64_t (&q)[BITS], uint64_t same, uint64_t below)
{
    uint64_t less = 0u;
#pragma unroll
    for (uint32_t b = BITS; b-- > 0u;) {
        const bool one = (v >> b) & 1u;
        less |= one ? same & ~q[b] : 0u;
        same &= one ? q[b] : ~q[b];
    }
    return static_cast<uint32_t>(__popcll(less)) + static_cast<uint32_t>(__popcll(same & below));
}
// ... of member x among the c of its front in blocks first, first + step, ...
template <uint32_t BITS>
__device__ __forceinline__ uint32_t place_among(uint32_t v, uint32_t x, uint32_t c, uint32_t first, uint32_t step,
                                                const uint64_t *__restrict__ vp)
{
    uint32_t pos = 0u;
    for (uint32_t w = first; 64u * w < c; w += step) {
        uint64_t q[BITS];
#pragma unroll
        for (uint32_t b = 0; b < BITS; ++b) q[b] = vp[w * kPlanes + b];
        const uint32_t left = c - 64u * w;
        const uint64_t valid = left >= 64u ? ~uint64_t(0) : (uint64_t(1) << left) - 1u;
        const uint64_t below = x >= 64u * w + 64u ? ~uint64_t(0)
                                                  : (x < 64u * w ? uint64_t(0) : (uint64_t(1) << (x & 63u)) - 1u);
        pos += place_in_word<BITS>(v, q, valid, below);
    }
    return pos;
}

// The largest number below 2^BITS whose bit is set in word, from planes held by
// the wavefront.
template <uint32_t BITS>
__device__ __forceinline__ uint32_t held_max(uint64_t word, const uint64_t (&p)[BITS])
{
    uint32_t v = 0u;
#pragma unroll
    for (uint32_t b = BITS; b-- > 0u;) {
        const uint64_t h = word & p[b];
        const bool some = h != 0u;
        word = some ? h : word;
        v = 2u * v + (some ? 1u : 0u);
    }
    return v;
}

// The members' positions in their fronts, front after front: the position of
// each member's last dominator from the bit planes of the front before, its own
// as the number of members with a smaller (that position, slot), again bit by
// bit, and from it the planes for the next front.
//  - A run of fronts of at most 128 members is done by wavefront 0 alone, lane l
//    members l and l + 64, with no barrier: 0.45 us for a front of at most 64,
//    (a front took 1.9 us with the whole workgroup).  Their words are staged in
//    LDS by the workgroup first, up to kStage at a time.
//  - A front of up to kWide members is shared among the wavefronts, with two to
//    four barriers; the first kAhead words per member and wavefront are loaded
//    while the front before is ordered.
//  - Beyond, where comparing all with all would cost more than its barriers, the
//    members are put in bins by the position of their last dominator and only
//    compared there.  Words of at most kFewBits bits in every member, as in fronts of
//    which each member has few dominators, are read bit by bit instead of plane by
//    plane (about 10 instructions a bit, 90 for 14 planes), and others only where the
//    largest position of their 64 is above a member's so far: with many dominators a
//    member that leaves a handful (from the last word on, since the first front's
//    positions ascend).
constexpr uint32_t kStage = 2048, kAhead = 8, kWaves = kWide / 64u, kBin = 64;
constexpr int kFewBits = 5;
__global__ __launch_bounds__(kWide) void k_chain(const uint32_t *__restrict__ fo, const uint64_t *__restrict__ masks,
                                                 uint64_t mask_words, uint32_t upto,
                                                 const uint64_t *__restrict__ scalars, uint32_t n, uint32_t P,
                                                 const uint32_t *__restrict__ first, uint32_t *__restrict__ pos_out)
{
    extern __shared__ __align__(16) uint64_t lds64[];
    const uint32_t W = (n + 63u) / 64u;
    uint64_t *planes = lds64;                                   // [W][kPlanes]
    uint32_t *F = reinterpret_cast<uint32_t *>(planes + kPlanes * W); // P + 64: members, then bins
    // a run's words, or a large front's slots by bin (max(2 P, 8 kStage) bytes)
    uint64_t *stage = reinterpret_cast<uint64_t *>(F + P + 64u);
    uint16_t *list = reinterpret_cast<uint16_t *>(stage);
    // s_words, a run's words, is stored by wavefront 0 alone, before the barrier that
    // ends a run; its next store lies behind the barriers of the next run, so every
    // wavefront has read it.  (s_run, which a next front stores at once, would not do.)
    __shared__ uint32_t fs[kWide + 2u], s_run, s_words, s_scan[kWide / 64u];
    __shared__ __align__(16) uint64_t vplanes[kWaves * kPlanes];
    __shared__ uint32_t s_v[kWide], s_pos[kWide]; // zero between fronts
    __shared__ uint16_t s_top[kChainMaxN / 64u];
    const uint32_t t = threadIdx.x, lane = t & 63u, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    // the fronts that start at or before `upto`
    uint32_t fronts = min(static_cast<uint32_t>(scalars[0]), n);
    if (upto < n) {
        uint32_t lo = 0u; // fo[lo] <= upto < fo[fronts]
        while (fronts - lo > 1u) {
            const uint32_t mid = (lo + fronts) / 2u;
            if (fo[mid] <= upto) lo = mid;
            else fronts = mid;
        }
    }
    s_v[t] = s_pos[t] = 0u;
    // front 0: ascending indices
    {
        const uint32_t s = fo[1];
        for (uint32_t x = t; x < s; x += kWide) pos_out[x] = x;
        for (uint32_t w = wave; w < (s + 63u) / 64u; w += kWide / 64u) {
            const uint64_t p = planes_by_lane<kRankBits>(min(64u * w + lane, s - 1u), lane);
            if (lane < kPlanes) planes[w * kPlanes + lane] = p;
        }
    }
    uint64_t ahead[kAhead]; // the first words of member t of front `ahead_of`
    uint32_t ahead_of = 0u;
    uint32_t L = 1, L0 = 1; // fs holds the offsets of fronts L0 - 1 .. L0 + kWide
    uint64_t wb = 0u;       // front L's words in masks
    bool load = true;
    while (L < fronts) {
        if (load) {
            __syncthreads();
            L0 = L;
            fs[t] = fo[min(L0 - 1u + t, fronts)];
            if (t < 2u) fs[kWide + t] = fo[min(L0 - 1u + kWide + t, fronts)];
            load = false;
            __syncthreads();
        }
        uint32_t run = 0u;
        {
            const uint32_t *q = fs + (L - L0);
            const bool small = q[1] - q[0] <= 128u && q[2] - q[1] <= 128u;
            if (__builtin_amdgcn_readfirstlane(small ? 1u : 0u)) {
                if (t == 0) s_run = kWide;
                __syncthreads();
                // how many fronts from L on are small together with the one
                // before, with at most kStage words (two per member) in all
                const uint32_t f = L + t;
                bool stop = f >= fronts || f >= L0 + kWide;
                if (!stop) {
                    q = fs + (f - L0);
                    stop = q[1] - q[0] > 128u || q[2] - q[1] > 128u || 2u * (q[2] - fs[L - L0 + 1u]) > kStage;
                }
                const uint64_t stops = __ballot(stop);
                if (stops && lane == 0u) {
                    atomicMin(&s_run, 64u * wave + static_cast<uint32_t>(__builtin_ctzll(stops)));
                }
                __syncthreads();
                run = __builtin_amdgcn_readfirstlane(s_run);
            }
        }
        const uint32_t *fl = fs + (L - L0); // fl[0], fl[1], fl[2]: offsets of L - 1, L, L + 1
        if (run > 0u) {
            const uint64_t *src = masks + wb;
            const uint32_t words = static_cast<uint32_t>(
                min(static_cast<uint64_t>(2u * (fl[run + 1u] - fl[1])), mask_words - wb)); // at least the run's
            for (uint32_t x = t; x < words; x += kWide) stage[x] = src[x];
            __syncthreads();
            if (wave == 0u) {
                uint64_t p0[7], p1[7];
                uint32_t prev = fl[1] - fl[0], at = fl[1], end = fl[2], off = 0u;
#pragma unroll
                for (uint32_t b = 0; b < 7u; ++b) {
                    p0[b] = planes[b];
                    p1[b] = prev > 64u ? planes[kPlanes + b] : 0u;
                }
                uint64_t word = stage[min(lane, kStage - 1u)]; // the first member's first word
                for (uint32_t k = 0; k < run; ++k) {
                    const uint32_t c = end - at, sw = prev > 64u ? 2u : 1u;
                    const bool on = lane < c, on2 = 64u + lane < c;
                    const uint32_t end2 = fl[min(k + 3u, run + 1u)], off2 = off + sw * c;
                    // the next front's, while this one is ordered
                    const uint64_t next = stage[min(off2 + lane, kStage - 1u)];
                    if (sw == 1u && c <= 64u) {
                        uint64_t p[6], q[6];
#pragma unroll
                        for (uint32_t b = 0; b < 6u; ++b) p[b] = p0[b];
                        const uint32_t v = on ? held_max<6u>(word, p) : 0u;
#pragma unroll
                        for (uint32_t b = 0; b < 6u; ++b) q[b] = __ballot((v >> b) & 1u);
                        uint32_t pos = place_in_word<6u>(v, q, __ballot(on), (uint64_t(1) << lane) - 1u);
                        if (on) pos_out[at + lane] = pos;
                        else pos = 0u;
#pragma unroll
                        for (uint32_t b = 0; b < 6u; ++b) p0[b] = __ballot((pos >> b) & 1u);
                        p0[6] = 0u; // (p1 is not read while a front has at most 64)
                    } else {
                        uint32_t v = on ? held_max<7u>(word, p0) : 0u, v2 = 0u;
                        if (sw == 2u) {
                            const uint64_t h = on ? stage[off + c + lane] : 0u;
                            if (h) v = max(v, held_max<7u>(h, p1));
                        }
                        if (c > 64u) {
                            const uint64_t w0 = on2 ? stage[off + 64u + lane] : 0u;
                            v2 = held_max<7u>(w0, p0);
                            if (sw == 2u) {
                                const uint64_t w1 = on2 ? stage[off + c + 64u + lane] : 0u;
                                if (w1) v2 = max(v2, held_max<7u>(w1, p1));
                            }
                        }
                        uint64_t q0[7], q1[7];
#pragma unroll
                        for (uint32_t b = 0; b < 7u; ++b) {
                            q0[b] = __ballot((v >> b) & 1u);
                            q1[b] = __ballot((v2 >> b) & 1u);
                        }
                        const uint64_t m0 = __ballot(on), m1 = __ballot(on2), lower = (uint64_t(1) << lane) - 1u;
                        uint32_t pos = place_in_word<7u>(v, q0, m0, lower), pos2 = 0u;
                        if (c > 64u) {
                            pos += place_in_word<7u>(v, q1, m1, 0u);
                            pos2 = place_in_word<7u>(v2, q0, m0, ~uint64_t(0)) + place_in_word<7u>(v2, q1, m1, lower);
                        }
                        if (on) pos_out[at + lane] = pos;
                        else pos = 0u;
                        if (on2) pos_out[at + 64u + lane] = pos2;
                        else pos2 = 0u;
#pragma unroll
                        for (uint32_t b = 0; b < 7u; ++b) {
                            p0[b] = __ballot((pos >> b) & 1u);
                            p1[b] = __ballot((pos2 >> b) & 1u);
                        }
                    }
                    word = next;
                    off = off2;
                    prev = c;
                    at = end;
                    end = end2;
                }
                if (lane == 0u) {
#pragma unroll
                    for (uint32_t b = 0; b < kPlanes; ++b) {
                        planes[b] = b < 7u ? p0[b] : 0u;
                        if (prev > 64u) planes[kPlanes + b] = b < 7u ? p1[b] : 0u;
                    }
                    s_words = off;
                }
            }
            L += run;
            load = L >= L0 + kWide;
            __syncthreads();
            wb += s_words;
            continue;
        }
        if (fl[2] - fl[1] <= kWide) {
            // one front of c members after one of s: wavefront (chunk, part)
            // takes the words part, part + parts, ... of 64 members, and then
            // compares them with the members of those blocks
            const uint32_t s = fl[1] - fl[0], c = fl[2] - fl[1], at = fl[1];
            const uint32_t sw = (s + 63u) / 64u, sb = bits_of(s - 1u), cw = (c + 63u) / 64u;
            const uint64_t *src = masks + wb;
            wb += static_cast<uint64_t>(c) * sw;
            const auto words_of = [&](const uint64_t *from, uint32_t members, uint32_t words) {
                const uint32_t chunks = (members + 63u) / 64u, parts = kWaves / chunks;
                const uint32_t x = 64u * (wave % chunks) + lane, part = wave / chunks;
#pragma unroll
                for (uint32_t k = 0; k < kAhead; ++k) {
                    const uint32_t w = part + k * parts;
                    ahead[k] = part < parts && x < members && w < words
                                   ? from[static_cast<uint64_t>(w) * members + x]
                                   : 0u;
                }
            };
            if (ahead_of != L) words_of(src, c, sw);
            const uint32_t parts = kWaves / cw, chunk = wave % cw, part = wave / cw, x = 64u * chunk + lane;
            uint32_t v = 0u;
            if (part < parts) { // uniform
#pragma unroll
                for (uint32_t k = 0; k < kAhead; ++k) {
                    const uint32_t w = part + k * parts;
                    if (w < sw && __ballot(ahead[k] != 0u)) v = max(v, plane_max(ahead[k], planes + w * kPlanes, sb));
                }
                for (uint32_t w = part + kAhead * parts; w < sw; w += parts) {
                    const uint64_t word = x < c ? src[static_cast<uint64_t>(w) * c + x] : 0u;
                    if (__ballot(word != 0u)) v = max(v, plane_max(word, planes + w * kPlanes, sb));
                }
                if (parts > 1u && v) atomicMax(&s_v[x], v);
            }
            // the next front's first words, in flight from here on
            if (L + 1u < fronts && L + 1u < L0 + kWide && fl[3] - fl[2] <= kWide) {
                words_of(src + static_cast<uint64_t>(c) * sw, fl[3] - fl[2], cw);
                ahead_of = L + 1u;
            }
            if (parts > 1u) __syncthreads();
            if (part < parts) {
                if (parts > 1u) v = s_v[x];
                if (part == 0u) {
                    const uint64_t p = sb <= 10u ? planes_by_lane<10u>(v, lane) : planes_by_lane<kRankBits>(v, lane);
                    if (lane < kPlanes) vplanes[chunk * kPlanes + lane] = p;
                }
            }
            __syncthreads();
            uint32_t pos = 0u;
            if (part < parts) {
                pos = sb <= 8u ? place_among<8u>(v, x, c, part, parts, vplanes)
                               : (sb <= 10u ? place_among<10u>(v, x, c, part, parts, vplanes)
                                            : place_among<kRankBits>(v, x, c, part, parts, vplanes));
                if (parts > 1u) {
                    if (pos) atomicAdd(&s_pos[x], pos);
                    if (part == 0u) s_v[x] = 0u; // for the next front; read before the barrier above
                }
            }
            if (parts > 1u) __syncthreads();
            if (part == 0u) {
                if (parts > 1u) {
                    pos = s_pos[x];
                    s_pos[x] = 0u;
                }
                if (x < c) pos_out[at + x] = pos;
                else pos = 0u;
                const uint64_t p = planes_by_lane<10u>(pos, lane);
                if (lane < kPlanes) planes[chunk * kPlanes + lane] = p;
            }
            ++L;
            load = L >= L0 + kWide;
            __syncthreads();
            continue;
        }
        // one front of c > kWide members after one of s, by the whole workgroup
        const uint32_t s = fl[1] - fl[0], c = fl[2] - fl[1], at = fl[1];
        const uint32_t sw = (s + 63u) / 64u, sb = bits_of(s - 1u), cw = (c + 63u) / 64u;
        const uint64_t *src = masks + wb;
        wb += static_cast<uint64_t>(c) * sw;
        uint32_t *bins = F + 64u * cw; // s of them; s + c <= n <= P
        // the positions of the front before by slot, for words of few bits, and the
        // largest of every 64
        for (uint32_t x = t; x < 64u * sw; x += kWide) {
            const uint32_t p = x < s ? pos_out[fl[0] + x] : 0u, most = wave_max(p);
            if (lane == 0u) s_top[x >> 6] = static_cast<uint16_t>(most);
            if (x < s) {
                bins[x] = 0u;
                list[x] = static_cast<uint16_t>(p);
            }
        }
        if (t == 0) s_run = 0u;
        __syncthreads();
        // (the second front's last dominators are known: see k_masks)
        const bool known = L == 1u && n > 2u * kWide;
        for (uint32_t x = t; x < 64u * cw; x += kWide) {
            uint32_t v = known && x < c ? first[at + x] : 0u;
            for (uint32_t left = known ? 0u : sw; left > 0u; left -= min(left, kAhead)) { // from the last: see above
                uint64_t word[kAhead];
#pragma unroll
                for (uint32_t k = 0; k < kAhead; ++k) {
                    word[k] = x < c && k < left ? src[static_cast<uint64_t>(left - 1u - k) * c + x] : 0u;
                }
#pragma unroll
                for (uint32_t k = 0; k < kAhead; ++k) {
                    if (k >= left) break; // uniform
                    const uint32_t w = left - 1u - k;
                    if (__ballot(__popcll(word[k]) > kFewBits)) {
                        if (__ballot(word[k] != 0u && s_top[w] > v)) {
                            v = max(v, plane_max(word[k], planes + w * kPlanes, sb));
                        }
                        continue;
                    }
                    while (__ballot(word[k] != 0u)) {
                        if (word[k]) {
                            v = max(v, static_cast<uint32_t>(list[64u * w + __builtin_ctzll(word[k])]));
                            word[k] &= word[k] - 1u;
                        }
                    }
                }
            }
            F[x] = v;
        }
        __syncthreads();
        constexpr uint32_t kLow = (1u << kRankBits) - 1u;
        for (uint32_t x = t; x < c; x += kWide) F[x] |= atomicAdd(&bins[F[x]], 1u) << kRankBits;
        __syncthreads();
        uint32_t largest = 0u;
        for (uint32_t x = t; x < s; x += kWide) largest = max(largest, bins[x]);
        largest = wave_max(largest);
        if (lane == 0u && largest > kBin) atomicMax(&s_run, largest);
        scan_bins(bins, s, s_scan);
        if (__builtin_amdgcn_readfirstlane(s_run) <= kBin) {
            for (uint32_t x = t; x < c; x += kWide) {
                list[bins[F[x] & kLow] + (F[x] >> kRankBits)] = static_cast<uint16_t>(x);
            }
            __syncthreads();
            for (uint32_t x = t; x < c; x += kWide) {
                const uint32_t v = F[x] & kLow, b0 = bins[v], b1 = v + 1u < s ? bins[v + 1u] : c;
                uint32_t pos = b0;
                for (uint32_t q = b0; q < b1; ++q) pos += list[q] < x ? 1u : 0u;
                F[x] = pos; // read by this thread alone
            }
        } else {
            uint32_t Pc = 1u;
            while (Pc < c) Pc <<= 1;
            for (uint32_t x = t; x < c; x += kWide) F[x] = ((F[x] & kLow) << 16) | x;
            __syncthreads(); // the keys end where the bins were
            for (uint32_t x = c + t; x < Pc; x += kWide) F[x] = 0xffffffffu;
            __syncthreads();
            wide_bitonic_sort(F, Pc);
            for (uint32_t x = t; x < c; x += kWide) list[F[x] & 0xffffu] = static_cast<uint16_t>(x);
            __syncthreads();
            for (uint32_t x = t; x < c; x += kWide) F[x] = list[x];
        }
        __syncthreads();
        for (uint32_t w = wave; w < cw; w += kWaves) {
            const uint32_t x = 64u * w + lane;
            const uint32_t pos = x < c ? F[x] : 0u;
            if (x < c) pos_out[at + x] = pos;
            const uint64_t p = planes_by_lane<kRankBits>(pos, lane);
            if (lane < kPlanes) planes[w * kPlanes + lane] = p;
        }
        ++L;
        load = L >= L0 + kWide;
        __syncthreads();
    }
}

__global__ __launch_bounds__(kBlock) void k_items(const uint32_t *__restrict__ members,
                                                  const uint32_t *__restrict__ rank, const uint32_t *__restrict__ fo,
                                                  const uint32_t *__restrict__ pos, uint32_t n, uint32_t upto,
                                                  uint64_t *__restrict__ front_items, uint64_t *__restrict__ rank_out)
{
    const uint32_t x = blockIdx.x * kBlock + threadIdx.x;
    if (x >= n) return;
    const uint32_t i = members[x], f = rank[i], a = fo[f];
    if (a <= upto) front_items[a + pos[x]] = i;
    rank_out[i] = f;
}

} // namespace

static uint32_t pow2_of(uint32_t n)
{
    uint32_t P = 1;
    while (P < n) P <<= 1;
    return P;
}
// The words of all fronts: each has its size times the words of the front
// before, at most n + n^2 / 256 in all.
static uint64_t mask_words_of(uint32_t n)
{
    return n + static_cast<uint64_t>(n) * n / 256u + 64u;
}
static size_t chain_lds_bytes(uint32_t n)
{
    const uint32_t P = pow2_of(n);
    return static_cast<size_t>((n + 63u) / 64u) * kPlanes * 8u + (P + 64u) * 4u + std::max(P * 2u, kStage * 8u);
}

// Row blocks per wavefront of k_pairs and k_tiles: four, so that a column is
// fetched once for 256 rows, unless that leaves SIMDs without a wavefront
// (k_pairs at 200 points: 17 us with four, 8 with one).
static uint32_t wave_rows(uint32_t nb)
{
    return nb > 64u ? 4u : 1u;
}

template <bool LISTS, uint32_t ROWS>
static void pairs_by_m(pgh_fnds_ws *ws, hipStream_t s, uint32_t n, uint32_t m)
{
    const uint32_t nb = (n + 63u) / 64u;
    const dim3 g(nb, (nb + ROWS * (kBlock / 64u) - 1u) / (ROWS * (kBlock / 64u)));
    const auto *keys = static_cast<const int64_t *>(ws->keys.ptr);
    auto *D = static_cast<uint64_t *>(ws->D.ptr);
    auto *cnt = static_cast<uint32_t *>(ws->cnt32.ptr), *nd = static_cast<uint32_t *>(ws->ndom32.ptr);
    const auto go = [&](auto f) { f<<<g, kBlock, 0, s>>>(keys, n, m, D, nb, cnt, nd); };
    switch (m) {
        case 1:
            return go(k_pairs<1, LISTS, ROWS>);
        case 2:
            return go(k_pairs<2, LISTS, ROWS>);
        case 3:
            return go(k_pairs<3, LISTS, ROWS>);
        case 4:
            return go(k_pairs<4, LISTS, ROWS>);
        case 5:
            return go(k_pairs<5, LISTS, ROWS>);
        case 6:
            return go(k_pairs<6, LISTS, ROWS>);
        default:
            return go(k_pairs<0, LISTS, ROWS>);
    }
}

pgh_status launch_pairs(pgh_fnds_ws *ws, hipStream_t s, uint32_t n, uint32_t m, bool lists)
{
    if (wave_rows((n + 63u) / 64u) == 1u) {
        if (lists) pairs_by_m<true, 1u>(ws, s, n, m);
        else pairs_by_m<false, 1u>(ws, s, n, m);
    } else {
        if (lists) pairs_by_m<true, 4u>(ws, s, n, m);
        else pairs_by_m<false, 4u>(ws, s, n, m);
    }
    PGH_HIP(hipGetLastError());
    return PGH_OK;
}

pgh_status launch_offsets(pgh_fnds_ws *ws, hipStream_t s, uint32_t n)
{
    static thread_local int dev_cached = -1;
    int dev = 0;
    PGH_HIP(hipGetDevice(&dev));
    if (dev != dev_cached) {
        PGH_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_offsets),
                                    hipFuncAttributeMaxDynamicSharedMemorySize,
                                    static_cast<int>((kChainMaxN + 1u) * 4u)));
        dev_cached = dev;
    }
    k_offsets<<<1, kWide, (n + 1u) * 4u, s>>>(
        static_cast<const uint32_t *>(ws->ndom32.ptr), static_cast<const uint32_t *>(ws->cnt32.ptr), n,
        static_cast<uint64_t *>(ws->dom_offsets.ptr), static_cast<uint64_t *>(ws->dom_count.ptr),
        static_cast<uint64_t *>(ws->scalars.ptr));
    PGH_HIP(hipGetLastError());
    return PGH_OK;
}

void chain_parts(pgh_fnds_ws *ws, uint32_t n, uint32_t m, std::vector<ws_part> &parts)
{
    const uint64_t nb = (n + 63u) / 64u;
    const ws_part own[] = {
        {&ws->perm, n * 4u},          {&ws->skeys, static_cast<uint64_t>(n) * m * 8u},
        {&ws->scnt, n * 4u},          {&ws->srank, n * 4u},
        {&ws->base, n * 4u},          {&ws->planes, nb * (kPlanes * 8u + 4u)},
        {&ws->any, n * 4u},           {&ws->tiles, nb * (nb + 1u) / 2u * 64u * 8u},
        {&ws->rank32, n * 4u},        {&ws->fo32, (n + 1u) * 4u},
        {&ws->wbase, (n + 1u) * 8u},  {&ws->members, n * 4u},
        {&ws->masks, mask_words_of(n) * 8u}, {&ws->pos32, n * 4u}, {&ws->first, n * 4u},
    };
    parts.insert(parts.end(), std::begin(own), std::end(own));
}

pgh_status launch_chain_fronts(pgh_fnds_ws *ws, hipStream_t s, uint32_t n, uint32_t m, uint32_t upto)
{
    const uint32_t nb = (n + 63u) / 64u;
    const auto *keys = static_cast<const int64_t *>(ws->keys.ptr);
    const auto *cnt = static_cast<const uint32_t *>(ws->cnt32.ptr);
    auto *perm = static_cast<uint32_t *>(ws->perm.ptr);
    auto *tiles = static_cast<uint64_t *>(ws->tiles.ptr);
    auto *rank = static_cast<uint32_t *>(ws->rank32.ptr);
    auto *fo = static_cast<uint32_t *>(ws->fo32.ptr);
    auto *wbase = static_cast<uint64_t *>(ws->wbase.ptr);
    auto *members = static_cast<uint32_t *>(ws->members.ptr);
    auto *masks = static_cast<uint64_t *>(ws->masks.ptr);
    auto *sc = static_cast<uint64_t *>(ws->scalars.ptr);
    const size_t order_lds = n * 4u, fronts_lds = (n + 1u) * 4u;
    static thread_local int dev_cached = -1;
    int dev = 0;
    PGH_HIP(hipGetDevice(&dev));
    if (dev != dev_cached) {
        const auto allow = [](const void *f, size_t bytes) {
            return hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes));
        };
        PGH_HIP(allow(reinterpret_cast<const void *>(&k_order), kChainMaxN * 4u));
        PGH_HIP(allow(reinterpret_cast<const void *>(&k_fronts), (kChainMaxN + 1u) * 4u));
        dev_cached = dev;
    }
    const uint32_t waves = (n + kBlock / 64u - 1u) / (kBlock / 64u);
    auto *skeys = static_cast<int64_t *>(ws->skeys.ptr);
    auto *scnt = static_cast<uint32_t *>(ws->scnt.ptr), *srank = static_cast<uint32_t *>(ws->srank.ptr);
    auto *base = static_cast<uint32_t *>(ws->base.ptr), *any = static_cast<uint32_t *>(ws->any.ptr);
    auto *planes = static_cast<uint64_t *>(ws->planes.ptr);
    auto *top = reinterpret_cast<uint32_t *>(planes + static_cast<uint64_t>(nb) * kPlanes);
    // (any, wbase: places to keep the places and the number of points without dominators)
    k_order<<<1, kWide, order_lds, s>>>(cnt, n, any, wbase);
    PGH_HIP(hipGetLastError());
    k_scatter<<<(n + kBlock - 1u) / kBlock, kBlock, 0, s>>>(keys, cnt, any, n, m, perm, scnt, skeys,
                                                            static_cast<uint32_t *>(ws->first.ptr));
    PGH_HIP(hipGetLastError());
    const uint32_t rows = wave_rows(nb);
    const dim3 tg(nb, (nb + rows * (kBlock / 64u) - 1u) / (rows * (kBlock / 64u)));
    const auto by_m = [m](auto f1, auto f2, auto f3) { return m == 1u ? f1 : (m == 2u ? f2 : f3); };
    if (rows == 1u) by_m(k_tiles<1, 1>, k_tiles<2, 1>, k_tiles<3, 1>)<<<tg, kBlock, 0, s>>>(skeys, scnt, n, wbase, tiles);
    else by_m(k_tiles<1, 4>, k_tiles<2, 4>, k_tiles<3, 4>)<<<tg, kBlock, 0, s>>>(skeys, scnt, n, wbase, tiles);
    PGH_HIP(hipGetLastError());
    for (uint32_t J0 = 0; J0 < nb; J0 += kSpan) {
        const uint32_t J1 = std::min(J0 + kSpan, nb);
        k_rank<<<1, kWide, 0, s>>>(tiles, n, J0, J1, J0 ? base : nullptr, srank, planes, top, wbase);
        if (J1 < nb) k_far<<<nb - J1, kFarBlock, 0, s>>>(tiles, n, J0, J1, planes, top, base, J0 == 0u ? 1u : 0u, wbase);
        PGH_HIP(hipGetLastError());
    }
    k_fronts<<<1, kWide, fronts_lds, s>>>(srank, perm, n, fo, static_cast<uint64_t *>(ws->front_offsets.ptr), wbase,
                                          rank, any, sc);
    PGH_HIP(hipGetLastError());
    const uint32_t big_groups = n > kBigFront ? (nb + kBlock / 64u - 1u) / (kBlock / 64u) : 0u;
    k_slots<<<waves + big_groups, kBlock, 0, s>>>(any, rank, fo, n, big_groups, members);
    PGH_HIP(hipGetLastError());
    const uint32_t large_x = (nb + kBlock / 64u - 1u) / (kBlock / 64u);
    const uint32_t large_y = n > 2u * kWide ? std::min((nb + kTileWords - 1u) / kTileWords, 64u) : 0u;
    by_m(k_masks<1>, k_masks<2>, k_masks<3>)<<<large_x * large_y + waves, kBlock, 0, s>>>(
        keys, cnt, members, rank, fo, wbase, n, large_x, large_y, masks, static_cast<uint32_t *>(ws->first.ptr));
    PGH_HIP(hipGetLastError());
    return launch_chain_items(ws, s, n, upto);
}

pgh_status launch_chain_items(pgh_fnds_ws *ws, hipStream_t s, uint32_t n, uint32_t upto)
{
    static thread_local int dev_cached = -1;
    int dev = 0;
    PGH_HIP(hipGetDevice(&dev));
    if (dev != dev_cached) {
        PGH_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_chain),
                                    hipFuncAttributeMaxDynamicSharedMemorySize,
                                    static_cast<int>(chain_lds_bytes(kChainMaxN))));
        dev_cached = dev;
    }
    const auto *rank = static_cast<const uint32_t *>(ws->rank32.ptr), *fo = static_cast<const uint32_t *>(ws->fo32.ptr);
    auto *pos = static_cast<uint32_t *>(ws->pos32.ptr);
    k_chain<<<1, kWide, chain_lds_bytes(n), s>>>(fo, static_cast<const uint64_t *>(ws->masks.ptr), mask_words_of(n),
                                                 upto, static_cast<const uint64_t *>(ws->scalars.ptr), n, pow2_of(n),
                                                 static_cast<const uint32_t *>(ws->first.ptr), pos);
    PGH_HIP(hipGetLastError());
    k_items<<<(n + kBlock - 1u) / kBlock, kBlock, 0, s>>>(static_cast<const uint32_t *>(ws->members.ptr), rank, fo, pos,
                                                          n, upto, static_cast<uint64_t *>(ws->front_items.ptr),
                                                          static_cast<uint64_t *>(ws->rank.ptr));
    PGH_HIP(hipGetLastError());
    return PGH_OK;
}

} // namespace pgh
