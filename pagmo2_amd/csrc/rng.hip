// rng.hip -- seeded inputs on the device: std::mt19937 words and
// batch_random_decision_vector (include/pagmo/utils/generic.hpp:326-388).
#include "fitness_dev.hpp"
#include "mt_dev.hpp"
#include "mt_jump_host.hpp"
#include "pgh_internal.hpp"

#include <vector>

namespace pgh
{
using namespace dev;

namespace
{

// Words handed out become U(lb_j, ub_j), two per element (generic.hpp:376-380),
// element e of the row-major matrix at column e mod nx.  Every run starts at an
// even word and has an even length.  COLS: the bounds depend on the column
// (lennard_jones); otherwise they are column 0's.
template <bool COLS>
struct uniform_sink {
    double *out;
    uint64_t e0; // element of the hand-out's first word
    uint32_t nx;
    int kind;
    double lb, w;
    __device__ __forceinline__ uniform_sink(double *out_, uint64_t e0_, uint32_t nx_, int kind_)
        : out(out_), e0(e0_), nx(nx_), kind(kind_)
    {
        double ub;
        bounds_of(kind, 0u, lb, ub);
        w = mt_width(lb, ub);
    }
    __device__ __forceinline__ void operator()(uint64_t at, const uint32_t *__restrict__ words, uint32_t n,
                                               uint32_t tid, uint32_t nthr) const
    {
        const uint64_t e = e0 + at / 2u;
        double *o = out + e;
        const uint32_t c0 = COLS ? static_cast<uint32_t>(e % nx) : 0u;
        for (uint32_t i = tid; i < n / 2u; i += nthr) {
            const uint2 v = reinterpret_cast<const uint2 *>(words)[i];
            double a = lb, wi = w;
            if constexpr (COLS) {
                double ub;
                bounds_of(kind, (c0 + i) % nx, a, ub);
                wi = mt_width(a, ub);
            }
            o[i] = mt_uniform(mt_temper(v.x), mt_temper(v.y), a, wi);
        }
    }
};

// Segment blockIdx.x = s of a stream split in segments of B words: words
// [s B, min((s + 1) B, n)) of the generator that `st` holds, after `skip`
// words (one segment only), handed to out (kElems, kElemsCols: as the elements
// of a matrix of nx columns; else as words).  The segment's generator reaches s B
// by one jump, z^(s B) (entry s - 1 of the table).
// The mapping to doubles in the same pass saves writing the words and reading
// them back.  65536 x 1000 on 500 segments: 1.13 ms -> 0.22 ms, about 0.1 ms of
// it the jumps; the 524 MB of stores alone take 0.1 ms.
enum : int { kWordsOut, kElems, kElemsCols };

template <int OUT>
__global__ __launch_bounds__(kMtBlock) void k_mt19937(mt_state st, uint64_t skip, uint64_t n, uint64_t B,
                                                      const uint32_t *__restrict__ table, void *__restrict__ out,
                                                      uint32_t nx, int kind)
{
    __shared__ __align__(16) uint32_t buf[kMtBuf];
    uint32_t pos;
    mt_load(st, buf, pos);
    const uint64_t s = blockIdx.x, begin = s * B;
    if (s > 0u) mt_jump(buf, table + (s - 1u) * kMtN);
    if (skip) mt_hand_out(buf, pos, skip, mt_no_sink{});
    const uint64_t count = min(B, n - begin);
    if constexpr (OUT != kWordsOut) {
        mt_hand_out(buf, pos, count,
                    uniform_sink<OUT == kElemsCols>(static_cast<double *>(out), begin / 2u, nx, kind));
    } else {
        mt_hand_out(buf, pos, count, mt_word_sink{static_cast<uint32_t *>(out) + begin});
    }
}

// The first n words after `skip` of std::mt19937(seed): one workgroup up to
// kMtSplitMin words, else segments of B words, a power of two that makes at
// most kMtMaxSegs of them and is at least kMtSegMin.  The jump polynomials
// z^(s B) depend on B alone: the host makes them once per process, as
// consecutive multiples, and the device keeps a table per B and power-of-two
// count of them (2.5 KB each).  At most two segments per CU: 2^27 words take
// 263 us in 512 segments, 291 us in 256 and 329 us in 1024 (a jump costs a CU as
// much as making 1.5 10^5 words).  Split from 2^17 words on: one workgroup makes
// 2^17 words in 52 us, a split call of 2^18 takes 77 us.
constexpr uint64_t kMtSplitMin = uint64_t(1) << 17, kMtSegMin = uint64_t(1) << 14;
constexpr uint32_t kMtMaxSegs = 512;
// While the caller's stream is being captured no table is made for calls of up
// to kMtCaptureSolo words: they run as one segment unless the table exists.  Nor
// is one made for a program's first such calls (mtj::without_table): 2^18 words
// take 118 us in one segment and 93 in several, 2^21 words 0.87 ms and 98 us, and
// the table for the first takes 1 ms, for the second 2 (and 6 more where its copy
// is the process's first).
constexpr uint64_t kMtCaptureSolo = mtj::kRentWords;

template <int OUT>
pgh_status launch_mt(uint32_t seed, uint64_t skip, uint64_t n, void *out, uint32_t nx, int kind, hipStream_t s)
{
    mt_state st;
    mt_seed_host(seed, st);
    uint64_t B = n;
    const uint32_t *table = nullptr;
    if (skip == 0u && n > kMtSplitMin) {
        B = kMtSegMin;
        while (B * kMtMaxSegs < n) B <<= 1;
        const uint32_t segs = static_cast<uint32_t>((n + B - 1u) / B);
        uint32_t count = 32u;
        while (count < segs) count <<= 1;
        PGH_TRY(jump_table_find(B, count - 1u, &table));
        if (!table) {
            hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
            if (hipStreamIsCapturing(s, &cs) != hipSuccess) (void)hipGetLastError();
            const bool capturing = cs != hipStreamCaptureStatusNone;
            if (!capturing || n > kMtCaptureSolo) {
                PGH_TRY(jump_table_make(B, count - 1u, n, capturing ? nullptr : &s, &table));
            }
            if (!table) B = n;
        }
    }
    const uint32_t segs = static_cast<uint32_t>((n + B - 1u) / B);
    k_mt19937<OUT><<<dim3(segs), dim3(kMtBlock), 0, s>>>(st, skip, n, B, table, out, nx, kind);
    PGH_HIP(hipGetLastError());
    return PGH_OK;
}

} // namespace

pgh_status launch_mt19937(uint32_t seed, uint64_t skip, uint64_t n, uint32_t *out, hipStream_t s)
{
    if (n == 0u) return PGH_OK;
    return launch_mt<kWordsOut>(seed, skip, n, out, 1u, 0, s);
}

pgh_status launch_batch_random_dv(const prob &p, uint64_t n, uint32_t seed, double *out, hipStream_t s)
{
    if (p.kind == ZDT || p.kind == DTLZ) return fail(PGH_UNSUPPORTED, "no device draws for ZDT and DTLZ");
    const uint64_t count = n * p.nx;
    if (count == 0u) return PGH_OK;
    // every bound pair of the supported problems has lb < ub, so each element
    // consumes exactly two words (generic.hpp:376-380)
    if (p.kind == LENNARD_JONES) return launch_mt<kElemsCols>(seed, 0u, 2u * count, out, p.nx, p.kind, s);
    return launch_mt<kElems>(seed, 0u, 2u * count, out, p.nx, p.kind, s);
}

} // namespace pgh
