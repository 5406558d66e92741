// mt_jump.hip -- device copies of the std::mt19937 jump polynomials
// (mt_jump_host.hpp; layout: mt_dev.hpp, mt_jump), made once per device, share
// size and count, and kept for the life of the process.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <map>
#include <mutex>
#include <thread>
#include <tuple>
#include <vector>

#include "mt_dev.hpp"
#include "mt_jump_host.hpp"
#include "pgh_internal.hpp"

namespace pgh
{

static_assert(2u * mtj::kWords == dev::kMtN, "a polynomial on the device is 624 32-bit words");

pgh_status jump_table_bytes(const std::vector<uint64_t> &dists, std::vector<uint8_t> &h)
{
    if (!mtj::the_field().ok) return fail(PGH_DEVICE_ERROR, "mt19937 characteristic polynomial not found");
    h.assign(dists.size() * kJumpPolyBytes, 0u);
    mtj::prefetch_jump_polys(dists, std::min(8u, std::thread::hardware_concurrency()));
    for (size_t k = 0; k < dists.size(); ++k) {
        std::memcpy(h.data() + k * kJumpPolyBytes, mtj::jump_poly(dists[k]).data(), kJumpPolyBytes);
    }
    return PGH_OK;
}

pgh_status jump_polys_multiples(uint64_t S, uint64_t count)
{
    if (!mtj::the_field().ok) return fail(PGH_DEVICE_ERROR, "mt19937 characteristic polynomial not found");
    mtj::prefetch_multiples(S, count);
    return PGH_OK;
}

namespace
{
// A device copy of the bytes, by the stream or, without one, by a stream of its own
// (a process's first stream takes 3 ms).
pgh_status upload_table(const std::vector<uint8_t> &h, const hipStream_t *on, void **out)
{
    void *ptr = nullptr;
    hipStream_t s = on ? *on : nullptr;
    PGH_HIP(hipMalloc(&ptr, h.size()));
    pgh_status st = PGH_OK;
    if (!on) st = hip_status(hipStreamCreateWithFlags(&s, hipStreamNonBlocking), "hipStreamCreateWithFlags");
    if (st == PGH_OK) {
        st = hip_status(hipMemcpyAsync(ptr, h.data(), h.size(), hipMemcpyHostToDevice, s), "hipMemcpyAsync");
        const pgh_status w = hip_status(hipStreamSynchronize(s), "hipStreamSynchronize");
        if (st == PGH_OK) st = w;
        if (!on) (void)hipStreamDestroy(s);
    }
    if (st != PGH_OK) {
        (void)hipFree(ptr);
        return st;
    }
    *out = ptr;
    return PGH_OK;
}

// The tables of the process, kept for its life.
struct table_entry {
    void *table = nullptr;
    uint64_t spent = 0u; // words of the calls that did without
};
std::mutex tables_mu;
std::map<std::tuple<int, uint64_t, uint32_t>, table_entry> tables; // by device, S, count
} // namespace

pgh_status jump_table_find(uint64_t S, uint32_t count, const uint32_t **out)
{
    int dev = 0;
    PGH_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(tables_mu);
    const auto it = tables.find(std::make_tuple(dev, S, count));
    *out = it == tables.end() ? nullptr : static_cast<const uint32_t *>(it->second.table);
    return PGH_OK;
}

pgh_status jump_table_make(uint64_t S, uint32_t count, uint64_t words, const hipStream_t *on, const uint32_t **out)
{
    *out = nullptr;
    int dev = 0;
    PGH_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(tables_mu);
    table_entry &e = tables[std::make_tuple(dev, S, count)];
    if (!e.table) {
        if (mtj::without_table(e.spent, words)) return PGH_OK;
        PGH_TRY(jump_polys_multiples(S, count));
        std::vector<uint64_t> dists;
        for (uint64_t k = 1; k <= count; ++k) dists.push_back(k * S);
        std::vector<uint8_t> h;
        PGH_TRY(jump_table_bytes(dists, h));
        hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
        PGH_HIP(hipThreadExchangeStreamCaptureMode(&mode));
        const pgh_status st = upload_table(h, on, &e.table);
        (void)hipThreadExchangeStreamCaptureMode(&mode);
        PGH_TRY(st);
    }
    *out = static_cast<const uint32_t *>(e.table);
    return PGH_OK;
}

} // namespace pgh
