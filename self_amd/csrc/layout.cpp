// layout.cpp -- pinned buffers of the transfers in layout.hpp.
#include "layout.hpp"

#include <emmintrin.h>

#include <cstdlib>
#include <mutex>

namespace self {

namespace {

// Buffers not in use, at most kKept of 8 MB; what is returned beyond that is
// freed at once.
constexpr size_t kKept = 4;
std::mutex g_mutex;
std::vector<StageBuffer> g_free;

void destroy(StageBuffer &b)
{
    if (b.p) (void)hipHostFree(b.p);
    for (hipEvent_t e : b.done)
        if (e) (void)hipEventDestroy(e);
    b = StageBuffer{};
}

}  // namespace

size_t stage_doubles()
{
    const char *s = std::getenv("SELF_AMD_STAGE_DOUBLES");
    if (s && *s) return (size_t)std::strtoull(s, nullptr, 10);
    return (size_t)1 << 19;
}

void store_past_caches(double *to, const double *from, size_t n)
{
    long long v;
    size_t k = 0;
    if (n > 0 && reinterpret_cast<uintptr_t>(to) % 16) {
        std::memcpy(&v, from, sizeof v);
        _mm_stream_si64(reinterpret_cast<long long *>(to), v);
        k = 1;
    }
    for (; k + 2 <= n; k += 2)
        _mm_stream_si128(reinterpret_cast<__m128i *>(to + k),
                         _mm_loadu_si128(reinterpret_cast<const __m128i *>(from + k)));
    if (k < n) {
        std::memcpy(&v, from + k, sizeof v);
        _mm_stream_si64(reinterpret_cast<long long *>(to + k), v);
    }
}

void store_past_caches_fence() { _mm_sfence(); }

StageLease::StageLease(size_t n, hipStream_t s) : s_(s)
{
    if (n == 0) return;
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        for (size_t k = 0; k < g_free.size(); ++k)
            if (g_free[k].device == device && g_free[k].cap >= n) {
                b_ = g_free[k];
                g_free.erase(g_free.begin() + (long)k);
                return;
            }
        g_free.reserve(kKept);
    }
    // A full-sized buffer serves every later call; a small one is had sooner.
    const size_t full = 2 * stage_doubles(), cap = n <= full / 8 ? full / 8 : n <= full ? full : n;
    b_.device = device;
    if (e == hipSuccess)
        e = hipHostMalloc(reinterpret_cast<void **>(&b_.p), sizeof(double) * cap, hipHostMallocDefault);
    if (e != hipSuccess) b_.p = nullptr;
    for (hipEvent_t &v : b_.done)
        if (e == hipSuccess) e = hipEventCreateWithFlags(&v, hipEventDisableTiming);
    if (e == hipSuccess) {
        b_.cap = cap;
    } else {
        (void)hipGetLastError();
        destroy(b_);
    }
}

StageLease::~StageLease()
{
    if (!b_.p) return;
    if (!over_) (void)hipStreamSynchronize(s_);
    StageBuffer out = b_;
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        if (g_free.size() < kKept) {
            g_free.push_back(b_);  // within the reserved capacity
            return;
        }
        for (StageBuffer &f : g_free)  // the larger one stays
            if (f.cap < out.cap) std::swap(f, out);
    }
    destroy(out);
}

}  // namespace self
