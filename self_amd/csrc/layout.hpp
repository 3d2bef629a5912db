// layout.hpp -- device fields [field][element][node] to the host's
// [element][field][node] arrays, and plain arrays either way.
//
// Pieces travel through two halves of a pinned buffer: while
// one piece is on its way, the piece before is put in the caller's order, which
// the copy out of the buffer does at no cost.  A copy from or to pageable memory
// has the runtime pin or stage the caller's pages on each call, the slower the
// fresher they are.  Measured, us, fresh pages (a hipMemcpy into a vector and a
// memcpy; a reordering kernel and a copy into the caller's array; this): 6 KB of
// three fields 12.8, 24.5, 12.2; 0.8 MB 415, 463, 114; 12.6 MB 1430, 954, 728;
// 50 MB 15250, 4470, 3900 (with ordinary stores; past the caches 31 MB of warm
// pages take 1600 instead of 2200).  Where no pinned memory is to be had, the vector
// serves.
#pragma once

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <vector>

#include "common.hpp"

namespace self {

// Most of one half: 4 MB (1 MB 5 to 10 % slower from 10 MB on, 512 KB 40 %).
// SELF_AMD_STAGE_DOUBLES overrides it (a test of the way without the buffer
// sets 0, of several pieces a small number).
size_t stage_doubles();

constexpr size_t kPastCaches = (size_t)1 << 17;  // doubles, 1 MB

// A pinned buffer for one transfer, from a small process-wide pool: a new one
// costs 0.3 ms a MB on its first use.  Any thread, any stream of the current
// device; a lease that ends before the transfer was seen to be over (an error
// on the way) waits for the stream.
struct StageBuffer {
    double *p = nullptr;
    size_t cap = 0;                           // doubles
    int device = -1;
    hipEvent_t done[2] = {nullptr, nullptr};  // the last copy of each half
};

class StageLease {
public:
    StageLease(size_t n, hipStream_t s);  // room for n values
    ~StageLease();
    StageLease(const StageLease &) = delete;
    StageLease &operator=(const StageLease &) = delete;
    bool ok() const { return b_.p != nullptr; }  // false: no pinned memory to be had
    double *half(size_t p, size_t n) const { return b_.p + (p & 1) * n; }
    hipEvent_t done(size_t p) const { return b_.done[p & 1]; }
    void over() { over_ = true; }

private:
    StageBuffer b_;
    hipStream_t s_;
    bool over_ = false;
};

// n values past the caches, any 8-byte alignment; fence() before others look.
void store_past_caches(double *to, const double *from, size_t n);
void store_past_caches_fence();

// Work queued on s before the call is waited for; the copy is complete on return.
inline int fields_to_host(const double *dev, double *host, size_t nE, int nf, int np, hipStream_t s)
{
    const size_t row = (size_t)nf * np, most = stage_doubles();
    const size_t piece = std::min(nE, std::max<size_t>(1, most / row)), n = piece ? (nE + piece - 1) / piece : 0;
    // An array of 1 MB does not stay in a core's second-level cache anyway, and
    // an ordinary store reads each line first: three fields of 26367 x 49 nodes
    // took 1773 us so, 983 past the caches, 804 without putting them anywhere.
    // Several fields of long rows, each a jump in the buffer, are better left to
    // memcpy: GetSolution with it and past the caches, us, 3 x 49 nodes 2210,
    // 1535; 5 x 216 950, 960; 2 x 343 1175, 1250; 5 x 512 8800, 11000; one field
    // of 67 MB 4880, 4400.
    const bool past = nE * row >= kPastCaches && (nf == 1 || np <= 128) &&
                      reinterpret_cast<uintptr_t>(host) % sizeof(double) == 0;
    const auto put = [&](double *to, const double *from, size_t k) {
        if (past) store_past_caches(to, from, k);
        else std::memcpy(to, from, sizeof(double) * k);
    };
    const auto order = [&](const double *src, size_t e0, size_t m) {  // src: [field][m][node]
        if (nf == 1) {
            put(host + e0 * row, src, m * row);
        } else {
            for (size_t e = 0; e < m; ++e)
                for (size_t f = 0; f < (size_t)nf; ++f)
                    put(host + ((e0 + e) * nf + f) * np, src + (f * m + e) * np, (size_t)np);
        }
        if (past) store_past_caches_fence();
    };
    StageLease st(most ? std::min<size_t>(n, 2) * piece * row : 0, s);
    if (!st.ok()) {
        std::vector<double> buf(nE * row);
        SELF_HIP(hipMemcpyAsync(buf.data(), dev, sizeof(double) * buf.size(), hipMemcpyDeviceToHost, s));
        SELF_HIP(hipStreamSynchronize(s));
        order(buf.data(), 0, nE);
        return SELF_OK;
    }
    const auto fetch = [&](size_t p) -> hipError_t {
        const size_t e0 = p * piece, m = std::min(piece, nE - e0);
        double *b = st.half(p, piece * row);
        hipError_t e = hipSuccess;
        if (m == nE)  // the whole field array
            e = hipMemcpyAsync(b, dev, sizeof(double) * nE * row, hipMemcpyDeviceToHost, s);
        else
            for (size_t f = 0; f < (size_t)nf && e == hipSuccess; ++f)
                e = hipMemcpyAsync(b + f * m * np, dev + (f * nE + e0) * np, sizeof(double) * m * np,
                                   hipMemcpyDeviceToHost, s);
        return e == hipSuccess && n > 1 ? hipEventRecord(st.done(p), s) : e;
    };
    if (n > 0) SELF_HIP(fetch(0));
    for (size_t p = 0; p < n; ++p) {
        if (p + 1 < n) SELF_HIP(fetch(p + 1));
        if (n > 1) SELF_HIP(hipEventSynchronize(st.done(p)));
        else SELF_HIP(hipStreamSynchronize(s));  // 7 us less than an event and a wait for it
        order(st.half(p, piece * row), p * piece, std::min(piece, nE - p * piece));
    }
    st.over();
    return SELF_OK;
}

// n values to the device, after the work queued on s; the copy is complete on return.
inline int array_to_device(const double *host, double *dev, size_t n, hipStream_t s)
{
    const size_t piece = std::min(n, stage_doubles());
    StageLease st(piece < n ? 2 * piece : piece, s);
    if (!st.ok()) {
        SELF_HIP(hipMemcpyAsync(dev, host, sizeof(double) * n, hipMemcpyHostToDevice, s));
        SELF_HIP(hipStreamSynchronize(s));
        return SELF_OK;
    }
    size_t p = 0;
    for (size_t k = 0; k < n; k += piece, ++p) {
        const size_t m = std::min(piece, n - k);
        double *b = st.half(p, piece);
        if (p >= 2) SELF_HIP(hipEventSynchronize(st.done(p)));
        std::memcpy(b, host + k, sizeof(double) * m);
        SELF_HIP(hipMemcpyAsync(dev + k, b, sizeof(double) * m, hipMemcpyHostToDevice, s));
        if (n > piece) SELF_HIP(hipEventRecord(st.done(p), s));
    }
    SELF_HIP(hipStreamSynchronize(s));
    st.over();
    return SELF_OK;
}

}  // namespace self
