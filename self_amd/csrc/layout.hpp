// layout.hpp -- device fields [field][element][node] to the host's
// [element][field][node] arrays.
//
// The reordering runs on the device, through a bounded staging buffer kept by
// the model, and each piece is copied straight into the caller's array.  A
// host vector of the whole field, filled by the copy and reordered by memcpy,
// costs three passes over fresh host pages: 44 ms for the 124 MB of a 24x21x12,
// N = 7 hydrostatic state against 13 ms.  It is the way where the device has no
// memory left for the buffer: reading a field must not fail for that.
#pragma once

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "common.hpp"

namespace self {

// Most of the staging buffer: 32 MB.  SELF_AMD_STAGE_DOUBLES overrides it (a
// test of the way without one sets 0, of several pieces a small number).
inline size_t stage_doubles()
{
    const char *s = std::getenv("SELF_AMD_STAGE_DOUBLES");
    if (s && *s) return (size_t)std::strtoull(s, nullptr, 10);
    return (size_t)4 << 20;
}

struct HostStage {
    double *buf = nullptr;
    size_t cap = 0;  // doubles
    HostStage() = default;
    HostStage(const HostStage &) = delete;
    HostStage &operator=(const HostStage &) = delete;
    ~HostStage() { release(); }
    void release()
    {
        if (buf) (void)hipFree(buf);
        buf = nullptr;
        cap = 0;
    }
    // room for n values, if the device has it
    bool reserve(size_t n)
    {
        if (n <= cap) return true;
        release();
        if (hipMalloc(reinterpret_cast<void **>(&buf), sizeof(double) * n) != hipSuccess) {
            (void)hipGetLastError();
            buf = nullptr;
            return false;
        }
        cap = n;
        return true;
    }
};

// element-first copy of elements e0 .. e0 + n - 1; a thread per value
template <typename T>
__global__ __launch_bounds__(256) void k_elements_first(const T *__restrict__ src, T *__restrict__ dst, size_t nE,
                                                        int nf, int np, size_t e0, size_t n)
{
    const size_t row = (size_t)nf * np, total = n * row;
    for (size_t k = (size_t)blockIdx.x * 256 + threadIdx.x; k < total; k += (size_t)gridDim.x * 256) {
        const size_t e = k / row, w = k - e * row, f = w / np, nd = w - f * np;
        dst[k] = src[(f * nE + e0 + e) * np + nd];
    }
}

// Work queued on s before the call is waited for; the copy is complete on return.
inline int fields_to_host(const double *dev, double *host, size_t nE, int nf, int np, HostStage &st, hipStream_t s)
{
    const size_t row = (size_t)nf * np;
    if (nf == 1) {  // the same layout
        SELF_HIP(hipMemcpyAsync(host, dev, sizeof(double) * nE * row, hipMemcpyDeviceToHost, s));
        SELF_HIP(hipStreamSynchronize(s));
        return SELF_OK;
    }
    const size_t most = stage_doubles(), piece = std::min(nE, std::max<size_t>(1, most / row));
    if (most == 0 || !st.reserve(piece * row)) {
        std::vector<double> buf(nE * row);
        SELF_HIP(hipMemcpyAsync(buf.data(), dev, sizeof(double) * buf.size(), hipMemcpyDeviceToHost, s));
        SELF_HIP(hipStreamSynchronize(s));
        for (size_t e = 0; e < nE; ++e)
            for (size_t f = 0; f < (size_t)nf; ++f)
                std::memcpy(host + (e * nf + f) * np, buf.data() + (f * nE + e) * np, sizeof(double) * np);
        return SELF_OK;
    }
    for (size_t e0 = 0; e0 < nE; e0 += piece) {
        const size_t n = std::min(piece, nE - e0);
        const unsigned grid = (unsigned)std::min<size_t>((n * row + 255) / 256, 4096);
        hipLaunchKernelGGL(k_elements_first<double>, dim3(grid), dim3(256), 0, s, dev, st.buf, nE, nf, np, e0, n);
        SELF_HIP(hipGetLastError());
        SELF_HIP(hipMemcpyAsync(host + e0 * row, st.buf, sizeof(double) * n * row, hipMemcpyDeviceToHost, s));
        SELF_HIP(hipStreamSynchronize(s));
    }
    return SELF_OK;
}

}  // namespace self
