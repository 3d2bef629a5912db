// layout.hpp -- device fields [field][element][node] to the host's
// [element][field][node] arrays.
//
// The reordering runs on the device, through a bounded staging buffer kept by
// the model, and each piece is copied straight into the caller's array.  A
// host vector of the whole field, filled by the copy and reordered by memcpy,
// cost three passes over fresh host pages: 44 ms for the 124 MB of a 24x21x12,
// N = 7 hydrostatic state against 13 ms.
#pragma once

#include <algorithm>

#include "common.hpp"

namespace self {

constexpr size_t kStageDoubles = (size_t)4 << 20;  // 32 MB

struct HostStage {
    double *buf = nullptr;
    size_t cap = 0;
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
    const size_t piece = std::min(nE, std::max<size_t>(1, kStageDoubles / row));
    if (st.cap < piece * row) {
        st.release();
        SELF_HIP(hipMalloc(reinterpret_cast<void **>(&st.buf), sizeof(double) * piece * row));
        st.cap = piece * row;
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
