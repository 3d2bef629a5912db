// dg3d_device.hpp -- pieces shared by the 3-D DG kernels (hexahedral
// elements, Gauss nodes, i fastest within an element, faces numbered as
// src/common/ModelFlags.f90:36-41 minus one: south 0 = p-, east 1 = s+,
// north 2 = p+, west 3 = s-, bottom 4 = q-, top 5 = q+).
#pragma once

#include <hip/hip_runtime.h>

#include "dg2d_device.hpp"

namespace self {

// Side descriptor (int2) of one element side: x = neighbour element (>= 0)
// or boundary flag (< 0); y: bits 0-2 neighbour side, 3 primary, 4 swap,
// 5 i reversed, 6 j reversed, bits 8.. boundary slot.
__host__ __device__ __forceinline__ int s3_nbr_side(int y) { return y & 7; }
__host__ __device__ __forceinline__ bool s3_primary(int y) { return (y >> 3) & 1; }
__host__ __device__ __forceinline__ int s3_slot(int y) { return y >> 8; }

// node of the neighbour's face matching own face node (a, b): the forward
// map (i,j) -> (k,l) of the reference's face loop when this side is
// primary, its inverse otherwise
__host__ __device__ __forceinline__ void s3_map_n(int N, int y, int a, int b, int &na, int &nb)
{
    const int sw = (y >> 4) & 1, fi = (y >> 5) & 1, fj = (y >> 6) & 1;
    if (s3_primary(y)) {
        const int ii = fi ? N - a : a, jj = fj ? N - b : b;
        na = sw ? (fj ? N - b : b) : ii;
        nb = sw ? (fi ? N - a : a) : jj;
    } else if (!sw) {
        na = fi ? N - a : a;
        nb = fj ? N - b : b;
    } else {
        na = fi ? N - b : b;
        nb = fj ? N - a : a;
    }
}

template <int N>
__device__ __forceinline__ void s3_map(int y, int a, int b, int &na, int &nb)
{
    s3_map_n(N, y, a, b, na, nb);
}

// value at side s, face node (a, b) of one element's nodal field q (i
// fastest) through the interpolants to -1 (lL) and +1 (lR)
template <int N>
__device__ __forceinline__ double face_trace3(const double *lL, const double *lR, const double *q, int s, int a,
                                              int b)
{
    constexpr int n1 = N + 1;
    const double *l = (s == 1 || s == 2 || s == 5) ? lR : lL;
    int off, stride;
    if (s == 1 || s == 3) { off = n1 * (a + n1 * b); stride = 1; }          // east / west: (p, q)
    else if (s == 0 || s == 2) { off = a + n1 * n1 * b; stride = n1; }      // south / north: (s, q)
    else { off = a + n1 * b; stride = n1 * n1; }                            // bottom / top: (s, p)
    double acc = l[0] * q[off];
    #pragma unroll
    for (int m = 1; m < n1; ++m) acc = __builtin_fma(l[m], q[off + m * stride], acc);
    return acc;
}

// ---- N = 7 on the FP64 matrix cores (Mf in dg2d_device.hpp).  An element's 512
// nodes are eight wavefronts, wavefront wv the plane k = wv with the node
// order of the instruction's layout: contractions in s and p give each lane its
// own node's value, 2 LDS reads instead of 16.  A contraction in q runs on the
// plane j = wv; its results go back through LDS, in place (a plane j = wv is
// read and written by wavefront wv only, in order).  Face traces take four
// instructions a wavefront: the four sides that cross plane k = wv in lanes of
// result rows 0 and 1, bottom and top of plane j = wv in rows 2 and 3.
// Rows 9 and planes 72 apart: the operand reads of all three directions then
// spread over the LDS banks (8 and 64: two lanes a bank in s, four in q).
constexpr int kMf3Size = 576;

__device__ __forceinline__ int mf3_at(int i, int j, int k)
{
    return i + 9 * j + 72 * k;
}

struct Mf3Ops {
    double a[2], b[2];  // left operand (rows), right operand (transposed)
};

__device__ __forceinline__ void mf3_load(Mf3Ops &M, const double *D, int tl)
{
    const MfLane<7> a(tl);
    #pragma unroll
    for (int q = 0; q < 2; ++q) {
        M.a[q] = D[(4 * a.bi + a.c) + 8 * (4 * q + a.k)];
        M.b[q] = D[(4 * a.bj + a.c) + 8 * (4 * q + a.k)];
    }
}

__device__ __forceinline__ double mf3_s(const Mf3Ops &M, const double *X, int wv, int tl)
{
    const MfLane<7> a(tl);
    double r = 0.0;
    #pragma unroll
    for (int q = 0; q < 2; ++q)
        r = __builtin_amdgcn_mfma_f64_4x4x4f64(M.a[q], X[mf3_at(4 * q + a.k, 4 * a.bj + a.c, wv)], r, 0, 0, 0);
    return r;
}

__device__ __forceinline__ double mf3_p(const Mf3Ops &M, const double *X, int wv, int tl)
{
    const MfLane<7> a(tl);
    double r = 0.0;
    #pragma unroll
    for (int q = 0; q < 2; ++q)
        r = __builtin_amdgcn_mfma_f64_4x4x4f64(X[mf3_at(4 * a.bi + a.c, 4 * q + a.k, wv)], M.b[q], r, 0, 0, 0);
    return r;
}

// q contraction on plane j = wv: the result's node is mf3_q_node
__device__ __forceinline__ double mf3_q(const Mf3Ops &M, const double *X, int wv, int tl)
{
    const MfLane<7> a(tl);
    double r = 0.0;
    #pragma unroll
    for (int q = 0; q < 2; ++q)
        r = __builtin_amdgcn_mfma_f64_4x4x4f64(M.a[q], X[mf3_at(4 * a.bj + a.c, wv, 4 * q + a.k)], r, 0, 0, 0);
    return r;
}

// its place in the array
__device__ __forceinline__ int mf3_q_node(int wv, int tl)
{
    const MfLane<7> a(tl);
    return mf3_at(4 * a.bj + a.c, wv, 4 * a.bi + a.k);
}

// left operand of the traces: rows 0 and 2 left, 1 and 3 right interpolation
struct Mf3Lag {
    double v[2];
};

__device__ __forceinline__ void mf3_load_lag(Mf3Lag &M, const double *lL, const double *lR, int tl)
{
    const MfLane<7> a(tl);
    #pragma unroll
    for (int q = 0; q < 2; ++q) M.v[q] = (a.c & 1 ? lR : lL)[4 * q + a.k];
}

// side and node of the lane's face node; false where it has none
__device__ __forceinline__ bool mf3_face(int wv, int tl, int &sd, int &node)
{
    const MfLane<7> a(tl);
    sd = a.k < 2 ? (a.bj ? 2 * a.k : 3 - 2 * a.k) : a.k + 2;
    node = (4 * a.bi + a.c) + 8 * wv;
    return a.k < 2 || a.bj == 0;
}

__device__ __forceinline__ double mf3_trace(const Mf3Lag &M, const double *X, int wv, int tl)
{
    const MfLane<7> a(tl);
    const int n = 4 * a.bi + a.c;
    double u = 0.0, v = 0.0;
    #pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int m = 4 * q + a.k;
        u = __builtin_amdgcn_mfma_f64_4x4x4f64(M.v[q], X[a.bj ? mf3_at(n, m, wv) : mf3_at(m, n, wv)], u, 0, 0, 0);
        v = __builtin_amdgcn_mfma_f64_4x4x4f64(M.v[q], X[mf3_at(n, wv, m)], v, 0, 0, 0);
    }
    return a.k < 2 ? u : v;
}

}  // namespace self
