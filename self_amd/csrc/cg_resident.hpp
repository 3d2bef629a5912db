// cg_resident.hpp -- the CGSEM conjugate-gradient iteration as one launch per
// solve.
//
// The two launches an iteration that k_cg_direction and k_cg_assemble_update
// need stream 126 MB through memory at 128x128, N = 7 (35.8 us an iteration),
// and for small problems cost their launches (13.9 us at 16x16, N = 3).  Up to
// 1 048 576 local nodes (4 a thread, one 1024-thread workgroup per CU) the
// whole problem fits the device's registers and LDS: solution, residual,
// direction, inverse diagonal and geometric factors of a thread's nodes stay
// there for all iterations, every copy of a shared node with the same bits.
// What travels are the element products of shared nodes (a tagged message per
// boundary node, read by the other copies) and the partial sums of the two
// reductions, which every workgroup reads from every other and adds in one
// fixed order (persist.hpp).  A reduction is also the barrier that lets the
// next iteration overwrite the messages of this one.  At N = 3 and 7 the
// element operator's contractions run on the FP64 matrix cores.
//
// Measured, us an iteration: 16x16 N = 3 13.9 -> 5.0, 32x32 N = 7 5.4, 90x90
// N = 7 8.0, 128x128 N = 7 35.8 -> 12.0 (1.5 of it the exchange, about 5 the
// latency of the two reductions: message to memory, poll, two sums over a
// wavefront and one over a workgroup each; the rest the element operators).
// The partial sums are written eight times, once for each XCD's readers: 12.3
// -> 12.0 there, 10.5 -> 9.5 at 100x100 N = 5.
//
// The recurrences, the copies' summation order (GlobalSum) and the stop test
// are those of the launched form for larger problems; the dot products are
// summed in another fixed order, which depends on the problem's shape only.  So
// that a result does not depend on whether the launch was resident (other work
// on the device, memory for its messages), a problem of a resident shape that
// does not run it takes three launches an iteration that form the same values
// in the same order (k_cg_ord_*), bit for bit.
#pragma once

#include "dg2d_device.hpp"
#include "krylov.hpp"
#include "persist.hpp"

namespace self {

struct CgResOut {
    double rNorm;
    int iter, done;
};

struct CgResArgs {
    const int *gid, *cs, *ci;
    const double *G3, *D, *dinv;  // dinv: null without a preconditioner
    const double *r, *u;          // residual and solution the solve begins with
    double *uOut;
    const SolverState *st;
    ll_quad *exch, *red1, *red2;  // [nLocal], [kCgResReplicas][256], [kCgResReplicas][256][2]
    unsigned exchBytes;
    int nE;
    unsigned tag0;                // tag of iteration it: tag0 + it
    PersistArgs P;
    CgResOut *out;
};

constexpr int kCgResThreads = 1024;
constexpr unsigned kNoMsg = 0xfffffff0u;  // past the end of every message buffer
// Partial sums are written once per XCD: 256 workgroups polling the same 32
// lines wait for each other.
constexpr int kCgResReplicas = 8;

// operands of the element operator's four contractions on the matrix cores
template <int N>
struct CgMfOps {
    double a[Mf<N>::K], b[Mf<N>::K], at[Mf<N>::K], bt[Mf<N>::K];
};

template <int N>
__device__ __forceinline__ void cg_mf_ops(CgMfOps<N> &M, const double *Dl, int tl)
{
    constexpr int n1 = N + 1;
    const MfLane<N> a(tl);
    #pragma unroll
    for (int q = 0; q < Mf<N>::K; ++q) {
        const int m = 4 * q + a.k;
        M.a[q] = Dl[(4 * a.bi + a.c) + n1 * m];
        M.b[q] = Dl[(4 * a.bj + a.c) + n1 * m];
        M.at[q] = Dl[m + n1 * (4 * a.bi + a.c)];
        M.bt[q] = Dl[m + n1 * (4 * a.bj + a.c)];
    }
}

// the element operator at one node of an element (in: the lane has one)
template <int N, int S, bool WL, typename F12, typename F22>
__device__ __forceinline__ double cg_element_product(const CgMfOps<N> &M, const double *Dl, double *usE, double *f1E,
                                                     double *f2E, double v, double g11, F12 g12of, F22 g22of, bool in,
                                                     int tl, int i, int j)
{
    #pragma clang fp contract(off)
    constexpr int n1 = N + 1;
    constexpr bool MF = Mf<N>::on;
    const int ns = i + S * j;
    if (in) usE[ns] = v;
    if constexpr (WL) wave_sync();
    else __syncthreads();
    double ds = 0.0, dp = 0.0;
    if constexpr (MF) {
        const MfLane<N> a(tl);
        #pragma unroll
        for (int q = 0; q < Mf<N>::K; ++q) {
            const int m = 4 * q + a.k;
            ds = __builtin_amdgcn_mfma_f64_4x4x4f64(M.a[q], usE[m + S * (4 * a.bj + a.c)], ds, 0, 0, 0);
            dp = __builtin_amdgcn_mfma_f64_4x4x4f64(usE[(4 * a.bi + a.c) + S * m], M.b[q], dp, 0, 0, 0);
        }
    } else {
        #pragma unroll
        for (int m = 0; m < n1; ++m) {
            ds = __builtin_fma(Dl[i + n1 * m], usE[m + S * j], ds);
            dp = __builtin_fma(Dl[j + n1 * m], usE[i + S * m], dp);
        }
    }
    if (in) {
        const double g12 = g12of(), g22 = g22of();
        f1E[ns] = __builtin_fma(g11, ds, g12 * dp);
        f2E[ns] = __builtin_fma(g12, ds, g22 * dp);
    }
    if constexpr (WL) wave_sync();
    else __syncthreads();
    double s1 = 0.0, s2 = 0.0;
    if constexpr (MF) {
        const MfLane<N> a(tl);
        #pragma unroll
        for (int q = 0; q < Mf<N>::K; ++q) {
            const int m = 4 * q + a.k;
            s1 = __builtin_amdgcn_mfma_f64_4x4x4f64(M.at[q], f1E[m + S * (4 * a.bj + a.c)], s1, 0, 0, 0);
            s2 = __builtin_amdgcn_mfma_f64_4x4x4f64(f2E[(4 * a.bi + a.c) + S * m], M.bt[q], s2, 0, 0, 0);
        }
    } else {
        #pragma unroll
        for (int m = 0; m < n1; ++m) {
            s1 = __builtin_fma(Dl[m + n1 * i], f1E[m + S * j], s1);
            s2 = __builtin_fma(Dl[m + n1 * j], f2E[i + S * m], s2);
        }
    }
    return -(s1 + s2);
}

// row stride of an element's arrays in LDS: at N = 7 an odd one, or the matrix
// operands' eight rows fall on four banks
template <int N>
constexpr int kCgRow = N == 7 ? N + 2 : N + 1;

template <int N, int K>
__global__ __launch_bounds__(kCgResThreads) void k_cg_resident(CgResArgs A)
{
    constexpr int n1 = N + 1, np = n1 * n1, T = kCgResThreads, epb = T / np, W = T / 64;
    constexpr bool WL = 64 % np == 0;
    constexpr int S = kCgRow<N>, ne = S * n1;
    // four nodes a thread: the solution, the inverse diagonal and as many of the
    // geometric factors as there is room for live in LDS (128 KB at N = 7)
    constexpr bool UD = K > 2;
    constexpr int kRest = 8 * (np + (WL ? 2 : 3) * epb * ne) + 24 * epb * K * 4 + 1024 + (UD ? 16 * K * T : 0);
    constexpr int GL = !UD ? 0 : kRest + 16 * K * T <= 163840 ? 2 : kRest + 8 * K * T <= 163840 ? 1 : 0;
    __shared__ double Dl[np], us[epb * ne], f1[WL ? 1 : epb * ne], f2[epb * ne];
    __shared__ double part[2][W], fold[2][4];
    __shared__ double ul[UD ? K * T : 1], dl[UD ? K * T : 1], gl[GL > 0 ? GL : 1][UD ? K * T : 1];
    // messages of the copies of each corner's degree of freedom (up to 4, the
    // own among them, in GlobalSum order) and their sum; the last entry is every
    // other node's
    constexpr int NC = epb * K * 4;
    __shared__ uint4 corner[NC];
    __shared__ double cornerSum[NC + 1];
    __shared__ int stop;
    const int t = threadIdx.x, wid = t >> 6;
    if (t == 0) stop = persist_given_up(A.P) || A.st->done;
    if (t < np) Dl[t] = A.D[t];
    for (int c = t; c < NC; c += T) corner[c] = make_uint4(kNoMsg, kNoMsg, kNoMsg, kNoMsg);
    if (t == 0) cornerSum[NC] = 0.0;
    __syncthreads();
    if (stop) return;
    const int b = xcd_block(blockIdx.x, gridDim.x), nB = gridDim.x;
    int tl;
    const int le = lane_element<N>(t, tl), nd = lane_node<N>(tl), i = nd % n1, j = nd / n1;
    const int ls = le < epb ? le : 0;
    // where a wavefront holds whole elements its flux takes the values' place
    // (a wavefront's LDS operations are done in order)
    double *usE = us + ls * ne, *f1E = WL ? usE : f1 + ls * ne, *f2E = f2 + ls * ne;
    CgMfOps<N> M;
    if constexpr (Mf<N>::on) cg_mf_ops<N>(M, Dl, tl);
    // corner lanes: entry (k epb + le) 4 + which of the table
    const bool isCorner = le < epb && (i == 0 || i == N) && (j == 0 || j == N);
    const int cEntry = isCorner ? ls * 4 + (i ? 1 : 0) + (j ? 2 : 0) : NC;
    const int cStep = isCorner ? epb * 4 : 0;
    // Per node: the byte offset of the other copy's message (edges) and, in bits
    // 4k of `mask`: 0 a product to send, 1 owner of its degree of freedom, 2 a
    // corner of more than two copies.  They are used as bit masks: a condition
    // per node and use would keep more scalar registers than there are.
    double r[K], v[K], g11[K], g12r[GL > 1 ? 1 : K], g22r[GL > 0 ? 1 : K], ur[UD ? 1 : K], dr[UD ? 1 : K];
    unsigned off[K];
    int mask = 0;
    const size_t nLocal = (size_t)A.nE * np;
    #pragma unroll
    for (int k = 0; k < K; ++k) {
        const int e = (b * K + k) * epb + le;
        const bool act = le < epb && e < A.nE;
        const size_t l = act ? (size_t)e * np + nd : 0;
        const int g = act ? A.gid[l] : -1;
        g11[k] = act ? A.G3[l] : 0.0;
        const double g12 = act ? A.G3[nLocal + l] : 0.0, g22 = act ? A.G3[2 * nLocal + l] : 0.0;
        off[k] = kNoMsg;
        r[k] = v[k] = 0.0;
        double uk = 0.0, dk = 0.0;  // a masked node's direction stays zero
        if (g >= 0) {
            const int c0 = A.cs[g], n = min(A.cs[g + 1] - c0, 4), first = A.ci[c0];
            int bits = (n > 1 ? 1 : 0) | (first == (int)l ? 2 : 0);
            if (n == 2) off[k] = 16u * (unsigned)(first == (int)l ? A.ci[c0 + 1] : first);
            if (n > 2) {
                bits |= 4;
                corner[cEntry + k * cStep] = make_uint4(16u * (unsigned)first, 16u * (unsigned)A.ci[c0 + 1],
                                                        16u * (unsigned)A.ci[c0 + 2],
                                                        n > 3 ? 16u * (unsigned)A.ci[c0 + 3] : kNoMsg);
            }
            mask |= bits << (4 * k);
            uk = A.u[g];
            r[k] = A.r[g];
            dk = A.dinv ? A.dinv[g] : 1.0;
        }
        if constexpr (UD) {
            ul[UD ? k * T + t : 0] = uk;
            dl[UD ? k * T + t : 0] = dk;
        } else {
            ur[UD ? 0 : k] = uk;
            dr[UD ? 0 : k] = dk;
        }
        if constexpr (GL > 0) gl[0][k * T + t] = g22;
        else g22r[k] = g22;
        if constexpr (GL > 1) gl[1][k * T + t] = g12;
        else g12r[k] = g12;
    }
    // all ones where bit `bit` of node k is set
    auto bits = [&](int k, int bit) { return (mask << (31 - 4 * k - bit)) >> 31; };
    auto dinv = [&](int k) { return UD ? dl[UD ? k * T + t : 0] : dr[UD ? 0 : k]; };
    const LLBuf exch(A.exch, A.exchBytes), red1(A.red1, 16 * 256 * kCgResReplicas),
        red2(A.red2, 32 * 256 * kCgResReplicas);
    const unsigned mine = (blockIdx.x & (kCgResReplicas - 1)) * 256 + t;
    const double r0 = A.st->r0, tol = A.st->tol;
    const int maxIters = A.st->maxIters, rule = A.st->stopRule;
    double num = A.st->numP[1], beta = 0.0, rn = 0.0;
    int it = 1, done = 0;
    __syncthreads();
    for (;; ++it) {
        #pragma clang fp contract(off)
        const unsigned tag = A.tag0 + (unsigned)it;
        double L[K], acc = 0.0;
        // ---- direction, element operator, products of shared nodes on their way
        #pragma unroll
        for (int k = 0; k < K; ++k) {
            v[k] = __builtin_fma(beta, v[k], dinv(k) * r[k]);  // beta = 0, v = 0 in the first iteration
            L[k] = cg_element_product<N, S, WL>(
                M, Dl, usE, f1E, f2E, v[k], g11[k],
                [&] {
                    if constexpr (GL > 1) return gl[1][k * T + t];
                    else return g12r[k];
                },
                [&] {
                    if constexpr (GL > 0) return gl[0][k * T + t];
                    else return g22r[k];
                },
                le < epb, tl, i, j);
            acc = __builtin_fma(v[k], L[k], acc);
            // a store past the buffer's end is dropped
            ll_store1(exch, (16u * (unsigned)(((b * K + k) * epb + le) * np + nd)) | (kNoMsg & ~(unsigned)bits(k, 0)), L[k], tag);
        }
        acc = wave_sum_dpp(acc);
        if ((t & 63) == 0) part[0][wid] = acc;
        __syncthreads();
        if (t < kCgResReplicas) {
            double p = part[0][0];
            #pragma unroll
            for (int q = 1; q < W; ++q) p += part[0][q];
            ll_store1(red1, 16u * (t * 256 + b), p, tag);
        }
        // ---- A v at shared nodes: the other copy's product (two copies in either
        // order have the same bits).  A load past the buffer's end (kNoMsg) returns
        // zero without an access, so no branch separates the loads.
        double o[K];
        bool good = ll_wait(true, A.P, [&] {
            unsigned w[K], wrong = 0;
            #pragma unroll
            for (int k = 0; k < K; ++k) o[k] = ll_load1(exch, off[k], tag, w[k]);
            #pragma unroll
            for (int k = 0; k < K; ++k) wrong |= w[k] & ~(unsigned)((int)off[k] >> 31);
            return (wrong >> 16) == 0;
        });
        // ---- corners: a thread each, all copies in GlobalSum order (the last
        // threads, while the first ones wait for the sums)
        for (int c0 = 0; c0 < NC; c0 += T) {
            const int c = c0 + T - 1 - t;
            const uint4 at = c < NC ? corner[c] : make_uint4(kNoMsg, kNoMsg, kNoMsg, kNoMsg);
            double x[4] = {0.0, 0.0, 0.0, 0.0};
            good = ll_wait(at.x != kNoMsg, A.P, [&] {
                unsigned w[4];
                x[0] = ll_load1(exch, at.x, tag, w[0]);
                x[1] = ll_load1(exch, at.y, tag, w[1]);
                x[2] = ll_load1(exch, at.z, tag, w[2]);
                x[3] = ll_load1(exch, at.w, tag, w[3]);
                w[3] &= ~(unsigned)((int)at.w >> 31);
                return ((w[0] | w[1] | w[2] | w[3]) >> 16) == 0;
            }) && good;
            if (c < NC) cornerSum[c] = ((x[0] + x[1]) + x[2]) + x[3];
        }
        // ---- v.Av of all workgroups
        if (t < 256) {
            double x = 0.0;
            good = ll_wait(t < nB, A.P, [&] { return ll_try1(red1, 16u * mine, tag, x); }) && good;
            x = wave_sum_dpp(t < nB ? x : 0.0);
            if ((t & 63) == 0) fold[0][wid] = x;
        }
        if (__syncthreads_or(!good)) return;
        const double vz = (fold[0][0] + fold[0][1]) + (fold[0][2] + fold[0][3]);
        const double alpha = num / vz;
        // ---- update; r.r and r.w over the owners (a masked node's residual
        // means nothing: its inverse diagonal is zero)
        double a0 = 0.0, a1 = 0.0;
        #pragma unroll
        for (int k = 0; k < K; ++k) {
            if constexpr (UD) {
                double &uk = ul[UD ? k * T + t : 0];
                uk = __builtin_fma(alpha, v[k], uk);
            } else {
                ur[UD ? 0 : k] = __builtin_fma(alpha, v[k], ur[UD ? 0 : k]);
            }
            const long long cm = bits(k, 2), ow = bits(k, 1);
            const double z = __longlong_as_double((__double_as_longlong(L[k] + o[k]) & ~cm) |
                                                  (__double_as_longlong(cornerSum[cEntry + k * cStep]) & cm));
            r[k] = __builtin_fma(-alpha, z, r[k]);
            const double ro = __longlong_as_double(__double_as_longlong(r[k]) & ow);
            a0 = __builtin_fma(ro, ro, a0);
            a1 = __builtin_fma(ro, dinv(k) * ro, a1);
        }
        a0 = wave_sum_dpp(a0);
        a1 = wave_sum_dpp(a1);
        if ((t & 63) == 0) {
            part[0][wid] = a0;
            part[1][wid] = a1;
        }
        __syncthreads();
        if (t < kCgResReplicas) {
            double p[3] = {part[0][0], part[1][0], 0.0};
            #pragma unroll
            for (int q = 1; q < W; ++q) {
                p[0] += part[0][q];
                p[1] += part[1][q];
            }
            const unsigned at = 32u * (t * 256 + b);
            ll_store3(red2, at, at + 16u, p, tag);
        }
        if (t < 256) {
            double x[3] = {0.0, 0.0, 0.0};
            good = ll_wait(t < nB, A.P, [&] { return ll_try3(red2, 32u * mine, 32u * mine + 16u, tag, x); });
            x[0] = wave_sum_dpp(t < nB ? x[0] : 0.0);
            x[1] = wave_sum_dpp(t < nB ? x[1] : 0.0);
            if ((t & 63) == 0) {
                fold[0][wid] = x[0];
                fold[1][wid] = x[1];
            }
        }
        if (__syncthreads_or(!good)) return;
        const double S0 = (fold[0][0] + fold[0][1]) + (fold[0][2] + fold[0][3]);
        const double S1 = (fold[1][0] + fold[1][1]) + (fold[1][2] + fold[1][3]);
        // ---- end of the iteration, the same in every workgroup (cg_end_apply)
        rn = sqrt(S0);
        if (b == 0 && t == 0 && it < A.st->resiLen) A.st->resi[it] = rn;
        const bool stopped = (rule == kStopSqrtNormRel) ? (sqrt(rn) / r0 < tol) : (rn / r0 < tol);
        if (stopped || it >= maxIters) {
            done = stopped ? 1 : 2;
            break;
        }
        beta = S1 / num;
        num = S1;
    }
    #pragma unroll
    for (int k = 0; k < K; ++k) {
        if (bits(k, 1)) {
            const size_t l = (size_t)((b * K + k) * epb + le) * np + nd;
            A.uOut[A.gid[l]] = UD ? ul[UD ? k * T + t : 0] : ur[UD ? 0 : k];
        }
    }
    if (b == 0 && t == 0) {
        A.out->rNorm = rn;
        A.out->iter = it;
        A.out->done = done;
    }
}

// The launch's end in the solver state; done = kCgGaveUp where it gave up.
constexpr int kCgGaveUp = 9;

__global__ void k_cg_res_commit(SolverState *st, const CgResOut *out, const int *status)
{
    if (st->done) return;  // nothing to solve: the launch returned at once
    if (*status != 0) {
        st->done = kCgGaveUp;
        return;
    }
    st->rNorm = out->rNorm;
    st->iter = out->iter;
    st->done = out->done;
}

// ---- the same iteration as three launches.  A thread has the resident form's
// nodes, so every sum has its order; vectors are indexed by degree of freedom,
// written by the owner copies (the direction to another array than it is read
// from).  Rows 0, 1, 2 of the partial sums: v.Av, r.r, r.w, an entry a workgroup.
struct CgOrdArgs {
    const int *gid, *cs, *ci;
    const double *G3, *D, *dinv;
    double *r, *u, *vNew, *L;
    const double *vOld;
    double *partials;  // rows of kRedBlocks
    SolverState *st;
    int nE, it;
};

// sum of 16 wavefronts' values, one after another (thread 0's result counts)
__device__ __forceinline__ double cg_ord_block(double v, double (&part)[kCgResThreads / 64])
{
    v = wave_sum_dpp(v);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    double p = part[0];
    #pragma unroll
    for (int q = 1; q < kCgResThreads / 64; ++q) p += part[q];
    return p;
}

// sum of nB workgroups' values in every thread; the first 256 threads call with
// on = true
__device__ __forceinline__ double cg_ord_fold(const double *row, int nB, bool on, double (&fold)[4])
{
    if (on) {
        const int t = threadIdx.x;
        const double x = wave_sum_dpp(t < nB ? row[t] : 0.0);
        if ((t & 63) == 0) fold[t >> 6] = x;
    }
    __syncthreads();
    return (fold[0] + fold[1]) + (fold[2] + fold[3]);
}

template <int N, int K>
__global__ __launch_bounds__(kCgResThreads) void k_cg_ord_direction(CgOrdArgs A)
{
    #pragma clang fp contract(off)
    constexpr int n1 = N + 1, np = n1 * n1, T = kCgResThreads, epb = T / np, S = kCgRow<N>, ne = S * n1;
    constexpr bool WL = 64 % np == 0;
    __shared__ double Dl[np], us[epb * ne], f1[WL ? 1 : epb * ne], f2[epb * ne], part[T / 64];
    if (A.st->done) return;  // nothing writes it during this kernel
    const int t = threadIdx.x;
    if (t < np) Dl[t] = A.D[t];
    __syncthreads();
    int tl;
    const int b = xcd_block(blockIdx.x, gridDim.x);
    const int le = lane_element<N>(t, tl), nd = lane_node<N>(tl), i = nd % n1, j = nd / n1, ls = le < epb ? le : 0;
    double *usE = us + ls * ne, *f1E = WL ? usE : f1 + ls * ne, *f2E = f2 + ls * ne;
    CgMfOps<N> M;
    if constexpr (Mf<N>::on) cg_mf_ops<N>(M, Dl, tl);
    const double beta = A.it == 1 ? 0.0 : A.st->beta;
    const size_t nLocal = (size_t)A.nE * np;
    double acc = 0.0;
    for (int k = 0; k < K; ++k) {
        const int e = (b * K + k) * epb + le;
        const bool act = le < epb && e < A.nE;
        const size_t l = act ? (size_t)e * np + nd : 0;
        const int g = act ? A.gid[l] : -1, gc = max(g, 0);
        const double g11 = act ? A.G3[l] : 0.0, g12 = act ? A.G3[nLocal + l] : 0.0,
                     g22 = act ? A.G3[2 * nLocal + l] : 0.0;
        const double r = g >= 0 ? A.r[gc] : 0.0, vo = g >= 0 && A.it > 1 ? A.vOld[gc] : 0.0;
        const double d = g >= 0 ? (A.dinv ? A.dinv[gc] : 1.0) : 0.0;
        const double v = __builtin_fma(beta, vo, d * r);
        const double L = cg_element_product<N, S, WL>(
            M, Dl, usE, f1E, f2E, v, g11, [&] { return g12; }, [&] { return g22; }, le < epb, tl, i, j);
        acc = __builtin_fma(v, L, acc);
        if (act) A.L[l] = L;
        if (g >= 0 && A.ci[A.cs[gc]] == (int)l) A.vNew[g] = v;
    }
    acc = cg_ord_block(acc, part);
    if (t == 0) A.partials[b] = acc;
}

template <int N, int K>
__global__ __launch_bounds__(kCgResThreads) void k_cg_ord_update(CgOrdArgs A)
{
    #pragma clang fp contract(off)
    constexpr int n1 = N + 1, np = n1 * n1, T = kCgResThreads, epb = T / np;
    __shared__ double part0[T / 64], part1[T / 64], fold[4];
    if (A.st->done) return;
    const int t = threadIdx.x, b = xcd_block(blockIdx.x, gridDim.x);
    const double vz = cg_ord_fold(A.partials, gridDim.x, t < 256, fold);
    const double alpha = A.st->numP[A.it & 1] / vz;
    int tl;
    const int le = lane_element<N>(t, tl), nd = lane_node<N>(tl);
    double a0 = 0.0, a1 = 0.0;
    for (int k = 0; k < K; ++k) {
        const int e = (b * K + k) * epb + le;
        if (le >= epb || e >= A.nE) continue;
        const size_t l = (size_t)e * np + nd;
        const int g = A.gid[l];
        if (g < 0) continue;
        const int c0 = A.cs[g], n = A.cs[g + 1] - c0;
        if (A.ci[c0] != (int)l) continue;
        double z = A.L[l] + (n > 1 ? A.L[A.ci[c0 + 1]] : 0.0);
        if (n > 2) z = (z + A.L[A.ci[c0 + 2]]) + (n > 3 ? A.L[A.ci[c0 + 3]] : 0.0);
        A.u[g] = __builtin_fma(alpha, A.vNew[g], A.u[g]);
        const double r = __builtin_fma(-alpha, z, A.r[g]);
        A.r[g] = r;
        a0 = __builtin_fma(r, r, a0);
        a1 = __builtin_fma(r, (A.dinv ? A.dinv[g] : 1.0) * r, a1);
    }
    a0 = cg_ord_block(a0, part0);
    a1 = cg_ord_block(a1, part1);
    if (t == 0) {
        A.partials[kRedBlocks + b] = a0;
        A.partials[2 * kRedBlocks + b] = a1;
    }
}

// one workgroup of 256: the end of iteration A.it from nB workgroups' sums
__global__ __launch_bounds__(256) void k_cg_ord_end(CgOrdArgs A, int nB)
{
    __shared__ double fold0[4], fold1[4];
    if (A.st->done) return;
    const double S0 = cg_ord_fold(A.partials + kRedBlocks, nB, true, fold0);
    const double S1 = cg_ord_fold(A.partials + 2 * kRedBlocks, nB, true, fold1);
    if (threadIdx.x == 0) cg_end_apply(A.st, A.it, S0, S1);
}

}  // namespace self
