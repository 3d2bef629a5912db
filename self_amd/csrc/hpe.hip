// hpe.hip -- the hydrostatic primitive equations (linear, Boussinesq, rigid
// lid) on a stacked hex mesh, gfx950.
//
// Reference: src/highend/hydrostaticprimitives/HydrostaticPrimitivesClass.f90
//   ForwardStepAB2 :1378-1424, GlobalTimeDerivative :1428-1506,
//   DiagnoseP :1739-1822, DiagnoseW :1826-1912,
//   CalculateBottomVerticalVelocity :1916-1945, EdgeFlux :2088-2183,
//   MappedTimeDerivative :2187-2400, RiemannSolver :2738-2778,
//   X/Y/ZFlux :2782-2832, Source :2836-2852 (zero), GetExternalState
//   :2856-2898; HydrostaticPrimitivesClass_implicit.f90 CalculateDivU
//   :2520-2691 and ForwardStepRK3 :1422-1471.  The reference class does not
//   compile; the gaps are filled as follows: divU is CalculateDivU of the
//   implicit variant, called before DiagnoseW; DiagnoseP runs inside the
//   time derivative when diagnoseP is set (the explicit class comments the
//   call out, the implicit variant makes it); the column integrals use the
//   interpolant of the Gauss nodes; the background's face values are
//   interpolated from its volume values; the steppers leave out the
//   barotropic step and the pressure correction.
//
// Variables u 0, v 1, b 2 (prognostic), w 3, p 4 (diagnosed).  Element
// e = hE + nHElems * layer (the reference's stackMap).  A stage is two
// kernels:
//   k_hpe_columns -- one workgroup per stack (a horizontal element and all
//     its layers).  Top to bottom it integrates the hydrostatic pressure
//     from the buoyancy; bottom to top it forms the divergence of the
//     lateral velocity (weak form with the element's own face values) and
//     integrates the vertical velocity up from the sea-floor value
//     -(u nx + v ny)/nz.  The reference's column quadrature (M + 1
//     Gauss-Lobatto points, M = (N+1)/2 + 1, on each sub-interval between
//     consecutive nodes) is folded on the host into two (N+1) x (N+1)
//     matrices, so each node's increment is one dot product along its
//     column line; the running sum is carried node by node in the
//     reference's order.  It writes p, w and the face values of b, w, p
//     of every element.
//   k_hpe_stage -- one workgroup per element: the Riemann flux on the six
//     faces from the face values and the face's primary normal and
//     background (computed from the primary's side so both sides see
//     exactly opposite fluxes), the weak divergence of the contravariant
//     fluxes in s, p, q with the lift, 1/J, then the RK3 or AB2 update of
//     u, v, b, or the tendency alone.
// At N = 7 both run on the FP64 matrix cores (k_hpe_columns_mf,
// k_hpe_stage_mf), the column's running sums folded into the matrices.

#include <cmath>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "common.hpp"
#include "dg3d_device.hpp"
#include "layout.hpp"

namespace self {
void cofactor3(const double *m, int dir, double out[3]);
int legendre_quadrature(int n, int type, double *x, double *w);
void barycentric(int n, const double *x, double *bw);
void lagrange_at(int n, const double *x, const double *bw, double xe, double *l);
}  // namespace self

using namespace self;

struct self_hpe_s {
    int N = 0, n1 = 0, n2 = 0, np = 0, device = 0, diagnoseP = 1;
    size_t nE = 0, nH = 0, nL = 0;
    double dt = 0.0;
    hipStream_t stream = nullptr;
    double *nodal = nullptr, *sol = nullptr, *G = nullptr, *tend = nullptr, *geo = nullptr, *height = nullptr;
    double *nrm = nullptr, *fdat = nullptr, *tr = nullptr, *Bvol = nullptr, *divU = nullptr;
    int2 *side = nullptr;
    std::vector<double> faceNrm;  // host copy of the per-side (nx, ny, nz, len) for the background face data
    std::vector<int2> sideHost;
    std::vector<double> lagL, lagR;
};

namespace {

constexpr double kRkA[3] = {0.0, -5.0 / 9.0, -153.0 / 128.0};
constexpr double kRkG[3] = {1.0 / 3.0, 15.0 / 16.0, 8.0 / 15.0};
constexpr int kNoNormalFlow = -100, kSeaFloor = -105;  // src/common/ModelFlags.f90:81-85

template <int N>
struct HShape {
    static constexpr int n1 = N + 1, n2 = n1 * n1, np = n2 * n1;
    static constexpr int threads = np < 64 ? 64 : ((np + 63) / 64) * 64;
};

// nodal constants: weak derivative matrix (column-major), 1/w, l(-1), l(+1),
// column integration rows downward and upward ([k][j], the increment of
// node k per unit column height)
template <int N>
struct HNodal {
    static constexpr int n1 = N + 1;
    double D[n1 * n1], iw[n1], lL[n1], lR[n1], Idn[n1 * n1], Iup[n1 * n1];
};

// global nodal buffer: D, w, lL, lR, Idn, Iup
template <int N>
__device__ __forceinline__ void stage_hnodal(HNodal<N> &L, const double *__restrict__ g)
{
    constexpr int n1 = N + 1, n11 = n1 * n1;
    for (int k = threadIdx.x; k < n11; k += blockDim.x) {
        L.D[k] = g[k];
        L.Idn[k] = g[n11 + 3 * n1 + k];
        L.Iup[k] = g[2 * n11 + 3 * n1 + k];
    }
    for (int k = threadIdx.x; k < n1; k += blockDim.x) {
        L.iw[k] = 1.0 / g[n11 + k];
        L.lL[k] = g[n11 + n1 + k];
        L.lR[k] = g[n11 + 2 * n1 + k];
    }
}

// The same constants in two steps around a kernel's element loads (fetch
// before them, LDS after them: the write then waits for these loads only,
// the counter of outstanding loads being in order).  LANES threads.
template <int N, int LANES>
struct HNodalRegs {
    static constexpr int n1 = N + 1, n11 = n1 * n1, nv = 3 * n11 + 3 * n1;  // D, Idn, Iup, w, lL, lR
    static constexpr int K = (nv + LANES - 1) / LANES;
    double v[K];
};

template <int N, int LANES>
__device__ __forceinline__ void hnodal_fetch(HNodalRegs<N, LANES> &R, const double *__restrict__ g, int lane)
{
    using Rg = HNodalRegs<N, LANES>;
    constexpr int n1 = Rg::n1, n11 = Rg::n11;
    #pragma unroll
    for (int q = 0; q < Rg::K; ++q) {
        const int k = min(lane + q * LANES, Rg::nv - 1);
        // buffer: D, w, lL, lR, Idn, Iup
        const int src = k < n11 ? k : (k < 3 * n11 ? k + 3 * n1 : k - 2 * n11);
        R.v[q] = g[src];
    }
}

template <int N, int LANES>
__device__ __forceinline__ void hnodal_put(HNodal<N> &L, const HNodalRegs<N, LANES> &R, int lane)
{
    using Rg = HNodalRegs<N, LANES>;
    constexpr int n1 = Rg::n1, n11 = Rg::n11;
    #pragma unroll
    for (int q = 0; q < Rg::K; ++q) {
        const int k = lane + q * LANES;
        const double v = R.v[q];
        if (k < n11) L.D[k] = v;
        else if (k < 2 * n11) L.Idn[k - n11] = v;
        else if (k < 3 * n11) L.Iup[k - 2 * n11] = v;
        else if (k < 3 * n11 + n1) L.iw[k - 3 * n11] = 1.0 / v;
        else if (k < 3 * n11 + 2 * n1) L.lL[k - 3 * n11 - n1] = v;
        else if (k < Rg::nv) L.lR[k - 3 * n11 - 2 * n1] = v;
    }
}

struct HpeArgs {
    int nE, nH, nL, diagnoseP, mode, first;
    double a, gdt, dt;
    const double *nodal, *geo, *height, *nrm, *fdat, *Bvol;
    double *sol, *G, *tend, *tr, *divU;
    const int2 *side;
};

// ---------------------------------------------------------------- columns
template <int N>
__global__ __launch_bounds__(HShape<N>::threads, 4) void k_hpe_columns(HpeArgs A)
{
    using S = HShape<N>;
    constexpr int n1 = S::n1, n2 = S::n2, np = S::np;
    __shared__ HNodal<N> L;
    __shared__ double s0[np], s1[np], s2[np], s3[np], s4[np], sd[np];
    __shared__ double fF[6 * n2], base[n2];
    stage_hnodal<N>(L, A.nodal);
    const int hE = blockIdx.x, tid = threadIdx.x;
    const bool act = tid < np;
    const int i = tid % n1, j = (tid / n1) % n1, k = tid / n2;
    const size_t NE = (size_t)A.nE, nEp = NE * np;
    const double *u = A.sol, *v = A.sol + nEp, *b = A.sol + 2 * nEp;
    double *w = A.sol + 3 * nEp, *p = A.sol + 4 * nEp;
    for (int t = tid; t < n2; t += blockDim.x) base[t] = 0.0;
    // Each layer's loads are issued one layer ahead (unconditionally, at
    // clamped addresses for threads without a node or face node), so they
    // are in flight while the layer before is integrated: the column walk
    // is otherwise one memory round trip per layer and sweep.
    const size_t tn = act ? (size_t)tid : 0, thn = (size_t)(act ? i + n1 * j : 0);
    constexpr int FQ = (6 * n2 + S::threads - 1) / S::threads;  // face nodes per thread
    // ---- DiagnoseP (top to bottom) and the face values of b and p
    double bNx, pNx = 0.0, hNx;
    {
        const size_t e0 = (size_t)hE + (size_t)A.nH * (A.nL - 1);
        bNx = b[e0 * np + tn];
        if (!A.diagnoseP) pNx = p[e0 * np + tn];
        hNx = A.height[e0 * n2 + thn];
    }
    for (int layer = A.nL - 1; layer >= 0; --layer) {
        const size_t e = (size_t)hE + (size_t)A.nH * layer;
        const double bCur = bNx, pCur = pNx, hCur = hNx;
        if (layer > 0) {
            const size_t en = e - (size_t)A.nH;
            bNx = b[en * np + tn];
            if (!A.diagnoseP) pNx = p[en * np + tn];
            hNx = A.height[en * n2 + thn];
        }
        __syncthreads();
        if (act) {
            s0[tid] = bCur;
            if (!A.diagnoseP) s1[tid] = pCur;
        }
        __syncthreads();
        if (A.diagnoseP) {
            if (act) {
                double acc = 0.0;
                #pragma unroll
                for (int m = 0; m < n1; ++m) acc = __builtin_fma(L.Idn[k * n1 + m], s0[i + n1 * (j + n1 * m)], acc);
                s2[tid] = acc * hCur;
            }
            __syncthreads();
            if (tid < n2) {
                double run = base[tid];
                for (int kk = N; kk >= 0; --kk) {
                    run = run + s2[tid + n2 * kk];
                    s1[tid + n2 * kk] = run;
                }
                double acc = 0.0;
                #pragma unroll
                for (int m = 0; m < n1; ++m) acc = __builtin_fma(L.lL[m], s1[tid + n2 * m], acc);
                base[tid] = acc;  // the bottom face value starts the layer below
            }
            __syncthreads();
            if (act) p[e * np + tid] = s1[tid];
        }
        for (int t = tid; t < 6 * n2; t += blockDim.x) {
            const int sdn = t / n2, node = t - sdn * n2, a = node % n1, bb = node / n1;
            double *o = A.tr + ((e * 6 + sdn) * 3) * n2 + node;
            o[0] = face_trace3<N>(L.lL, L.lR, s0, sdn, a, bb);
            o[2 * n2] = face_trace3<N>(L.lL, L.lR, s1, sdn, a, bb);
        }
    }
    // ---- CalculateDivU, CalculateBottomVerticalVelocity, DiagnoseW (bottom to top)
    // one layer's node values (u, v, the six cofactors that meet them, J,
    // the column height) and this thread's face node normal (nx, ny, nz, |n|)
    struct Layer {
        double u, v, g0, g1, g3, g4, g6, g7, J, h, nx[FQ], ny[FQ], nz[FQ], len[FQ];
    };
    const auto loadLayer = [&](size_t e) {
        Layer Y;
        const size_t g = e * np + tn;
        Y.u = u[g];
        Y.v = v[g];
        Y.g0 = A.geo[0 * nEp + g];
        Y.g1 = A.geo[1 * nEp + g];
        Y.g3 = A.geo[3 * nEp + g];
        Y.g4 = A.geo[4 * nEp + g];
        Y.g6 = A.geo[6 * nEp + g];
        Y.g7 = A.geo[7 * nEp + g];
        Y.J = A.geo[9 * nEp + g];
        Y.h = A.height[e * n2 + thn];
        #pragma unroll
        for (int q = 0; q < FQ; ++q) {
            const int t = tid + q * S::threads, tf = t < 6 * n2 ? t : 0;
            const int sdn = tf / n2, node = tf - sdn * n2;
            const double *nr = A.nrm + ((e * 6 + sdn) * 4) * n2 + node;
            Y.nx[q] = nr[0];
            Y.ny[q] = nr[n2];
            Y.nz[q] = nr[2 * n2];
            Y.len[q] = nr[3 * n2];
        }
        return Y;
    };
    Layer Ynx = loadLayer((size_t)hE);
    for (int layer = 0; layer < A.nL; ++layer) {
        const size_t e = (size_t)hE + (size_t)A.nH * layer;
        const Layer Y = Ynx;
        if (layer + 1 < A.nL) Ynx = loadLayer(e + (size_t)A.nH);
        __syncthreads();
        if (act) {
            s0[tid] = Y.u;
            s1[tid] = Y.v;
            s2[tid] = Y.g0 * Y.u + Y.g1 * Y.v;
            s3[tid] = Y.g3 * Y.u + Y.g4 * Y.v;
            s4[tid] = Y.g6 * Y.u + Y.g7 * Y.v;
        }
        __syncthreads();
        #pragma unroll
        for (int q = 0; q < FQ; ++q) {
            const int t = tid + q * S::threads;
            if (t >= 6 * n2) continue;
            const int sdn = t / n2, node = t - sdn * n2, a = node % n1, bb = node / n1;
            const double ub = face_trace3<N>(L.lL, L.lR, s0, sdn, a, bb);
            const double vb = face_trace3<N>(L.lL, L.lR, s1, sdn, a, bb);
            fF[sdn * n2 + node] = (ub * Y.nx[q] + vb * Y.ny[q]) * Y.len[q];
            if (layer == 0 && sdn == 4) base[node] = -(ub * Y.nx[q] + vb * Y.ny[q]) / Y.nz[q];
        }
        __syncthreads();
        if (act) {
            double ds = 0.0, dp = 0.0, dq = 0.0;
            #pragma unroll
            for (int m = 0; m < n1; ++m) {
                ds = __builtin_fma(L.D[i + n1 * m], s2[m + n1 * (j + n1 * k)], ds);
                dp = __builtin_fma(L.D[j + n1 * m], s3[i + n1 * (m + n1 * k)], dp);
                dq = __builtin_fma(L.D[k + n1 * m], s4[i + n1 * (j + n1 * m)], dq);
            }
            ds += (fF[1 * n2 + j + n1 * k] * L.lR[i] + fF[3 * n2 + j + n1 * k] * L.lL[i]) * L.iw[i];
            dp += (fF[2 * n2 + i + n1 * k] * L.lR[j] + fF[0 * n2 + i + n1 * k] * L.lL[j]) * L.iw[j];
            dq += (fF[5 * n2 + i + n1 * j] * L.lR[k] + fF[4 * n2 + i + n1 * j] * L.lL[k]) * L.iw[k];
            const double div = ((ds + dp) + dq) / Y.J;
            sd[tid] = div;
            if (A.divU) A.divU[e * np + tid] = div;
        }
        __syncthreads();
        if (act) {
            double acc = 0.0;
            #pragma unroll
            for (int m = 0; m < n1; ++m) acc = __builtin_fma(L.Iup[k * n1 + m], sd[i + n1 * (j + n1 * m)], acc);
            s2[tid] = acc * Y.h;
        }
        __syncthreads();
        if (tid < n2) {
            double run = base[tid];
            for (int kk = 0; kk <= N; ++kk) {
                run = run - s2[tid + n2 * kk];
                s3[tid + n2 * kk] = run;
            }
            double acc = 0.0;
            #pragma unroll
            for (int m = 0; m < n1; ++m) acc = __builtin_fma(L.lR[m], s3[tid + n2 * m], acc);
            base[tid] = acc;  // the top face value starts the layer above
        }
        __syncthreads();
        if (act) w[e * np + tid] = s3[tid];
        for (int t = tid; t < 6 * n2; t += blockDim.x) {
            const int sdn = t / n2, node = t - sdn * n2, a = node % n1, bb = node / n1;
            A.tr[((e * 6 + sdn) * 3 + 1) * n2 + node] = face_trace3<N>(L.lL, L.lR, s3, sdn, a, bb);
        }
    }
}

// N = 7 on the matrix cores (Mf3Ops).  One loop: iteration l integrates the
// pressure of layer nL-1-l and the vertical velocity of layer l, three
// barriers for both.  Wavefront wv owns plane k = wv of the lateral
// derivatives and plane j = wv of everything along the column, where lane and
// running value stay in registers: the increments' running sums are folded on
// the host into one matrix each (HpeColumn), and the face value that starts
// the next layer into one more row, so no thread sums for others.  The
// face values of w are formed one iteration later, behind the next barrier.
// Bound: HBM, 433 MB at 24x21x12 (90 us at the rate of a large copy).  Measured
// there: 113.7 us for the two sweeps of k_hpe_columns, 85.9 here; with the
// operands kept in registers (24 spilled) the stage as a whole was slower
// than before (292 us against 284).
struct HpeColumn {  // in the nodal buffer after Iup
    double Cdn[64], Cup[64];  // [k][m], running sums of Idn from the top, of Iup from the bottom
    double td[8], tu[8];      // their face values: lL . Cdn, lR . Cup
    double sl, sr;            // the face value of a constant
};

__global__ __launch_bounds__(512, 4) void k_hpe_columns_mf(HpeArgs A)
{
    constexpr int n1 = 8, n2 = 64, np = 512;
    __shared__ HNodal<7> L;
    __shared__ double su[kMf3Size], sv[kMf3Size], Fs[kMf3Size], Fp[kMf3Size], Fq[kMf3Size];
    __shared__ double sb[kMf3Size], sp[kMf3Size], sw[kMf3Size], sd[kMf3Size];
    __shared__ double fF[6 * n2], floor0[n2];
    stage_hnodal<7>(L, A.nodal);
    constexpr int nC = sizeof(HpeColumn) / sizeof(double);
    __shared__ HpeColumn C;
    if (threadIdx.x < nC) ((double *)&C)[threadIdx.x] = A.nodal[3 * n2 + 3 * n1 + threadIdx.x];
    const int hE = blockIdx.x, tl = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const size_t nEp = (size_t)A.nE * np;
    const double *u = A.sol, *v = A.sol + nEp, *b = A.sol + 2 * nEp;
    double *w = A.sol + 3 * nEp, *p = A.sol + 4 * nEp;
    const int qi = 4 * MfLane<7>(tl).bj + MfLane<7>(tl).c;
    // uniform address plus 32-bit lane offset: no 64-bit lane addresses to keep
    const unsigned on = 64 * wv + lane_node<7>(tl), qh = qi + 8 * wv, qn = qh + 64 * (4 * MfLane<7>(tl).bi + MfLane<7>(tl).k);
    int sdn, node;
    (void)mf3_face(wv, tl, sdn, node);
    const unsigned of = sdn * 4 * n2 + node, ot = sdn * 3 * n2 + node;
    // the next layers' loads are in flight while the current ones are integrated
    struct Layer {
        double b, p, hp, u, v, g0, g1, g3, g4, g6, g7, J, h, nx, ny, nz, len;
    };
    const auto load = [&](int l) {
        Layer Y;
        const size_t ep = (size_t)hE + (size_t)A.nH * (A.nL - 1 - l), e = (size_t)hE + (size_t)A.nH * l;
        Y.b = (b + ep * np)[qn];
        Y.p = A.diagnoseP ? 0.0 : (p + ep * np)[qn];
        Y.hp = (A.height + ep * n2)[qh];
        Y.u = (u + e * np)[on];
        Y.v = (v + e * np)[on];
        const double *g = A.geo + e * np;
        Y.g0 = g[on];
        Y.g1 = (g + nEp)[on];
        Y.g3 = (g + 3 * nEp)[on];
        Y.g4 = (g + 4 * nEp)[on];
        Y.g6 = (g + 6 * nEp)[on];
        Y.g7 = (g + 7 * nEp)[on];
        Y.J = (g + 9 * nEp)[on];
        Y.h = (A.height + e * n2)[qh];
        const double *nr = A.nrm + e * 6 * 4 * n2;
        Y.nx = nr[of];
        Y.ny = (nr + n2)[of];
        Y.nz = (nr + 2 * n2)[of];
        Y.len = (nr + 3 * n2)[of];
        return Y;
    };
    Layer Ynx = load(0);
    double baseP = 0.0, baseW = 0.0;
    __syncthreads();
    for (int l = 0; l < A.nL; ++l) {
        const size_t ep = (size_t)hE + (size_t)A.nH * (A.nL - 1 - l), e = (size_t)hE + (size_t)A.nH * l;
        // A lane number that the compiler cannot follow over iterations: the
        // addresses and operands derived from it are formed again, not kept
        // in registers (they spilled, and a spilled value's load waits for
        // the layer loads in flight).
        const bool first = l == 0;
        int lane = tl;
        asm volatile("" : "+v"(lane));
        const MfLane<7> a(lane);
        const int i = lane_node<7>(lane) % n1, j = lane_node<7>(lane) / n1, k = wv;
        const int ln = mf3_at(i, j, k), qi = 4 * a.bj + a.c, ql = mf3_q_node(wv, lane);  // own node; plane j = wv
        const int row = 4 * a.bi + a.c;  // of a left operand
        int sdn, node;
        const bool has = mf3_face(wv, lane, sdn, node);
        const Layer &X = Ynx;
        su[ln] = X.u;
        sv[ln] = X.v;
        Fs[ln] = X.g0 * X.u + X.g1 * X.v;
        Fp[ln] = X.g3 * X.u + X.g4 * X.v;
        Fq[ln] = X.g6 * X.u + X.g7 * X.v;
        sb[ql] = X.b;
        const Layer Y = X;  // J, heights and face normal are used below
        if (l + 1 < A.nL) Ynx = load(l + 1);
        double pv = Y.p;
        if (A.diagnoseP) {
            wave_sync();  // plane j = wv is this wavefront's
            double acc = 0.0, top = 0.0;
            #pragma unroll
            for (int q = 0; q < 2; ++q) {
                const double x = sb[mf3_at(qi, wv, 4 * q + a.k)];
                acc = __builtin_amdgcn_mfma_f64_4x4x4f64(C.Cdn[row * n1 + 4 * q + a.k], x, acc, 0, 0, 0);
                top = __builtin_amdgcn_mfma_f64_4x4x4f64(C.td[4 * q + a.k], x, top, 0, 0, 0);
            }
            pv = __builtin_fma(Y.hp, acc, baseP);
            baseP = __builtin_fma(Y.hp, top, C.sl * baseP);
            (p + ep * np)[qn] = pv;
        }
        sp[ql] = pv;
        __syncthreads();
        Mf3Lag ML;
        mf3_load_lag(ML, L.lL, L.lR, lane);
        {
            const double ub = mf3_trace(ML, su, wv, lane), vb = mf3_trace(ML, sv, wv, lane);
            const double un = ub * Y.nx + vb * Y.ny;
            if (has) fF[sdn * n2 + node] = un * Y.len;
            if (first && has && sdn == 4) floor0[node] = -un / Y.nz;
            const double bt = mf3_trace(ML, sb, wv, lane), pt = mf3_trace(ML, sp, wv, lane);
            const double wt = !first ? mf3_trace(ML, sw, wv, lane) : 0.0;
            if (has) {
                double *o = A.tr + ep * 18 * n2;
                o[ot] = bt;
                (o + 2 * n2)[ot] = pt;
                if (!first) (A.tr + ((e - A.nH) * 18 + 1) * n2)[ot] = wt;
            }
        }
        Mf3Ops M;
        mf3_load(M, L.D, lane);
        const double tq = mf3_q(M, Fq, wv, lane);
        Fq[ql] = tq;  // read back after the barrier
        __syncthreads();
        {
            double ds = mf3_s(M, Fs, wv, lane), dp = mf3_p(M, Fp, wv, lane), dq = Fq[ln];
            ds += (fF[1 * n2 + j + n1 * k] * L.lR[i] + fF[3 * n2 + j + n1 * k] * L.lL[i]) * L.iw[i];
            dp += (fF[2 * n2 + i + n1 * k] * L.lR[j] + fF[0 * n2 + i + n1 * k] * L.lL[j]) * L.iw[j];
            dq += (fF[5 * n2 + i + n1 * j] * L.lR[k] + fF[4 * n2 + i + n1 * j] * L.lL[k]) * L.iw[k];
            const double div = ((ds + dp) + dq) / Y.J;
            sd[ln] = div;
            if (A.divU) (A.divU + e * np)[on] = div;
        }
        __syncthreads();
        {
            if (first) baseW = floor0[qi + 8 * wv];
            double acc = 0.0, top = 0.0;
            #pragma unroll
            for (int q = 0; q < 2; ++q) {
                const double x = sd[mf3_at(qi, wv, 4 * q + a.k)];
                acc = __builtin_amdgcn_mfma_f64_4x4x4f64(C.Cup[row * n1 + 4 * q + a.k], x, acc, 0, 0, 0);
                top = __builtin_amdgcn_mfma_f64_4x4x4f64(C.tu[4 * q + a.k], x, top, 0, 0, 0);
            }
            const double wval = __builtin_fma(-Y.h, acc, baseW);
            baseW = __builtin_fma(-Y.h, top, C.sr * baseW);
            (w + e * np)[qn] = wval;
            sw[ql] = wval;
        }
    }
    __syncthreads();
    {
        const size_t e = (size_t)hE + (size_t)A.nH * (A.nL - 1);
        Mf3Lag ML;
        mf3_load_lag(ML, L.lL, L.lR, tl);
        const double wt = mf3_trace(ML, sw, wv, tl);
        if (mf3_face(wv, tl, sdn, node)) (A.tr + (e * 18 + 1) * n2)[ot] = wt;
    }
}

// ---------------------------------------------------------------- stage
// RiemannSolver (:2738-2778) with in = the primary side's state
__device__ __forceinline__ void hpe_riemann(double bIn, double wIn, double pIn, double bEx, double wEx, double pEx,
                                            double nx, double ny, double nz, double Bf, double Wf, double &f0,
                                            double &f1, double &f2)
{
    const double jump = bEx - bIn;
    const double fIn = (Bf * wIn) * nz, fEx = (Bf * wEx) * nz;
    const double uN = fmax(fabs((wIn + Wf) * nz), fabs((wEx + Wf) * nz));
    const double pa = 0.5 * (pIn + pEx);
    f0 = pa * nx;
    f1 = pa * ny;
    f2 = 0.5 * (fEx + fIn - uN * jump);
}

template <int N>
__global__ __launch_bounds__(HShape<N>::threads) void k_hpe_stage(HpeArgs A)
{
    using S = HShape<N>;
    constexpr int n1 = S::n1, n2 = S::n2, np = S::np;
    __shared__ HNodal<N> L;
    __shared__ double fl[9 * np];   // [dir s,p,q][eq u,v,b][node]
    __shared__ double su[np], sv[np];
    __shared__ double F[6 * 3 * n2];  // [side][eq][node]
    constexpr int FQ = (6 * n2 + S::threads - 1) / S::threads;  // face nodes per thread
    const size_t e = blockIdx.x;
    const int tid = threadIdx.x;
    const bool act = tid < np;
    const int i = tid % n1, j = (tid / n1) % n1, k = tid / n2;
    const size_t NE = (size_t)A.nE, nEp = NE * np, g = e * np + (act ? tid : 0);
    // Loads first, with no thread-dependent branch around them (threads
    // without a node or face node load at clamped addresses and ignore the
    // values): nodal constants, face data, node values, the RK register,
    // then the neighbours' traces addressed by the face data.
    HNodalRegs<N, S::threads> R;
    hnodal_fetch<N, S::threads>(R, A.nodal, tid);
    int2 finfo[FQ];
    double fown[FQ][3], fdat[FQ][6], fnbr[FQ][3];
    #pragma unroll
    for (int q = 0; q < FQ; ++q) {
        const int t = tid + q * S::threads, tf = t < 6 * n2 ? t : 0;
        const int sdn = tf / n2, node = tf - sdn * n2;
        finfo[q] = A.side[e * 6 + sdn];
        const double *own = A.tr + ((e * 6 + sdn) * 3) * n2 + node;
        fown[q][0] = own[0]; fown[q][1] = own[n2]; fown[q][2] = own[2 * n2];
        const double *fd = A.fdat + ((e * 6 + sdn) * 6) * n2 + node;
        #pragma unroll
        for (int c = 0; c < 6; ++c) fdat[q][c] = fd[c * n2];
    }
    const double pv = A.sol[4 * nEp + g], Bw = A.Bvol[g] * A.sol[3 * nEp + g];
    const double uu = A.sol[g], vv = A.sol[nEp + g], bb0 = A.sol[2 * nEp + g];
    double geo[9];
    #pragma unroll
    for (int c = 0; c < 9; ++c) geo[c] = A.geo[c * nEp + g];
    const double Jv = A.geo[9 * nEp + g];
    double Gold[3] = {0.0, 0.0, 0.0};
    asm volatile("" ::: "memory");  // the register after the others
    if ((A.mode == 0 && !A.first) || A.mode == 2) {
        #pragma unroll
        for (int f = 0; f < 3; ++f) Gold[f] = A.G[(size_t)f * nEp + g];
    }
    #pragma unroll
    for (int q = 0; q < FQ; ++q) {
        const int t = tid + q * S::threads, tf = t < 6 * n2 ? t : 0;
        const int node = tf % n2, a = node % n1, bq = node / n1;
        const int2 info = finfo[q];
        int na = a, nb = bq;
        if (info.x >= 0) s3_map<N>(info.y, a, bq, na, nb);
        // a boundary face node reads element 0's slot and ignores it
        const size_t nbase = info.x >= 0 ? ((size_t)info.x * 6 + s3_nbr_side(info.y)) * 3 : 0;
        const double *nbr = A.tr + nbase * n2 + na + n1 * nb;
        fnbr[q][0] = nbr[0]; fnbr[q][1] = nbr[n2]; fnbr[q][2] = nbr[2 * n2];
    }
    hnodal_put<N, S::threads>(L, R, tid);
    if (act) {
        su[tid] = uu;
        sv[tid] = vv;
        #pragma unroll
        for (int d = 0; d < 3; ++d) {
            fl[(3 * d + 0) * np + tid] = geo[3 * d + 0] * pv;
            fl[(3 * d + 1) * np + tid] = geo[3 * d + 1] * pv;
            fl[(3 * d + 2) * np + tid] = geo[3 * d + 2] * Bw;
        }
    }
    __syncthreads();
    #pragma unroll
    for (int q = 0; q < FQ; ++q) {
        const int t = tid + q * S::threads;
        if (t >= 6 * n2) continue;
        const int sdn = t / n2, node = t - sdn * n2, a = node % n1, bq = node / n1;
        const int2 info = finfo[q];
        const double bO = fown[q][0], wO = fown[q][1], pO = fown[q][2];
        const double nx = fdat[q][0], ny = fdat[q][1], nz = fdat[q][2], len = fdat[q][3], Bf = fdat[q][4],
                     Wf = fdat[q][5];
        double f0, f1, f2, sgn = 1.0;
        if (info.x >= 0) {
            const double bN = fnbr[q][0], wN = fnbr[q][1], pN = fnbr[q][2];
            if (s3_primary(info.y)) {
                hpe_riemann(bO, wO, pO, bN, wN, pN, nx, ny, nz, Bf, Wf, f0, f1, f2);
            } else {
                hpe_riemann(bN, wN, pN, bO, wO, pO, nx, ny, nz, Bf, Wf, f0, f1, f2);
                sgn = -1.0;
            }
        } else {
            double wE = 0.0;
            if (info.x == kSeaFloor) {
                const double ub = face_trace3<N>(L.lL, L.lR, su, sdn, a, bq);
                const double vb = face_trace3<N>(L.lL, L.lR, sv, sdn, a, bq);
                wE = -(wO + 2.0 * (ub * nx + vb * ny)) / nz;
            }
            // NO_NORMAL_FLOW and SEA_FLOOR: zero exterior buoyancy, interior pressure
            hpe_riemann(bO, wO, pO, 0.0, wE, pO, nx, ny, nz, Bf, Wf, f0, f1, f2);
        }
        F[(sdn * 3 + 0) * n2 + node] = sgn * (f0 * len);
        F[(sdn * 3 + 1) * n2 + node] = sgn * (f1 * len);
        F[(sdn * 3 + 2) * n2 + node] = sgn * (f2 * len);
    }
    __syncthreads();
    if (!act) return;
    double tendv[3];
    #pragma unroll
    for (int f = 0; f < 3; ++f) {
        const double *fs = fl + (0 + f) * np, *fp = fl + (3 + f) * np, *fq = fl + (6 + f) * np;
        double ds = 0.0, dp = 0.0, dq = 0.0;
        #pragma unroll
        for (int m = 0; m < n1; ++m) {
            ds = __builtin_fma(L.D[i + n1 * m], fs[m + n1 * (j + n1 * k)], ds);
            dp = __builtin_fma(L.D[j + n1 * m], fp[i + n1 * (m + n1 * k)], dp);
            dq = __builtin_fma(L.D[k + n1 * m], fq[i + n1 * (j + n1 * m)], dq);
        }
        ds += (F[(1 * 3 + f) * n2 + j + n1 * k] * L.lR[i] + F[(3 * 3 + f) * n2 + j + n1 * k] * L.lL[i]) * L.iw[i];
        dp += (F[(2 * 3 + f) * n2 + i + n1 * k] * L.lR[j] + F[(0 * 3 + f) * n2 + i + n1 * k] * L.lL[j]) * L.iw[j];
        dq += (F[(5 * 3 + f) * n2 + i + n1 * j] * L.lR[k] + F[(4 * 3 + f) * n2 + i + n1 * j] * L.lL[k]) * L.iw[k];
        tendv[f] = ((-ds - dp) - dq) / Jv;
    }
    const double sol0[3] = {uu, vv, bb0};
    #pragma unroll
    for (int f = 0; f < 3; ++f) {
        const size_t gi = (size_t)f * nEp + g;
        if (A.mode == 1) {  // the time derivative alone
            A.tend[gi] = tendv[f];
        } else if (A.mode == 0) {  // RK3 stage
            const double Gn = A.first ? tendv[f] : A.a * Gold[f] + tendv[f];
            A.G[gi] = Gn;
            A.sol[gi] = sol0[f] + A.gdt * Gn;
        } else {  // AB2 step, G the previous tendency
            const double Gn = 0.5 * (3.0 * tendv[f] - Gold[f]);
            A.sol[gi] = sol0[f] + A.dt * Gn;
            A.G[gi] = tendv[f];
        }
    }
}

// N = 7 on the matrix cores (Mf3Ops): wavefront wv owns plane k = wv for s and
// p and plane j = wv for q.  The element's own face values are formed from
// the node values it has loaded anyway (the same instructions as in
// k_hpe_columns_mf, so both sides of a face still see the same values).
// Bound: HBM, 786 MB at 24x21x12 (164 us at the rate of a large copy, which
// writes half of its bytes; this reads four in five).  Measured there: 174.0 us for
// k_hpe_stage<7> (214 registers, one workgroup a CU), 139.9 here (84, two).
__global__ __launch_bounds__(512, 4) void k_hpe_stage_mf(HpeArgs A)
{
    constexpr int n1 = 8, n2 = 64, np = 512, nl = kMf3Size;
    __shared__ HNodal<7> L;
    __shared__ double fl[9 * nl];             // [dir s,p,q][eq u,v,b][node]
    __shared__ double sq[5 * nl];             // u, v, b, w, p
    __shared__ double F[6 * 3 * n2];          // [side][eq][node]
    const size_t e = blockIdx.x;
    const int tl = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const unsigned on = 64 * wv + lane_node<7>(tl);
    const int i = lane_node<7>(tl) % n1, j = lane_node<7>(tl) / n1, k = wv, ln = mf3_at(i, j, k);
    const size_t NE = (size_t)A.nE, nEp = NE * np;
    int sdn, node;
    const bool has = mf3_face(wv, tl, sdn, node);
    const int a = node % n1, bq = node / n1;
    // loads first: nodal constants, face data, node values, the register,
    // then the neighbours' face values addressed by the face data
    HNodalRegs<7, 512> R;
    hnodal_fetch<7, 512>(R, A.nodal, threadIdx.x);
    const int2 info = (A.side + e * 6)[sdn];
    double fd[6];
    const unsigned of = sdn * 6 * n2 + node;
    #pragma unroll
    for (int c = 0; c < 6; ++c) fd[c] = (A.fdat + (e * 36 + c) * n2)[of];
    double q5[5], geo[9];
    #pragma unroll
    for (int c = 0; c < 5; ++c) q5[c] = (A.sol + c * nEp + e * np)[on];
    const double Bv = (A.Bvol + e * np)[on];
    #pragma unroll
    for (int c = 0; c < 9; ++c) geo[c] = (A.geo + c * nEp + e * np)[on];
    const double Jv = (A.geo + 9 * nEp + e * np)[on];
    double Gold[3] = {0.0, 0.0, 0.0};
    asm volatile("" ::: "memory");  // the register after the others
    if ((A.mode == 0 && !A.first) || A.mode == 2) {
        #pragma unroll
        for (int f = 0; f < 3; ++f) Gold[f] = (A.G + f * nEp + e * np)[on];
    }
    int na = a, nb = bq;
    if (info.x >= 0) s3_map<7>(info.y, a, bq, na, nb);
    // a boundary face node reads element 0's slot and ignores it
    const size_t nbase = info.x >= 0 ? ((size_t)info.x * 6 + s3_nbr_side(info.y)) * 3 : 0;
    const double *nbr = A.tr + nbase * n2 + na + n1 * nb;
    const double bN = nbr[0], wN = nbr[n2], pN = nbr[2 * n2];
    hnodal_put<7, 512>(L, R, threadIdx.x);
    #pragma unroll
    for (int c = 0; c < 5; ++c) sq[c * nl + ln] = q5[c];
    const double Bw = Bv * q5[3];
    #pragma unroll
    for (int d = 0; d < 3; ++d) {
        fl[(3 * d + 0) * nl + ln] = geo[3 * d + 0] * q5[4];
        fl[(3 * d + 1) * nl + ln] = geo[3 * d + 1] * q5[4];
        fl[(3 * d + 2) * nl + ln] = geo[3 * d + 2] * Bw;
    }
    __syncthreads();
    Mf3Lag ML;
    mf3_load_lag(ML, L.lL, L.lR, tl);
    const double bO = mf3_trace(ML, sq + 2 * nl, wv, tl), wO = mf3_trace(ML, sq + 3 * nl, wv, tl),
                 pO = mf3_trace(ML, sq + 4 * nl, wv, tl);
    double ub = 0.0, vb = 0.0;
    if (__any(info.x == kSeaFloor)) {  // the whole wavefront forms them
        ub = mf3_trace(ML, sq, wv, tl);
        vb = mf3_trace(ML, sq + nl, wv, tl);
    }
    if (has) {
        const double nx = fd[0], ny = fd[1], nz = fd[2], len = fd[3], Bf = fd[4], Wf = fd[5];
        double f0, f1, f2, sgn = 1.0;
        if (info.x >= 0) {
            if (s3_primary(info.y)) {
                hpe_riemann(bO, wO, pO, bN, wN, pN, nx, ny, nz, Bf, Wf, f0, f1, f2);
            } else {
                hpe_riemann(bN, wN, pN, bO, wO, pO, nx, ny, nz, Bf, Wf, f0, f1, f2);
                sgn = -1.0;
            }
        } else {
            double wE = 0.0;
            if (info.x == kSeaFloor) wE = -(wO + 2.0 * (ub * nx + vb * ny)) / nz;
            // NO_NORMAL_FLOW and SEA_FLOOR: zero exterior buoyancy, interior pressure
            hpe_riemann(bO, wO, pO, 0.0, wE, pO, nx, ny, nz, Bf, Wf, f0, f1, f2);
        }
        F[(sdn * 3 + 0) * n2 + node] = sgn * (f0 * len);
        F[(sdn * 3 + 1) * n2 + node] = sgn * (f1 * len);
        F[(sdn * 3 + 2) * n2 + node] = sgn * (f2 * len);
    }
    Mf3Ops M;
    mf3_load(M, L.D, tl);
    #pragma unroll
    for (int f = 0; f < 3; ++f) {
        const double tq = mf3_q(M, fl + (6 + f) * nl, wv, tl);
        fl[(6 + f) * nl + mf3_q_node(wv, tl)] = tq;  // read back after the barrier
    }
    __syncthreads();
    #pragma unroll
    for (int f = 0; f < 3; ++f) {
        double ds = mf3_s(M, fl + f * nl, wv, tl), dp = mf3_p(M, fl + (3 + f) * nl, wv, tl), dq = fl[(6 + f) * nl + ln];
        ds += (F[(1 * 3 + f) * n2 + j + n1 * k] * L.lR[i] + F[(3 * 3 + f) * n2 + j + n1 * k] * L.lL[i]) * L.iw[i];
        dp += (F[(2 * 3 + f) * n2 + i + n1 * k] * L.lR[j] + F[(0 * 3 + f) * n2 + i + n1 * k] * L.lL[j]) * L.iw[j];
        dq += (F[(5 * 3 + f) * n2 + i + n1 * j] * L.lR[k] + F[(4 * 3 + f) * n2 + i + n1 * j] * L.lL[k]) * L.iw[k];
        const double tend = ((-ds - dp) - dq) / Jv;
        double *G = A.G + f * nEp + e * np, *sol = A.sol + f * nEp + e * np;
        if (A.mode == 1) {  // the time derivative alone
            (A.tend + f * nEp + e * np)[on] = tend;
        } else if (A.mode == 0) {  // RK3 stage
            const double Gn = A.first ? tend : A.a * Gold[f] + tend;
            G[on] = Gn;
            sol[on] = q5[f] + A.gdt * Gn;
        } else {  // AB2 step, G the previous tendency
            const double Gn = 0.5 * (3.0 * tend - Gold[f]);
            sol[on] = q5[f] + A.dt * Gn;
            G[on] = tend;
        }
    }
}

#define HPE_DISPATCH_N(N_, CALL)                                                            \
    switch (N_) {                                                                           \
    case 1: { constexpr int NN = 1; CALL; } break;                                          \
    case 2: { constexpr int NN = 2; CALL; } break;                                          \
    case 3: { constexpr int NN = 3; CALL; } break;                                          \
    case 4: { constexpr int NN = 4; CALL; } break;                                          \
    case 5: { constexpr int NN = 5; CALL; } break;                                          \
    case 6: { constexpr int NN = 6; CALL; } break;                                          \
    case 7: { constexpr int NN = 7; CALL; } break;                                          \
    default: break;                                                                         \
    }

HpeArgs args_of(self_hpe_s *h)
{
    HpeArgs A{};
    A.nE = (int)h->nE;
    A.nH = (int)h->nH;
    A.nL = (int)h->nL;
    A.diagnoseP = h->diagnoseP;
    A.dt = h->dt;
    A.nodal = h->nodal;
    A.geo = h->geo;
    A.height = h->height;
    A.nrm = h->nrm;
    A.fdat = h->fdat;
    A.Bvol = h->Bvol;
    A.sol = h->sol;
    A.G = h->G;
    A.tend = h->tend;
    A.tr = h->tr;
    A.side = h->side;
    return A;
}

// The two kernels of a time derivative and update; N = 7, where a plane of 64
// nodes is a wavefront's four matrix-core tiles, has its own.  Their single sweep
// and folded sums would serve other degrees, whose kernels do not have them.
int launch_columns(self_hpe_s *h, const HpeArgs &A)
{
    HPE_DISPATCH_N(h->N, {
        if constexpr (NN == 7)
            hipLaunchKernelGGL(k_hpe_columns_mf, dim3((unsigned)h->nH), dim3(512), 0, h->stream, A);
        else
            hipLaunchKernelGGL((k_hpe_columns<NN>), dim3((unsigned)h->nH), dim3(HShape<NN>::threads), 0, h->stream, A);
    });
    SELF_HIP(hipGetLastError());
    return SELF_OK;
}

int launch_stage(self_hpe_s *h, const HpeArgs &A)
{
    HPE_DISPATCH_N(h->N, {
        if constexpr (NN == 7)
            hipLaunchKernelGGL(k_hpe_stage_mf, dim3((unsigned)h->nE), dim3(512), 0, h->stream, A);
        else
            hipLaunchKernelGGL((k_hpe_stage<NN>), dim3((unsigned)h->nE), dim3(HShape<NN>::threads), 0, h->stream, A);
    });
    SELF_HIP(hipGetLastError());
    return SELF_OK;
}

// one GlobalTimeDerivative followed by the update of `mode` (0 RK3 stage m,
// 1 tendency only, 2 AB2)
int hpe_stage(self_hpe_s *h, int mode, int m, bool keepDivU)
{
    HpeArgs A = args_of(h);
    A.mode = mode;
    A.first = (mode == 0 && m == 0) ? 1 : 0;
    A.a = mode == 0 ? kRkA[m] : 0.0;
    A.gdt = mode == 0 ? kRkG[m] * h->dt : 0.0;
    A.divU = keepDivU ? h->divU : nullptr;
    if (int rc = launch_columns(h, A)) return rc;
    return launch_stage(h, A);
}

void free_all(self_hpe_s *h)
{
    void *p[] = {h->nodal, h->sol, h->G, h->tend, h->geo, h->height, h->nrm, h->fdat, h->tr, h->Bvol, h->divU, h->side};
    for (void *q : p)
        if (q) (void)hipFree(q);
    if (h->stream) (void)hipStreamDestroy(h->stream);
}

// face value of a volume field (element-local, i fastest) at side s, node (a, b)
double host_trace(int N, const double *lL, const double *lR, const double *q, int s, int a, int b)
{
    const int n1 = N + 1;
    const double *l = (s == 1 || s == 2 || s == 5) ? lR : lL;
    int off, stride;
    if (s == 1 || s == 3) { off = n1 * (a + n1 * b); stride = 1; }
    else if (s == 0 || s == 2) { off = a + n1 * n1 * b; stride = n1; }
    else { off = a + n1 * b; stride = n1 * n1; }
    double acc = 0.0;
    for (int m = 0; m < n1; ++m) acc += l[m] * q[off + m * stride];
    return acc;
}

}  // namespace

extern "C" {

int self_hpe_create(int N, int nHElems, int nLayers, int nFaces, const int *faces, const double *cov, const double *J,
                    const double *nHat, const double *nLen, const double *bpos, const double *nodes,
                    const double *qWeight, const double *dMat, const double *lagLeft, const double *lagRight,
                    int diagnoseP, double dt, self_hpe_t *out)
try {
    SELF_REQUIRE(out && faces && cov && J && nHat && nLen && bpos && nodes && qWeight && dMat && lagLeft && lagRight,
                 SELF_ERR_ARG, "self_hpe_create: null argument");
    SELF_REQUIRE(N >= 1 && N <= 7 && nHElems >= 1 && nLayers >= 1 && nFaces >= 1, SELF_ERR_ARG,
                 "self_hpe_create: N=%d (1..7), nHElems=%d, nLayers=%d", N, nHElems, nLayers);
    const int n1 = N + 1, n2 = n1 * n1, np = n2 * n1;
    const size_t nE = (size_t)nHElems * nLayers;
    // side descriptors from the face table; bottom boundary sides are SEA_FLOOR
    std::vector<int2> sd(nE * 6, make_int2(0, 0));
    std::vector<int> seen(nE * 6, 0);
    for (int f = 0; f < nFaces; ++f) {
        const int *r = faces + 9 * (size_t)f;
        const int e1 = r[0] - 1, s1 = r[1] - 1, e2 = r[2], s2 = std::abs(r[3]) - 1;
        const int iS = r[4], jS = r[5], iI = r[6], jI = r[7], sw = r[8];
        SELF_REQUIRE(e1 >= 0 && (size_t)e1 < nE && s1 >= 0 && s1 < 6, SELF_ERR_ARG, "face %d: bad primary", f + 1);
        if (e2 > 0) {
            SELF_REQUIRE((size_t)(e2 - 1) < nE && s2 >= 0 && s2 < 6, SELF_ERR_ARG, "face %d: bad secondary", f + 1);
            SELF_REQUIRE((iI == 1 || iI == -1) && (jI == 1 || jI == -1) && (sw == 0 || sw == 1), SELF_ERR_ARG,
                         "face %d: increments/swap", f + 1);
            SELF_REQUIRE(iS == (iI > 0 ? 0 : N) && jS == (jI > 0 ? 0 : N), SELF_ERR_ARG,
                         "face %d: start must be 0 (inc 1) or N (inc -1)", f + 1);
            const int bits = (sw << 4) | ((iI < 0) << 5) | ((jI < 0) << 6);
            sd[(size_t)e1 * 6 + s1] = make_int2(e2 - 1, s2 | (1 << 3) | bits);
            sd[(size_t)(e2 - 1) * 6 + s2] = make_int2(e1, s1 | bits);
            seen[(size_t)e1 * 6 + s1]++;
            seen[(size_t)(e2 - 1) * 6 + s2]++;
        } else {
            SELF_REQUIRE(e2 < 0, SELF_ERR_ARG, "face %d: secondary element 0", f + 1);
            sd[(size_t)e1 * 6 + s1] = make_int2(s1 == 4 ? kSeaFloor : kNoNormalFlow, 1 << 3);
            seen[(size_t)e1 * 6 + s1]++;
        }
    }
    for (size_t q = 0; q < nE * 6; ++q)
        SELF_REQUIRE(seen[q] == 1, SELF_ERR_ARG, "element %zu side %zu is on %d faces", q / 6 + 1, q % 6 + 1, seen[q]);
    // geometry: cofactor rows and J; column heights; own normals
    std::vector<double> geo(10 * nE * np), height(nE * n2), nrm(nE * 6 * 4 * n2);
    for (size_t id = 0; id < nE * np; ++id) {
        SELF_REQUIRE(J[id] != 0.0, SELF_ERR_ARG, "zero Jacobian at element %zu", id / np + 1);
        for (int dir = 0; dir < 3; ++dir) {
            double cf[3];
            cofactor3(cov + 9 * id, dir, cf);
            for (int r = 0; r < 3; ++r) geo[(3 * dir + r) * nE * np + id] = cf[r];
        }
        geo[9 * nE * np + id] = J[id];
    }
    for (size_t e = 0; e < nE; ++e)
        for (int q = 0; q < n2; ++q) {
            const double zt = bpos[3 * (q + (size_t)n2 * (5 + 6 * e)) + 2];
            const double zb = bpos[3 * (q + (size_t)n2 * (4 + 6 * e)) + 2];
            height[e * n2 + q] = zt - zb;
        }
    for (size_t es = 0; es < nE * 6; ++es)
        for (int q = 0; q < n2; ++q) {
            const size_t hb = q + (size_t)n2 * es;
            for (int r = 0; r < 3; ++r) nrm[(es * 4 + r) * n2 + q] = nHat[3 * hb + r];
            nrm[(es * 4 + 3) * n2 + q] = nLen[hb];
        }
    // column integration rows: the increment of node k over the sub-interval
    // from the previous node (down: from the node above or +1; up: from the
    // node below or -1) by the M+1 point Gauss-Lobatto rule on the
    // interpolant of the Gauss nodes, times 1/2 (dz/dxi per unit height)
    const int M = (N + 1) / 2 + 1;
    std::vector<double> gx(M + 1), gw(M + 1), bw(n1), lv(n1);
    SELF_REQUIRE(legendre_quadrature(M, SELF_GAUSS_LOBATTO, gx.data(), gw.data()) == 0, SELF_ERR_ARG, "column quadrature");
    barycentric(N, nodes, bw.data());
    std::vector<double> Idn(n1 * n1, 0.0), Iup(n1 * n1, 0.0);
    for (int kk = 0; kk <= N; ++kk)
        for (int dir = 0; dir < 2; ++dir) {
            const double xiI = dir == 0 ? (kk == N ? 1.0 : nodes[kk + 1]) : (kk == 0 ? -1.0 : nodes[kk - 1]);
            const double xiIp1 = nodes[kk];
            std::vector<double> &I = dir == 0 ? Idn : Iup;
            for (int m = 0; m <= M; ++m) {
                const double xiK = 0.5 * (xiIp1 - xiI) * (gx[m] + 1.0) + xiI;
                lagrange_at(N, nodes, bw.data(), xiK, lv.data());
                for (int jj = 0; jj <= N; ++jj) I[kk * n1 + jj] += gw[m] * lv[jj];
            }
            for (int jj = 0; jj <= N; ++jj) I[kk * n1 + jj] *= 0.25 * (xiIp1 - xiI);
        }
    // running sums of the increments, their face values, a constant's face value
    HpeColumn col{};
    if (N == 7) {
        for (int m = 0; m <= N; ++m) {
            double run = 0.0;
            for (int kk = N; kk >= 0; --kk) {
                col.Cdn[kk * n1 + m] = run += Idn[kk * n1 + m];
                col.td[m] += lagLeft[kk] * run;
            }
            run = 0.0;
            for (int kk = 0; kk <= N; ++kk) {
                col.Cup[kk * n1 + m] = run += Iup[kk * n1 + m];
                col.tu[m] += lagRight[kk] * run;
            }
            col.sl += lagLeft[m];
            col.sr += lagRight[m];
        }
    }
    std::vector<double> nod(3 * n1 * n1 + 3 * n1 + sizeof(HpeColumn) / sizeof(double));
    std::memcpy(nod.data() + 3 * n1 * n1 + 3 * n1, &col, sizeof(HpeColumn));
    std::memcpy(nod.data(), dMat, sizeof(double) * n1 * n1);
    std::memcpy(nod.data() + n1 * n1, qWeight, sizeof(double) * n1);
    std::memcpy(nod.data() + n1 * n1 + n1, lagLeft, sizeof(double) * n1);
    std::memcpy(nod.data() + n1 * n1 + 2 * n1, lagRight, sizeof(double) * n1);
    std::memcpy(nod.data() + n1 * n1 + 3 * n1, Idn.data(), sizeof(double) * n1 * n1);
    std::memcpy(nod.data() + 2 * n1 * n1 + 3 * n1, Iup.data(), sizeof(double) * n1 * n1);

    auto *h = new self_hpe_s();
    h->N = N; h->n1 = n1; h->n2 = n2; h->np = np; h->nE = nE; h->nH = nHElems; h->nL = nLayers;
    h->dt = dt;
    h->diagnoseP = diagnoseP ? 1 : 0;
    h->faceNrm = nrm;
    h->sideHost = sd;
    h->lagL.assign(lagLeft, lagLeft + n1);
    h->lagR.assign(lagRight, lagRight + n1);
    hipError_t e = hipGetDevice(&h->device);
    if (e == hipSuccess) e = hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking);
    auto Mal = [&](double **p, size_t n) { if (e == hipSuccess) e = hipMalloc(p, sizeof(double) * n); };
    Mal(&h->nodal, nod.size());
    Mal(&h->sol, 5 * nE * np);
    Mal(&h->G, 3 * nE * np);
    Mal(&h->tend, 3 * nE * np);
    Mal(&h->geo, geo.size());
    Mal(&h->height, height.size());
    Mal(&h->nrm, nrm.size());
    Mal(&h->fdat, nE * 6 * 6 * n2);
    Mal(&h->tr, nE * 6 * 3 * n2);
    Mal(&h->Bvol, nE * np);
    Mal(&h->divU, nE * np);
    if (e == hipSuccess) e = hipMalloc(&h->side, sizeof(int2) * sd.size());
    if (e == hipSuccess) e = hipMemcpy(h->nodal, nod.data(), sizeof(double) * nod.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(h->geo, geo.data(), sizeof(double) * geo.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(h->height, height.data(), sizeof(double) * height.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(h->nrm, nrm.data(), sizeof(double) * nrm.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(h->side, sd.data(), sizeof(int2) * sd.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemset(h->sol, 0, sizeof(double) * 5 * nE * np);
    if (e == hipSuccess) e = hipMemset(h->G, 0, sizeof(double) * 3 * nE * np);
    if (e == hipSuccess) e = hipMemset(h->tend, 0, sizeof(double) * 3 * nE * np);
    if (e == hipSuccess) e = hipMemset(h->divU, 0, sizeof(double) * nE * np);
    if (e != hipSuccess) {
        free_all(h);
        delete h;
        return hip_fail(e, "self_hpe_create", __FILE__, __LINE__);
    }
    // zero background
    std::vector<double> zero(5 * nE * np, 0.0);
    const int rc = self_hpe_set_field(h, 1, zero.data());
    if (rc != SELF_OK) {
        self_hpe_destroy(h);
        return rc;
    }
    *out = h;
    return SELF_OK;
}
SELF_CATCH_ALL

int self_hpe_destroy(self_hpe_t h)
{
    if (!h) return SELF_OK;
    (void)hipSetDevice(h->device);
    if (h->stream) (void)hipStreamSynchronize(h->stream);
    free_all(h);
    delete h;
    return SELF_OK;
}

// field 0: solution (0:N,0:N,0:N,1:5) per element (u, v, b, w, p);
// 1: background state (same shape); 2: previous tendency of AB2 (1:3)
int self_hpe_set_field(self_hpe_t h, int field, const double *data)
try {
    SELF_REQUIRE(h && data, SELF_ERR_ARG, "null argument");
    SELF_REQUIRE(field >= 0 && field <= 2, SELF_ERR_ARG, "field %d", field);
    SELF_HIP(hipSetDevice(h->device));
    SELF_HIP(hipStreamSynchronize(h->stream));
    const size_t nE = h->nE, np = h->np, n2 = h->n2;
    const int nf = field == 2 ? 3 : 5;
    if (field != 1) {
        std::vector<double> buf((size_t)nf * nE * np);
        for (size_t e = 0; e < nE; ++e)
            for (int f = 0; f < nf; ++f)
                std::memcpy(buf.data() + ((size_t)f * nE + e) * np, data + (e * nf + f) * np, sizeof(double) * np);
        SELF_HIP(hipMemcpy(field == 0 ? h->sol : h->G, buf.data(), sizeof(double) * buf.size(),
                           hipMemcpyHostToDevice));
        return SELF_OK;
    }
    // background: the volume buoyancy and, for every element side, the face
    // data of the face's primary side at this side's node order: normal,
    // |n|, background buoyancy and vertical velocity
    std::vector<double> B(nE * np), fd(nE * 6 * 6 * n2);
    const int N = h->N, n1 = h->n1;
    for (size_t e = 0; e < nE; ++e) std::memcpy(B.data() + e * np, data + (e * 5 + 2) * np, sizeof(double) * np);
    for (size_t e = 0; e < nE; ++e)
        for (int s = 0; s < 6; ++s) {
            const int2 info = h->sideHost[e * 6 + s];
            for (int q = 0; q < (int)n2; ++q) {
                size_t pe = e;
                int ps = s, pq = q;
                if (info.x >= 0 && !s3_primary(info.y)) {
                    int na, nb;
                    s3_map_n(N, info.y, q % n1, q / n1, na, nb);
                    pe = (size_t)info.x;
                    ps = s3_nbr_side(info.y);
                    pq = na + n1 * nb;
                }
                double *o = fd.data() + ((e * 6 + s) * 6) * n2 + q;
                for (int r = 0; r < 4; ++r) o[r * n2] = h->faceNrm[((pe * 6 + ps) * 4 + r) * n2 + pq];
                o[4 * n2] = host_trace(N, h->lagL.data(), h->lagR.data(), data + (pe * 5 + 2) * np, ps, pq % n1,
                                       pq / n1);
                o[5 * n2] = host_trace(N, h->lagL.data(), h->lagR.data(), data + (pe * 5 + 3) * np, ps, pq % n1,
                                       pq / n1);
            }
        }
    SELF_HIP(hipMemcpy(h->Bvol, B.data(), sizeof(double) * B.size(), hipMemcpyHostToDevice));
    SELF_HIP(hipMemcpy(h->fdat, fd.data(), sizeof(double) * fd.size(), hipMemcpyHostToDevice));
    return SELF_OK;
}
SELF_CATCH_ALL

// field 0: solution (5 variables); 1: tendency (3); 2: divergence of the
// lateral velocity of the last time derivative (1); 3: face values of b, w,
// p of the last time derivative ([e][side][var][node])
int self_hpe_get_field(self_hpe_t h, int field, double *data)
try {
    SELF_REQUIRE(h && data, SELF_ERR_ARG, "null argument");
    SELF_REQUIRE(field >= 0 && field <= 3, SELF_ERR_ARG, "field %d", field);
    SELF_HIP(hipSetDevice(h->device));
    SELF_HIP(hipStreamSynchronize(h->stream));
    const size_t nE = h->nE, np = h->np;
    if (field == 3) {
        SELF_HIP(hipMemcpy(data, h->tr, sizeof(double) * nE * 6 * 3 * h->n2, hipMemcpyDeviceToHost));
        return SELF_OK;
    }
    const int nf = field == 0 ? 5 : field == 1 ? 3 : 1;
    const double *src = field == 0 ? h->sol : field == 1 ? h->tend : h->divU;
    return fields_to_host(src, data, nE, nf, (int)np, h->stream);
}
SELF_CATCH_ALL

int self_hpe_global_time_derivative(self_hpe_t h)
{
    SELF_REQUIRE(h, SELF_ERR_ARG, "null handle");
    SELF_HIP(hipSetDevice(h->device));
    return hpe_stage(h, 1, 0, true);
}

// method 0: RK3 (nSteps steps of three stages), 1: AB2
int self_hpe_forward_step(self_hpe_t h, int method, int nSteps, double *elapsed_ms)
{
    SELF_REQUIRE(h && nSteps >= 0 && (method == 0 || method == 1), SELF_ERR_ARG, "bad arguments");
    SELF_HIP(hipSetDevice(h->device));
    hipEvent_t e0 = nullptr, e1 = nullptr;
    if (elapsed_ms) {
        SELF_HIP(hipEventCreate(&e0));
        SELF_HIP(hipEventCreate(&e1));
        SELF_HIP(hipEventRecord(e0, h->stream));
    }
    int rc = SELF_OK;
    for (int s = 0; s < nSteps && !rc; ++s) {
        if (method == 0)
            for (int m = 0; m < 3 && !rc; ++m) rc = hpe_stage(h, 0, m, false);
        else
            rc = hpe_stage(h, 2, 0, false);
    }
    if (elapsed_ms) {
        SELF_HIP(hipEventRecord(e1, h->stream));
        SELF_HIP(hipEventSynchronize(e1));
        float ms = 0;
        SELF_HIP(hipEventElapsedTime(&ms, e0, e1));
        *elapsed_ms = ms;
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
    }
    return rc;
}

// average duration (ms) of each of the two kernels over nSteps RK3 steps,
// timed with events on the model's stream around every launch
int self_hpe_kernel_times(self_hpe_t h, int nSteps, double *avg_ms)
{
    SELF_REQUIRE(h && nSteps >= 1 && avg_ms, SELF_ERR_ARG, "bad arguments");
    SELF_HIP(hipSetDevice(h->device));
    hipEvent_t ev[3];
    for (auto &x : ev) SELF_HIP(hipEventCreate(&x));
    double tot[2] = {0.0, 0.0};
    for (int s = 0; s < nSteps; ++s)
        for (int m = 0; m < 3; ++m) {
            HpeArgs A = args_of(h);
            A.mode = 0;
            A.first = m == 0;
            A.a = kRkA[m];
            A.gdt = kRkG[m] * h->dt;
            A.divU = nullptr;
            SELF_HIP(hipEventRecord(ev[0], h->stream));
            if (int rc = launch_columns(h, A)) return rc;
            SELF_HIP(hipEventRecord(ev[1], h->stream));
            if (int rc = launch_stage(h, A)) return rc;
            SELF_HIP(hipEventRecord(ev[2], h->stream));
            SELF_HIP(hipEventSynchronize(ev[2]));
            float a = 0, b = 0;
            SELF_HIP(hipEventElapsedTime(&a, ev[0], ev[1]));
            SELF_HIP(hipEventElapsedTime(&b, ev[1], ev[2]));
            tot[0] += a;
            tot[1] += b;
        }
    for (auto &x : ev) (void)hipEventDestroy(x);
    avg_ms[0] = tot[0] / (3.0 * nSteps);
    avg_ms[1] = tot[1] / (3.0 * nSteps);
    return SELF_OK;
}

int self_hpe_synchronize(self_hpe_t h)
{
    SELF_REQUIRE(h, SELF_ERR_ARG, "null handle");
    SELF_HIP(hipStreamSynchronize(h->stream));
    return SELF_OK;
}

}  // extern "C"
