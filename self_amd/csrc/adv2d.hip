// adv2d.hip -- 2-D advection-diffusion DGSEM (BR1-type gradient) on gfx950.
//
// Reference: src/highend/advection-diffusion2d/AdvectionClass.f90
//   CalculateConcentrationGradient :1123-1264, ForwardStepRK3 :1268-1312,
//   GlobalTimeDerivative :1316-1378, EdgeFlux :1382-1478,
//   EdgeGradientFlux :1482-1563, MappedTimeDerivative :1567-1723,
//   RiemannSolver :1756-1787, XFlux/YFlux :1791-1825, Source :1829-1847,
//   GetExternalState :1851-1886.
//
// Each RK stage needs two neighbour exchanges (concentration traces for the
// central gradient flux, then gradient traces for the diffusive flux), so a
// stage is two kernels:
//   k_adv_gradient  own traces + neighbour traces -> central gradient flux
//                   -> weak gradient (dc/dx, dc/dy) -> gradient traces
//   k_adv_stage     upwind + diffusive flux of every side node, volume flux
//                   c u - kappa grad c, weak divergence + lift, relaxation
//                   source, low-storage RK3 update, traces of the new state
// Side fluxes are evaluated in the edge's primary orientation (primary
// normal, primary velocity trace, primary + secondary order in the averages)
// so each side holds exactly the value EdgeFlux/EdgeGradientFlux would store.
// Velocity is static: its traces are computed once when it is set (the
// reference recomputes them every stage).

#include <algorithm>
#include <chrono>
#include <cstring>
#include <vector>

#include "common.hpp"
#include "dg2d_device.hpp"
#include "dg2d_host.hpp"
#include "layout.hpp"
#include "persist.hpp"

namespace self {
namespace {

constexpr double kRkA[3] = {0.0, -5.0 / 9.0, -153.0 / 128.0};
constexpr double kRkB[3] = {0.0, 1.0 / 3.0, 3.0 / 4.0};
constexpr double kRkG[3] = {1.0 / 3.0, 15.0 / 16.0, 8.0 / 15.0};

struct AdvArgs {
    int nE, mode;  // mode 0: RK update, 1: tendency only
    double kappa, t, a, gdt;
    int hasRelax;
    const double *nodal;
    double *c, *G, *tend, *grad;  // grad [2][nq][nE][np]
    const double *vel;            // [2][nE][np]
    const double *fvel;           // [nE][4][2][n1]
    const double *metric, *fnrm;
    const int2 *side;
    const double *trIn;
    double *trOut;                // c traces [nE][4][nq][n1]
    double *trG;                  // gradient traces [nE][4][2][nq][n1]
    const double *relax, *rFac;   // [nq][nE][np]
};

// GetExternalState :1851-1886
__device__ __forceinline__ double adv_external(int bc, int f, double t)
{
    if (bc == -103 && f == 0) return tanh(t);  // InflowOne
    if (bc == -104 && f == 1) return tanh(t);  // InflowTwo
    return 0.0;
}

template <int N>
__device__ __forceinline__ double trace1(const NodalLDS<N> &L, const double *q, int s, int k)
{
    constexpr int n1 = N + 1;
    const double *l = (s == 0) ? L.lS : (s == 1) ? L.lE : (s == 2) ? L.lN : L.lW;
    const int off = (s == 0 || s == 2) ? k : n1 * k;
    const int stride = (s == 0 || s == 2) ? n1 : 1;
    double acc = l[0] * q[off];
    #pragma unroll
    for (int m = 1; m < n1; ++m) acc = __builtin_fma(l[m], q[off + m * stride], acc);
    return acc;
}

// The pointwise functions write their fused multiply-adds out and switch the
// compiler's contraction off: the launched and the resident form of a stage
// have the same bits.

// line contractions of one node: sum_m D(i,m) sl[m] and sum_m D(j,m) pl[m]
template <int N>
__device__ __forceinline__ void dg_lines(const NodalLDS<N> &L, const double *sl, const double *pl, int i, int j,
                                         double &a, double &b)
{
    constexpr int n1 = N + 1;
    a = L.dS[i] * sl[0];
    b = L.dP[j] * pl[0];
    #pragma unroll
    for (int m = 1; m < n1; ++m) {
        a = __builtin_fma(L.dS[i + n1 * m], sl[m], a);
        b = __builtin_fma(L.dP[j + n1 * m], pl[n1 * m], b);
    }
}

// DGSystemDerivative in s and p of one node: line contractions plus lift
template <int N>
__device__ __forceinline__ void dg_lift(const NodalLDS<N> &L, int i, int j, double bE, double bW, double bN, double bS,
                                        double &a, double &b)
{
    #pragma clang fp contract(off)
    a = __builtin_fma(__builtin_fma(bE, L.lE[i], bW * L.lW[i]), L.iwS[i], a);
    b = __builtin_fma(__builtin_fma(bN, L.lN[j], bS * L.lS[j]), L.iwP[j], b);
}

// The two sides of a side node in the edge's primary orientation (boundary:
// the external state behind it), so that both elements form the value the
// reference stores once.
struct AdvSides {
    double in, ex, dx, dy, sign;
};

// own, nbr: tracer and its gradient's two components at the node
__device__ __forceinline__ AdvSides adv_sides(int2 info, const double own[3], const double nbr[3], double ext)
{
    AdvSides o;
    const bool bnd = info.x < 0, prim = bnd || side_primary(info.y);
    const double oc = bnd ? ext : nbr[0];
    o.in = prim ? own[0] : oc;
    o.ex = prim ? oc : own[0];
    o.dx = bnd ? own[1] : (own[1] + nbr[1]) * 0.5;
    o.dy = bnd ? own[2] : (own[2] + nbr[2]) * 0.5;
    o.sign = prim ? 1.0 : -1.0;
    return o;
}

// upwind plus diffusive flux of a side node (EdgeFlux, RiemannSolver :1756-1787)
__device__ __forceinline__ double adv_side_flux(const AdvSides &o, double uN, double nx, double ny, double len,
                                                double kappa)
{
    #pragma clang fp contract(off)
    const double fl = 0.5 * __builtin_fma(uN, o.ex + o.in, -(fabs(uN) * (o.ex - o.in)));
    const double dcdn = __builtin_fma(o.dx, nx, o.dy * ny);
    return o.sign * (__builtin_fma(-kappa, dcdn, fl) * len);
}

// contravariant volume flux of c u - kappa grad c (XFlux, YFlux :1791-1825)
__device__ __forceinline__ void adv_volume_flux(double c, double u, double v, double kappa, double dx, double dy,
                                                const double met[4], double &s, double &p)
{
    #pragma clang fp contract(off)
    const double xF = __builtin_fma(c, u, -(kappa * dx)), yF = __builtin_fma(c, v, -(kappa * dy));
    s = __builtin_fma(met[3], xF, -(met[1] * yF));
    p = __builtin_fma(met[0], yF, -(met[2] * xF));
}

__device__ __forceinline__ double adv_tendency(double t1, double t2, double J, bool relax, double field, double factor,
                                               double c)
{
    #pragma clang fp contract(off)
    const double tend = (-t1 - t2) / J;
    return relax ? __builtin_fma(field - c, factor, tend) : tend;
}

template <int N, int NQ>
__global__ __launch_bounds__(256) void k_adv_traces(const double *__restrict__ q, const double *__restrict__ nodal,
                                                    double *__restrict__ out, int nE)
{
    using S = Shape<N>;
    constexpr int n1 = S::n1, np = S::np, epb = S::epb;
    __shared__ NodalLDS<N> L;
    __shared__ double qs[epb * NQ * np];
    stage_nodal<N, false>(L, nodal, nullptr, nullptr);
    const int t = threadIdx.x, le = t / np, nd = t - le * np;
    const int e = blockIdx.x * epb + le;
    const bool act = le < epb && e < nE;
    if (act)
        for (int f = 0; f < NQ; ++f) qs[(le * NQ + f) * np + nd] = q[((size_t)f * nE + e) * np + nd];
    __syncthreads();
    if (!act) return;
    for (int w = nd; w < 4 * n1; w += np) {
        const int s = w / n1, k = w - s * n1;
        for (int f = 0; f < NQ; ++f)
            out[(((size_t)e * 4 + s) * NQ + f) * n1 + k] = trace1<N>(L, qs + (le * NQ + f) * np, s, k);
    }
}

__global__ void k_adv_fvel(const double *__restrict__ velTr, const int *__restrict__ pnode, double *__restrict__ fvel,
                           int nSideNodes, int n1)
{
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= nSideNodes) return;
    const int es = q / n1, k = q - es * n1;
    const int p = pnode[q], pes = p / n1, pk = p - pes * n1;
    // velTr/fvel layout [e*4+s][2][n1]
    fvel[((size_t)es * 2 + 0) * n1 + k] = velTr[((size_t)pes * 2 + 0) * n1 + pk];
    fvel[((size_t)es * 2 + 1) * n1 + k] = velTr[((size_t)pes * 2 + 1) * n1 + pk];
}

// ---- gradient kernel: EdgeGradientFlux + CalculateConcentrationGradient + gradient traces
template <int N, int NQ>
__global__ __launch_bounds__(256) void k_adv_gradient(AdvArgs A)
{
    using S = Shape<N>;
    constexpr int n1 = S::n1, np = S::np, epb = S::epb;
    __shared__ NodalLDS<N> L;
    __shared__ double cs[epb * NQ * np], sx[epb * NQ * np], sy[epb * NQ * np], px[epb * NQ * np],
        py[epb * NQ * np], bf[epb * 4 * 2 * NQ * n1];
    stage_nodal<N, false>(L, A.nodal, nullptr, nullptr);
    const int t = threadIdx.x, le = t / np, nd = t - le * np;
    const int e = blockIdx.x * epb + le;
    const bool act = le < epb && e < A.nE;
    const int i = nd % n1, j = nd / n1;
    const size_t mstride = (size_t)A.nE * np, base = (size_t)e * np + nd;
    const int lo = le * NQ * np;
    double *bfE = bf + le * 4 * 2 * NQ * n1;  // [side][dir][f][k]
    double J = 1.0;
    if (act) {
        const double dxds = A.metric[base], dxdp = A.metric[mstride + base];
        const double dyds = A.metric[2 * mstride + base], dydp = A.metric[3 * mstride + base];
        J = A.metric[4 * mstride + base];
        for (int f = 0; f < NQ; ++f) {
            const double c = A.c[f * mstride + base];
            cs[lo + f * np + nd] = c;
            // contravariant fluxes of (c, 0) and (0, c)
            sx[lo + f * np + nd] = dydp * c;
            sy[lo + f * np + nd] = -(dxdp * c);
            px[lo + f * np + nd] = -(dyds * c);
            py[lo + f * np + nd] = dxds * c;
        }
    }
    __syncthreads();
    if (act) {
        for (int w = nd; w < 4 * n1; w += np) {
            const int sd = w / n1, k = w - sd * n1;
            const int2 info = A.side[(size_t)e * 4 + sd];
            const size_t nb = ((size_t)e * 4 + sd) * 3 * n1 + k;
            const double nx = A.fnrm[nb], ny = A.fnrm[nb + n1], len = A.fnrm[nb + 2 * n1];
            for (int f = 0; f < NQ; ++f) {
                const double own = trace1<N>(L, cs + lo + f * np, sd, k);
                double pri, sec, sign = 1.0;
                if (info.x < 0) {
                    pri = own;
                    sec = adv_external(info.x, f, A.t);
                } else {
                    const int kk = side_flip(info.y) ? N - k : k;
                    const double nbr = A.trIn[(((size_t)info.x * 4 + side_nbr_side(info.y)) * NQ + f) * n1 + kk];
                    if (side_primary(info.y)) { pri = own; sec = nbr; }
                    else { pri = nbr; sec = own; sign = -1.0; }
                }
                const double avg = 0.5 * (pri + sec);
                bfE[((sd * 2 + 0) * NQ + f) * n1 + k] = sign * (avg * nx * len);
                bfE[((sd * 2 + 1) * NQ + f) * n1 + k] = sign * (avg * ny * len);
            }
        }
    }
    __syncthreads();
    double gxv[NQ], gyv[NQ];
    if (act) {
        for (int f = 0; f < NQ; ++f) {
            const int o = lo + f * np;
            double t1, t2, u1, u2;
            dg_lines<N>(L, sx + o + n1 * j, px + o + i, i, j, t1, t2);
            dg_lift<N>(L, i, j, bfE[((1 * 2 + 0) * NQ + f) * n1 + j], bfE[((3 * 2 + 0) * NQ + f) * n1 + j],
                       bfE[((2 * 2 + 0) * NQ + f) * n1 + i], bfE[((0 * 2 + 0) * NQ + f) * n1 + i], t1, t2);
            dg_lines<N>(L, sy + o + n1 * j, py + o + i, i, j, u1, u2);
            dg_lift<N>(L, i, j, bfE[((1 * 2 + 1) * NQ + f) * n1 + j], bfE[((3 * 2 + 1) * NQ + f) * n1 + j],
                       bfE[((2 * 2 + 1) * NQ + f) * n1 + i], bfE[((0 * 2 + 1) * NQ + f) * n1 + i], u1, u2);
            gxv[f] = (t1 + t2) / J;
            gyv[f] = (u1 + u2) / J;
            A.grad[((size_t)0 * NQ + f) * mstride + base] = gxv[f];
            A.grad[((size_t)1 * NQ + f) * mstride + base] = gyv[f];
        }
    }
    __syncthreads();  // every lane is done reading sx/sy before they hold the gradient
    if (act) {
        for (int f = 0; f < NQ; ++f) {
            sx[lo + f * np + nd] = gxv[f];
            sy[lo + f * np + nd] = gyv[f];
        }
    }
    __syncthreads();
    if (act) {
        for (int w = nd; w < 4 * n1; w += np) {
            const int sd = w / n1, k = w - sd * n1;
            for (int f = 0; f < NQ; ++f) {
                A.trG[((((size_t)e * 4 + sd) * 2 + 0) * NQ + f) * n1 + k] = trace1<N>(L, sx + lo + f * np, sd, k);
                A.trG[((((size_t)e * 4 + sd) * 2 + 1) * NQ + f) * n1 + k] = trace1<N>(L, sy + lo + f * np, sd, k);
            }
        }
    }
}

// ---- stage kernel: EdgeFlux + MappedTimeDerivative + Source + RK3 update
template <int N, int NQ>
__global__ __launch_bounds__(256) void k_adv_stage(AdvArgs A)
{
    using S = Shape<N>;
    constexpr int n1 = S::n1, np = S::np, epb = S::epb;
    __shared__ NodalLDS<N> L;
    __shared__ double cs[epb * NQ * np], gx[epb * NQ * np], gy[epb * NQ * np];
    __shared__ double sC[epb * NQ * np], pC[epb * NQ * np], bf[epb * 4 * NQ * n1];
    stage_nodal<N, false>(L, A.nodal, nullptr, nullptr);
    const int t = threadIdx.x, le = t / np, nd = t - le * np;
    const int e = blockIdx.x * epb + le;
    const bool act = le < epb && e < A.nE;
    const int i = nd % n1, j = nd / n1;
    const size_t mstride = (size_t)A.nE * np, base = (size_t)e * np + nd;
    double *cE = cs + le * NQ * np, *gxE = gx + le * NQ * np, *gyE = gy + le * NQ * np;
    double *sCE = sC + le * NQ * np, *pCE = pC + le * NQ * np, *bfE = bf + le * 4 * NQ * n1;
    double c[NQ], J = 1.0;
    if (act) {
        const double dxds = A.metric[base], dxdp = A.metric[mstride + base];
        const double dyds = A.metric[2 * mstride + base], dydp = A.metric[3 * mstride + base];
        J = A.metric[4 * mstride + base];
        const double u = A.vel[base], v = A.vel[mstride + base];
        for (int f = 0; f < NQ; ++f) {
            c[f] = A.c[f * mstride + base];
            const double dx = A.grad[((size_t)0 * NQ + f) * mstride + base];
            const double dy = A.grad[((size_t)1 * NQ + f) * mstride + base];
            cE[f * np + nd] = c[f];
            gxE[f * np + nd] = dx;
            gyE[f * np + nd] = dy;
            const double met[4] = {dxds, dxdp, dyds, dydp};
            adv_volume_flux(c[f], u, v, A.kappa, dx, dy, met, sCE[f * np + nd], pCE[f * np + nd]);
        }
    }
    __syncthreads();
    if (act) {
        for (int w = nd; w < 4 * n1; w += np) {
            const int sd = w / n1, k = w - sd * n1;
            const int2 info = A.side[(size_t)e * 4 + sd];
            const size_t nb = ((size_t)e * 4 + sd) * 3 * n1 + k;
            const double nx = A.fnrm[nb], ny = A.fnrm[nb + n1], len = A.fnrm[nb + 2 * n1];
            const double u = A.fvel[(((size_t)e * 4 + sd) * 2 + 0) * n1 + k];
            const double v = A.fvel[(((size_t)e * 4 + sd) * 2 + 1) * n1 + k];
            const double uN = __builtin_fma(u, nx, v * ny);
            for (int f = 0; f < NQ; ++f) {
                const double ownC = trace1<N>(L, cE + f * np, sd, k);
                const double ownX = trace1<N>(L, gxE + f * np, sd, k);
                const double ownY = trace1<N>(L, gyE + f * np, sd, k);
                AdvSides o;
                o.sign = 1.0;
                if (info.x < 0) {
                    o.in = ownC; o.ex = adv_external(info.x, f, A.t); o.dx = ownX; o.dy = ownY;
                } else {
                    const int kk = side_flip(info.y) ? N - k : k;
                    const size_t ns = (size_t)info.x * 4 + side_nbr_side(info.y);
                    const double nbC = A.trIn[(ns * NQ + f) * n1 + kk];
                    const double nbX = A.trG[((ns * 2 + 0) * NQ + f) * n1 + kk];
                    const double nbY = A.trG[((ns * 2 + 1) * NQ + f) * n1 + kk];
                    if (side_primary(info.y)) {
                        o.in = ownC; o.ex = nbC; o.dx = (ownX + nbX) * 0.5; o.dy = (ownY + nbY) * 0.5;
                    } else {
                        o.in = nbC; o.ex = ownC; o.dx = (nbX + ownX) * 0.5; o.dy = (nbY + ownY) * 0.5; o.sign = -1.0;
                    }
                }
                bfE[(sd * NQ + f) * n1 + k] = adv_side_flux(o, uN, nx, ny, len, A.kappa);
            }
        }
    }
    __syncthreads();
    if (act) {
        for (int f = 0; f < NQ; ++f) {
            double t1, t2;
            dg_lines<N>(L, sCE + f * np + n1 * j, pCE + f * np + i, i, j, t1, t2);
            dg_lift<N>(L, i, j, bfE[(1 * NQ + f) * n1 + j], bfE[(3 * NQ + f) * n1 + j], bfE[(2 * NQ + f) * n1 + i],
                       bfE[(0 * NQ + f) * n1 + i], t1, t2);
            const double tend = adv_tendency(t1, t2, J, A.hasRelax, A.hasRelax ? A.relax[f * mstride + base] : 0.0,
                                             A.hasRelax ? A.rFac[f * mstride + base] : 0.0, c[f]);
            if (A.mode == 1) {
                A.tend[f * mstride + base] = tend;
            } else {
                const double gold = (A.a != 0.0) ? A.G[f * mstride + base] : 0.0;
                const double gv = __builtin_fma(A.a, gold, tend);
                A.G[f * mstride + base] = gv;
                const double qn = __builtin_fma(A.gdt, gv, c[f]);
                A.c[f * mstride + base] = qn;
                cE[f * np + nd] = qn;
            }
        }
    }
    if (A.mode == 1) return;
    __syncthreads();
    if (act) {
        for (int w = nd; w < 4 * n1; w += np) {
            const int sd = w / n1, k = w - sd * n1;
            for (int f = 0; f < NQ; ++f)
                A.trOut[(((size_t)e * 4 + sd) * NQ + f) * n1 + k] = trace1<N>(L, cE + f * np, sd, k);
        }
    }
}

// ---- several RK3 steps in one launch, for models whose every element is
// resident at once.  The launched stage is two kernels (4.6 us each with their
// gaps for 10x10, N = 7: launch latency) that pass gradient, state and traces
// through memory.  Here tracers, register and geometry stay in registers and
// the two exchanges of a stage travel as tagged messages into the neighbours'
// slots (persist.hpp); contractions that need no neighbour run while they are
// under way.  One buffer each is enough: a neighbour sends its next tracer
// traces only after my gradient traces, which I send after reading its
// tracers, and its next gradient traces after my next tracers.  Measured, us a
// stage: 10x10 N = 7 8.1 -> 3.4, 61x45 N = 4 of three tracers 19.2 -> 7.9,
// 40x40 N = 3 of four 14.5 -> 6.0; a call of one step 26.8 -> 20.
struct AdvStepsArgs {
    PersistArgs P;
    int nStages;
    unsigned tag0;          // tag of the first stage
    int first;              // steps of the call before this launch's
    double tn, dt;          // tn: start of the call
    double a[3], b[3], gc[3];
    double *cOut;
    ll_quad *llC, *llG;     // [nE][NQ][4 n1], [nE][2 NQ][4 n1]
    unsigned bytesC;        // of llC; llG has twice as many
};

// Workgroups a CU decide up to which size a model is resident: where two registers
// stand between three and two of them, three are asked for.
template <int N, int NQ>
constexpr int kAdvWaves = NQ == 1 && (N == 1 || N > 6) ? 3 : 1;

template <int N, int NQ>
__global__ __launch_bounds__(256, (kAdvWaves<N, NQ>)) void k_adv_steps(AdvArgs A, AdvStepsArgs T)
{
    using S = Shape<N>;
    constexpr int n1 = S::n1, np = S::np, epb = S::epb, ns4 = 4 * n1, kSide = (ns4 + np - 1) / np;
    constexpr bool WL = 64 % np == 0;
    __shared__ NodalLDS<N> L;
    __shared__ double cs[epb * NQ * np], sx[epb * NQ * np], sy[epb * NQ * np], px[epb * NQ * np],
        py[epb * NQ * np], bf[epb * 4 * 2 * NQ * n1];
    __shared__ int stop;
    if (threadIdx.x == 0) stop = persist_given_up(T.P);
    stage_nodal<N, false>(L, A.nodal, nullptr, nullptr);
    __syncthreads();
    if (stop) return;  // an earlier launch of this model gave up: leave the state to the host
    auto sync = [] {
        if constexpr (WL) wave_sync();
        else __syncthreads();
    };
    const int t = threadIdx.x, le = t / np, nd = t - le * np;
    const int e = xcd_block(blockIdx.x, gridDim.x) * epb + le;
    const bool act = le < epb && e < A.nE;
    const int i = nd % n1, j = nd / n1;
    const size_t mstride = (size_t)A.nE * np, base = act ? (size_t)e * np + nd : 0;
    const int lo = (le < epb ? le : 0) * NQ * np;
    double *bfE = bf + (le < epb ? le : 0) * 4 * 2 * NQ * n1;
    const LLBuf llC(T.llC, T.bytesC), llG(T.llG, 2 * T.bytesC);
    double c[NQ], G[NQ], met[4];
    #pragma unroll
    for (int k = 0; k < 4; ++k) met[k] = A.metric[k * mstride + base];
    const double J = A.metric[4 * mstride + base], u = A.vel[base], v = A.vel[mstride + base];
    #pragma unroll
    for (int f = 0; f < NQ; ++f) {
        c[f] = A.c[f * mstride + base];
        G[f] = 0.0;
        if (act) cs[lo + f * np + nd] = c[f];
    }
    // the thread's side nodes: descriptor, normal, normal velocity, own and neighbour's tracers
    int2 info[kSide];
    double nx[kSide], ny[kSide], len[kSide], uN[kSide], ownC[kSide][NQ], nbC[kSide][NQ], ownX[kSide][NQ], ownY[kSide][NQ];
    bool side[kSide];
    #pragma unroll
    for (int q = 0; q < kSide; ++q) {
        const int w = nd + q * np;
        side[q] = act && w < ns4;
        const int sd = side[q] ? w / n1 : 0, k = side[q] ? w - sd * n1 : 0;
        const size_t es = (size_t)(act ? e : 0) * 4 + sd, nb = es * 3 * n1 + k;
        info[q] = A.side[es];
        nx[q] = A.fnrm[nb];
        ny[q] = A.fnrm[nb + n1];
        len[q] = A.fnrm[nb + 2 * n1];
        uN[q] = __builtin_fma(A.fvel[(es * 2) * n1 + k], nx[q], A.fvel[(es * 2 + 1) * n1 + k] * ny[q]);
    }
    // byte offset of value f of the neighbour's side node that matches mine
    auto dest = [&](int q, int nf, int f) {
        const int w = nd + q * np, k = w % n1;
        const int kk = side_nbr_side(info[q].y) * n1 + (side_flip(info[q].y) ? N - k : k);
        return 16u * (((unsigned)info[q].x * nf + f) * ns4 + kk);
    };
    auto mine = [&](int q, int nf, int f) {
        return side[q] ? 16u * (((unsigned)e * nf + f) * ns4 + nd + q * np) : 0u;
    };
    auto send_c = [&](unsigned tag) {
        #pragma unroll
        for (int q = 0; q < kSide; ++q) {
            if (!side[q]) continue;
            const int w = nd + q * np, sd = w / n1, k = w - sd * n1;
            #pragma unroll
            for (int f = 0; f < NQ; ++f) {
                ownC[q][f] = trace1<N>(L, cs + lo + f * np, sd, k);
                if (info[q].x >= 0) ll_store1(llC, dest(q, NQ, f), ownC[q][f], tag);
            }
        }
    };
    sync();
    send_c(T.tag0);
    int rk = 0;
    double tStep = T.tn + (double)T.first * T.dt;
    for (int st = 0, step = T.first; st < T.nStages; ++st) {
        #pragma clang fp contract(off)
        const unsigned tag = T.tag0 + st;
        const double time = tStep + (rk == 0 ? T.b[0] : rk == 1 ? T.b[1] : T.b[2]) * T.dt;
        bool good = true;
        // ---- contractions of the gradient
        if (act) {
            #pragma unroll
            for (int f = 0; f < NQ; ++f) {
                sx[lo + f * np + nd] = met[3] * c[f];
                sy[lo + f * np + nd] = -(met[1] * c[f]);
                px[lo + f * np + nd] = -(met[2] * c[f]);
                py[lo + f * np + nd] = met[0] * c[f];
            }
        }
        sync();
        double x1[NQ], x2[NQ], y1[NQ], y2[NQ];
        if (act) {
            #pragma unroll
            for (int f = 0; f < NQ; ++f) {
                const int o = lo + f * np;
                dg_lines<N>(L, sx + o + n1 * j, px + o + i, i, j, x1[f], x2[f]);
                dg_lines<N>(L, sy + o + n1 * j, py + o + i, i, j, y1[f], y2[f]);
            }
        }
        // ---- neighbours' tracers, central gradient flux
        #pragma unroll
        for (int q = 0; q < kSide; ++q) {
            good = ll_wait(side[q] && info[q].x >= 0, T.P, [&] {
                unsigned wrong = 0, w1;
                #pragma unroll
                for (int f = 0; f < NQ; ++f) {
                    nbC[q][f] = ll_load1(llC, mine(q, NQ, f), tag, w1);
                    wrong |= w1;
                }
                return (wrong >> 16) == 0;
            }) && good;
            if (side[q]) {
                const int w = nd + q * np, sd = w / n1, k = w - sd * n1;
                #pragma unroll
                for (int f = 0; f < NQ; ++f) {
                    const double ext = info[q].x < 0 ? adv_external(info[q].x, f, time) : 0.0;
                    const double own[3] = {ownC[q][f], 0.0, 0.0}, nbr[3] = {nbC[q][f], 0.0, 0.0};
                    const AdvSides o = adv_sides(info[q], own, nbr, ext);
                    const double avg = 0.5 * (o.in + o.ex);
                    bfE[((sd * 2 + 0) * NQ + f) * n1 + k] = o.sign * (avg * nx[q] * len[q]);
                    bfE[((sd * 2 + 1) * NQ + f) * n1 + k] = o.sign * (avg * ny[q] * len[q]);
                }
            }
        }
        if constexpr (WL) {
            if (!good) return;  // the whole wavefront, and no workgroup barrier follows
            wave_sync();
        } else {
            if (__syncthreads_or(!good)) return;
        }
        // ---- gradient, its traces on their way, contravariant volume flux
        double gx[NQ], gy[NQ];
        if (act) {
            #pragma unroll
            for (int f = 0; f < NQ; ++f) {
                dg_lift<N>(L, i, j, bfE[((1 * 2 + 0) * NQ + f) * n1 + j], bfE[((3 * 2 + 0) * NQ + f) * n1 + j],
                           bfE[((2 * 2 + 0) * NQ + f) * n1 + i], bfE[((0 * 2 + 0) * NQ + f) * n1 + i], x1[f], x2[f]);
                dg_lift<N>(L, i, j, bfE[((1 * 2 + 1) * NQ + f) * n1 + j], bfE[((3 * 2 + 1) * NQ + f) * n1 + j],
                           bfE[((2 * 2 + 1) * NQ + f) * n1 + i], bfE[((0 * 2 + 1) * NQ + f) * n1 + i], y1[f], y2[f]);
                gx[f] = (x1[f] + x2[f]) / J;
                gy[f] = (y1[f] + y2[f]) / J;
                // Every lane is past its contractions: the arrays of the gradient's
                // flux take the gradient (sx, sy, until the next stage) and the volume
                // flux (py, px).
                sx[lo + f * np + nd] = gx[f];
                sy[lo + f * np + nd] = gy[f];
            }
        }
        sync();
        #pragma unroll
        for (int q = 0; q < kSide; ++q) {
            if (!side[q]) continue;
            const int w = nd + q * np, sd = w / n1, k = w - sd * n1;
            #pragma unroll
            for (int f = 0; f < NQ; ++f) {
                ownX[q][f] = trace1<N>(L, sx + lo + f * np, sd, k);
                ownY[q][f] = trace1<N>(L, sy + lo + f * np, sd, k);
                if (info[q].x >= 0) {
                    ll_store1(llG, dest(q, 2 * NQ, f), ownX[q][f], tag);
                    ll_store1(llG, dest(q, 2 * NQ, NQ + f), ownY[q][f], tag);
                }
            }
        }
        sync();  // every lane is past its traces of the gradient
        if (act) {
            #pragma unroll
            for (int f = 0; f < NQ; ++f)
                adv_volume_flux(c[f], u, v, A.kappa, gx[f], gy[f], met, py[lo + f * np + nd], px[lo + f * np + nd]);
        }
        sync();
        if (act) {
            #pragma unroll
            for (int f = 0; f < NQ; ++f)
                dg_lines<N>(L, py + lo + f * np + n1 * j, px + lo + f * np + i, i, j, x1[f], x2[f]);
        }
        // ---- neighbours' gradients, upwind and diffusive flux
        #pragma unroll
        for (int q = 0; q < kSide; ++q) {
            double nb[2 * NQ];
            good = ll_wait(side[q] && info[q].x >= 0, T.P, [&] {
                unsigned wrong = 0, w1;
                #pragma unroll
                for (int f = 0; f < 2 * NQ; ++f) {
                    nb[f] = ll_load1(llG, mine(q, 2 * NQ, f), tag, w1);
                    wrong |= w1;
                }
                return (wrong >> 16) == 0;
            }) && good;
            if (side[q]) {
                const int w = nd + q * np, sd = w / n1, k = w - sd * n1;
                #pragma unroll
                for (int f = 0; f < NQ; ++f) {
                    const double ext = info[q].x < 0 ? adv_external(info[q].x, f, time) : 0.0;
                    const double own[3] = {ownC[q][f], ownX[q][f], ownY[q][f]}, nbr[3] = {nbC[q][f], nb[f], nb[NQ + f]};
                    bfE[(sd * NQ + f) * n1 + k] = adv_side_flux(adv_sides(info[q], own, nbr, ext), uN[q], nx[q], ny[q], len[q],
                                                                A.kappa);
                }
            }
        }
        if constexpr (WL) {
            if (!good) return;
            wave_sync();
        } else {
            if (__syncthreads_or(!good)) return;
        }
        // ---- lift, source, RK3 update
        if (act) {
            const double ra = rk == 0 ? T.a[0] : rk == 1 ? T.a[1] : T.a[2];
            const double gdt = (rk == 0 ? T.gc[0] : rk == 1 ? T.gc[1] : T.gc[2]) * T.dt;
            #pragma unroll
            for (int f = 0; f < NQ; ++f) {
                dg_lift<N>(L, i, j, bfE[(1 * NQ + f) * n1 + j], bfE[(3 * NQ + f) * n1 + j], bfE[(2 * NQ + f) * n1 + i],
                           bfE[(0 * NQ + f) * n1 + i], x1[f], x2[f]);
                const double tend = adv_tendency(x1[f], x2[f], J, A.hasRelax, A.hasRelax ? A.relax[f * mstride + base] : 0.0,
                                                 A.hasRelax ? A.rFac[f * mstride + base] : 0.0, c[f]);
                G[f] = __builtin_fma(ra, ra != 0.0 ? G[f] : 0.0, tend);
                c[f] = __builtin_fma(gdt, G[f], c[f]);
                cs[lo + f * np + nd] = c[f];
            }
        }
        if (++rk == 3) {
            rk = 0;
            tStep = T.tn + (double)(++step) * T.dt;
        }
        sync();
        if (st + 1 < T.nStages) send_c(tag + 1);
    }
    if (act) {
        // the model's gradient is the last stage's, as the launched stages leave it
        #pragma unroll
        for (int f = 0; f < NQ; ++f) {
            T.cOut[f * mstride + base] = c[f];
            A.grad[f * mstride + base] = sx[lo + f * np + nd];
            A.grad[(NQ + f) * mstride + base] = sy[lo + f * np + nd];
        }
    }
}

}  // namespace
}  // namespace self

using namespace self;

struct self_adv2d_s {
    int N = 0, n1 = 0, np = 0, nq = 0, device = 0;
    size_t nE = 0;
    double kappa = 0.0, dt = 0.0;
    hipStream_t stream = nullptr;
    double *nodal = nullptr, *c = nullptr, *G = nullptr, *tend = nullptr, *grad = nullptr, *vel = nullptr;
    double *velTr = nullptr, *fvel = nullptr, *metric = nullptr, *fnrm = nullptr, *tr[2] = {nullptr, nullptr};
    double *trG = nullptr, *relax = nullptr, *rFac = nullptr;
    int2 *side = nullptr;
    int *pnode = nullptr;
    int cur = 0;
    bool trValid = false, ready = false, hasRelax = false;
    // several steps in one launch (k_adv_steps): second state, messages, launches in flight
    double *cAlt = nullptr;
    ResidentRuns runs;
};

namespace {

#define ADV_DISPATCH(N_, NQ_, CALL)                                                         \
    switch ((N_) * 10 + (NQ_)) {                                                            \
    case 11: { constexpr int NN = 1, QQ = 1; CALL; } break;                                 \
    case 21: { constexpr int NN = 2, QQ = 1; CALL; } break;                                 \
    case 31: { constexpr int NN = 3, QQ = 1; CALL; } break;                                 \
    case 41: { constexpr int NN = 4, QQ = 1; CALL; } break;                                 \
    case 51: { constexpr int NN = 5, QQ = 1; CALL; } break;                                 \
    case 61: { constexpr int NN = 6, QQ = 1; CALL; } break;                                 \
    case 71: { constexpr int NN = 7, QQ = 1; CALL; } break;                                 \
    case 81: { constexpr int NN = 8, QQ = 1; CALL; } break;                                 \
    case 12: { constexpr int NN = 1, QQ = 2; CALL; } break;                                 \
    case 22: { constexpr int NN = 2, QQ = 2; CALL; } break;                                 \
    case 32: { constexpr int NN = 3, QQ = 2; CALL; } break;                                 \
    case 42: { constexpr int NN = 4, QQ = 2; CALL; } break;                                 \
    case 52: { constexpr int NN = 5, QQ = 2; CALL; } break;                                 \
    case 62: { constexpr int NN = 6, QQ = 2; CALL; } break;                                 \
    case 72: { constexpr int NN = 7, QQ = 2; CALL; } break;                                 \
    case 82: { constexpr int NN = 8, QQ = 2; CALL; } break;                                 \
    case 13: { constexpr int NN = 1, QQ = 3; CALL; } break;                                 \
    case 23: { constexpr int NN = 2, QQ = 3; CALL; } break;                                 \
    case 33: { constexpr int NN = 3, QQ = 3; CALL; } break;                                 \
    case 43: { constexpr int NN = 4, QQ = 3; CALL; } break;                                 \
    case 53: { constexpr int NN = 5, QQ = 3; CALL; } break;                                 \
    case 63: { constexpr int NN = 6, QQ = 3; CALL; } break;                                 \
    case 73: { constexpr int NN = 7, QQ = 3; CALL; } break;                                 \
    case 83: { constexpr int NN = 8, QQ = 3; CALL; } break;                                 \
    case 14: { constexpr int NN = 1, QQ = 4; CALL; } break;                                 \
    case 24: { constexpr int NN = 2, QQ = 4; CALL; } break;                                 \
    case 34: { constexpr int NN = 3, QQ = 4; CALL; } break;                                 \
    case 44: { constexpr int NN = 4, QQ = 4; CALL; } break;                                 \
    case 54: { constexpr int NN = 5, QQ = 4; CALL; } break;                                 \
    case 64: { constexpr int NN = 6, QQ = 4; CALL; } break;                                 \
    case 74: { constexpr int NN = 7, QQ = 4; CALL; } break;                                 \
    case 84: { constexpr int NN = 8, QQ = 4; CALL; } break;                                 \
    default: break;                                                                         \
    }

template <int N>
int agrid(size_t nE) { return (int)((nE + Shape<N>::epb - 1) / Shape<N>::epb); }

AdvArgs adv_args(self_adv2d_s *h)
{
    AdvArgs A{};
    A.nE = (int)h->nE;
    A.kappa = h->kappa;
    A.hasRelax = h->hasRelax;
    A.nodal = h->nodal;
    A.c = h->c;
    A.G = h->G;
    A.tend = h->tend;
    A.grad = h->grad;
    A.vel = h->vel;
    A.fvel = h->fvel;
    A.metric = h->metric;
    A.fnrm = h->fnrm;
    A.side = h->side;
    A.trG = h->trG;
    A.relax = h->relax;
    A.rFac = h->rFac;
    return A;
}

int launch_c_traces(self_adv2d_s *h, double *dst)
{
    ADV_DISPATCH(h->N, h->nq, hipLaunchKernelGGL((k_adv_traces<NN, QQ>), dim3(agrid<NN>(h->nE)), dim3(256), 0,
                                                 h->stream, h->c, h->nodal, dst, (int)h->nE));
    SELF_HIP(hipGetLastError());
    return SELF_OK;
}

int stage(self_adv2d_s *h, double t, int m, int mode)
{
    AdvArgs A = adv_args(h);
    A.t = t;
    A.mode = mode;
    A.a = m >= 0 ? kRkA[m] : 0.0;
    A.gdt = m >= 0 ? kRkG[m] * h->dt : 0.0;
    A.trIn = h->tr[h->cur];
    A.trOut = h->tr[1 - h->cur];
    ADV_DISPATCH(h->N, h->nq, hipLaunchKernelGGL((k_adv_gradient<NN, QQ>), dim3(agrid<NN>(h->nE)), dim3(256), 0,
                                                 h->stream, A));
    ADV_DISPATCH(h->N, h->nq, hipLaunchKernelGGL((k_adv_stage<NN, QQ>), dim3(agrid<NN>(h->nE)), dim3(256), 0,
                                                 h->stream, A));
    SELF_HIP(hipGetLastError());
    if (mode == 0) h->cur = 1 - h->cur;
    return SELF_OK;
}

// ---- several steps in one launch
size_t ll_quads(const self_adv2d_s *h) { return h->nE * (size_t)h->nq * 4 * h->n1; }  // of the tracers' messages

template <int N, int NQ>
int resident_blocks(self_adv2d_s *h, int &perCu, size_t &blocks)
{
    perCu = persist_blocks_per_cu(reinterpret_cast<const void *>(&k_adv_steps<N, NQ>), 256);
    blocks = (size_t)agrid<N>(h->nE);
    return perCu >= 1 && 32 * ll_quads(h) < (1u << 31) && blocks <= (size_t)perCu * persist_cus(h->device);
}

// Buffers of the resident form, at creation, where the model fits it; without
// memory for them it keeps to the ordinary launches, which need none.
int resident_prepare(self_adv2d_s *h)
{
    int fits = 0, perCu = 0;
    size_t blocks = 0;
    ADV_DISPATCH(h->N, h->nq, fits = (resident_blocks<NN, QQ>(h, perCu, blocks)));
    h->runs.off = !fits;
    if (!fits) return SELF_OK;
    h->runs.messageBytes = 3 * sizeof(ll_quad) * ll_quads(h);
    if (hipMalloc(reinterpret_cast<void **>(&h->cAlt), sizeof(double) * h->nq * h->nE * h->np) != hipSuccess ||
        hipMalloc(reinterpret_cast<void **>(&h->runs.messages), h->runs.messageBytes) != hipSuccess ||
        hipMalloc(reinterpret_cast<void **>(&h->runs.status), sizeof(int)) != hipSuccess ||
        h->runs.alloc_host() != hipSuccess) {
        (void)hipGetLastError();
        if (h->cAlt) (void)hipFree(h->cAlt);
        if (h->runs.messages) (void)hipFree(h->runs.messages);
        h->cAlt = nullptr;
        h->runs.messages = nullptr;
        h->runs.off = true;
        return SELF_OK;
    }
    return h->runs.clear(h->stream);
}

template <int N, int NQ>
int launch_steps(self_adv2d_s *h, double tn, int first, int nSteps)
{
    int perCu = 0;
    size_t blocks = 0;
    (void)resident_blocks<N, NQ>(h, perCu, blocks);
    AdvArgs A = adv_args(h);
    AdvStepsArgs T{};
    T.P = h->runs.args();
    T.nStages = 3 * nSteps;
    T.tag0 = h->runs.tag + 1;
    T.first = first;
    T.tn = tn;
    T.dt = h->dt;
    for (int m = 0; m < 3; ++m) {
        T.a[m] = kRkA[m];
        T.b[m] = kRkB[m];
        T.gc[m] = kRkG[m];
    }
    T.cOut = h->cAlt;
    T.llC = h->runs.messages;
    T.llG = h->runs.messages + ll_quads(h);
    T.bytesC = (unsigned)(sizeof(ll_quad) * ll_quads(h));
    h->runs.pending.reserve(h->runs.pending.size() + 1);  // nothing fails between the launch and its record
    PersistGate gate(h->device, h->stream, (int)blocks, perCu);
    if (gate.rc) return gate.rc;
    hipLaunchKernelGGL((k_adv_steps<N, NQ>), dim3((unsigned)blocks), dim3(256), 0, h->stream, A, T);
    SELF_HIP(hipGetLastError());
    h->runs.launched(first, nSteps, tn, h->c);
    std::swap(h->c, h->cAlt);
    h->trValid = false;
    return gate.launched();
}

// steps first .. nSteps - 1 of a call that begins at tn
int launched_steps(self_adv2d_s *h, double tn, int first, int nSteps)
{
    int rc = SELF_OK;
    if (!h->trValid) {
        if ((rc = launch_c_traces(h, h->tr[h->cur]))) return rc;
        h->trValid = true;
    }
    for (int s = first; s < nSteps && !rc; ++s) {
        const double t0 = tn + s * h->dt;
        for (int m = 0; m < 3 && !rc; ++m) rc = stage(h, t0 + kRkB[m] * h->dt, m, 0);
    }
    return rc;
}

// Every call but a further ForwardStepRK3 settles the launches in flight first.
int settle(self_adv2d_s *h)
{
    if (h->runs.pending.empty()) return SELF_OK;
    SELF_HIP(hipSetDevice(h->device));
    std::vector<ResidentRuns::Run> again;
    if (int rc = h->runs.settle(h->stream, again)) return rc;
    if (again.empty()) return SELF_OK;
    if (h->c != again[0].in) std::swap(h->c, h->cAlt);
    h->trValid = false;
    for (const auto &r : again)
        if (int rc = launched_steps(h, r.t0, r.first, r.first + r.steps)) return rc;
    SELF_HIP(hipStreamSynchronize(h->stream));
    return SELF_OK;
}

void to_dev(const double *src, double *dst, size_t nE, int nf, int np)
{
    for (size_t e = 0; e < nE; ++e)
        for (int f = 0; f < nf; ++f)
            std::memcpy(dst + ((size_t)f * nE + e) * np, src + (e * nf + f) * np, sizeof(double) * np);
}

}  // namespace

extern "C" {

int self_adv2d_create(int N, int nTracers, int nElems, int nEdges, const int *edges, const double *dxds,
                      const double *dxdp, const double *dyds, const double *dydp, const double *J, const double *nHat,
                      const double *nLen, const double *dMatS, const double *dMatP, const double *qWeight,
                      const double *lagWest, const double *lagEast, const double *lagSouth, const double *lagNorth,
                      double kappa, double dt, self_adv2d_t *out)
try {
    SELF_REQUIRE(out && edges && dxds && dxdp && dyds && dydp && J && nHat && nLen && dMatS && dMatP && qWeight &&
                     lagWest && lagEast && lagSouth && lagNorth,
                 SELF_ERR_ARG, "self_adv2d_create: null argument");
    SELF_REQUIRE(N >= 1 && N <= 8 && nTracers >= 1 && nTracers <= 4 && nElems >= 1, SELF_ERR_ARG,
                 "self_adv2d_create: N=%d (1..8), nTracers=%d (1..4)", N, nTracers);
    Geo2D G;
    int rc = build_geo2d(N, (size_t)nElems, nEdges, edges, dxds, dxdp, dyds, dydp, J, nHat, nLen, G);
    if (rc) return rc;
    auto *h = new self_adv2d_s();
    h->N = N;
    h->n1 = N + 1;
    h->np = h->n1 * h->n1;
    h->nq = nTracers;
    h->nE = (size_t)nElems;
    h->kappa = kappa;
    h->dt = dt;
    const size_t nE = h->nE, np = h->np, n1 = h->n1, nq = h->nq;
    auto fail = [&](hipError_t e) {
        void *p[] = {h->nodal, h->c, h->G, h->tend, h->grad, h->vel, h->velTr, h->fvel, h->metric, h->fnrm,
                     h->tr[0], h->tr[1], h->trG, h->relax, h->rFac, h->side, h->pnode, h->cAlt, h->runs.messages, h->runs.status};
        for (void *q : p)
            if (q) (void)hipFree(q);
        h->runs.free_host();
        if (h->stream) (void)hipStreamDestroy(h->stream);
        delete h;
        return hip_fail(e, "self_adv2d_create", __FILE__, __LINE__);
    };
    hipError_t e = hipGetDevice(&h->device);
    if (e == hipSuccess) e = hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking);
    auto M = [&](double **p, size_t n) { if (e == hipSuccess) e = hipMalloc(p, sizeof(double) * n); };
    M(&h->nodal, nodal_buffer_size(n1));
    M(&h->c, nq * nE * np);
    M(&h->G, nq * nE * np);
    M(&h->tend, nq * nE * np);
    M(&h->grad, 2 * nq * nE * np);
    M(&h->vel, 2 * nE * np);
    M(&h->velTr, nE * 8 * n1);
    M(&h->fvel, nE * 8 * n1);
    M(&h->metric, 5 * nE * np);
    M(&h->fnrm, nE * 12 * n1);
    M(&h->tr[0], nE * 4 * nq * n1);
    M(&h->tr[1], nE * 4 * nq * n1);
    M(&h->trG, nE * 8 * nq * n1);
    if (e == hipSuccess) e = hipMalloc(&h->side, sizeof(int2) * nE * 4);
    if (e == hipSuccess) e = hipMalloc(&h->pnode, sizeof(int) * nE * 4 * n1);
    if (e != hipSuccess) return fail(e);
    std::vector<double> nod(nodal_buffer_size(n1));
    std::memcpy(nod.data(), dMatS, sizeof(double) * n1 * n1);
    std::memcpy(nod.data() + n1 * n1, dMatP, sizeof(double) * n1 * n1);
    double *p = nod.data() + 2 * n1 * n1;
    std::memcpy(p, qWeight, sizeof(double) * n1);
    std::memcpy(p + n1, qWeight, sizeof(double) * n1);
    std::memcpy(p + 2 * n1, lagWest, sizeof(double) * n1);
    std::memcpy(p + 3 * n1, lagEast, sizeof(double) * n1);
    std::memcpy(p + 4 * n1, lagSouth, sizeof(double) * n1);
    std::memcpy(p + 5 * n1, lagNorth, sizeof(double) * n1);
    nodal_buffer_derived(nod.data(), n1);
    std::vector<int2> sd(nE * 4);
    for (size_t k = 0; k < nE * 4; ++k) sd[k] = make_int2(G.sideX[k], G.sideY[k]);
    e = hipMemcpy(h->nodal, nod.data(), sizeof(double) * nod.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(h->metric, G.metric.data(), sizeof(double) * G.metric.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(h->fnrm, G.fnrm.data(), sizeof(double) * G.fnrm.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(h->side, sd.data(), sizeof(int2) * sd.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(h->pnode, G.primaryNode.data(), sizeof(int) * G.primaryNode.size(),
                                       hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemset(h->c, 0, sizeof(double) * nq * nE * np);
    if (e == hipSuccess) e = hipMemset(h->vel, 0, sizeof(double) * 2 * nE * np);
    if (e == hipSuccess) e = hipMemset(h->fvel, 0, sizeof(double) * nE * 8 * n1);
    if (e != hipSuccess) return fail(e);
    if (resident_prepare(h) != SELF_OK) return fail(hipErrorUnknown);
    *out = h;
    return SELF_OK;
}
SELF_CATCH_ALL

int self_adv2d_destroy(self_adv2d_t h)
{
    if (!h) return SELF_OK;
    (void)hipSetDevice(h->device);
    if (h->stream) (void)hipStreamSynchronize(h->stream);
    void *p[] = {h->nodal, h->c, h->G, h->tend, h->grad, h->vel, h->velTr, h->fvel, h->metric, h->fnrm,
                 h->tr[0], h->tr[1], h->trG, h->relax, h->rFac, h->side, h->pnode, h->cAlt, h->runs.messages, h->runs.status};
    for (void *q : p)
        if (q) (void)hipFree(q);
    h->runs.free_host();
    if (h->stream) (void)hipStreamDestroy(h->stream);
    delete h;
    return SELF_OK;
}

// field: 0 concentration (0:N,0:N,1:nTracers), 1 velocity (0:N,0:N,1:2),
// 2 relaxation field, 3 relaxation factor (both (0:N,0:N,1:nTracers))
int self_adv2d_set_field(self_adv2d_t h, int field, const double *data)
try {
    SELF_REQUIRE(h && data, SELF_ERR_ARG, "null argument");
    SELF_HIP(hipSetDevice(h->device));
    if (int rc = settle(h)) return rc;
    SELF_HIP(hipStreamSynchronize(h->stream));
    const size_t nE = h->nE, np = h->np;
    const int nf = field == 1 ? 2 : h->nq;
    std::vector<double> buf((size_t)nf * nE * np);
    to_dev(data, buf.data(), nE, nf, (int)np);
    double **dst = nullptr;
    switch (field) {
    case 0: dst = &h->c; h->trValid = false; break;
    case 1: dst = &h->vel; break;
    case 2: dst = &h->relax; h->hasRelax = true; break;
    case 3: dst = &h->rFac; h->hasRelax = true; break;
    default: SELF_REQUIRE(false, SELF_ERR_ARG, "field %d", field);
    }
    if (!*dst) SELF_HIP(hipMalloc(dst, sizeof(double) * buf.size()));
    SELF_HIP(hipMemcpy(*dst, buf.data(), sizeof(double) * buf.size(), hipMemcpyHostToDevice));
    if (field == 2 || field == 3) {
        if (!h->relax) { SELF_HIP(hipMalloc(&h->relax, sizeof(double) * buf.size())); SELF_HIP(hipMemset(h->relax, 0, sizeof(double) * buf.size())); }
        if (!h->rFac) { SELF_HIP(hipMalloc(&h->rFac, sizeof(double) * buf.size())); SELF_HIP(hipMemset(h->rFac, 0, sizeof(double) * buf.size())); }
    }
    if (field == 1) {  // CalculateVelocityAtBoundaries, once: velocity is static
        const int N = h->N;
        ADV_DISPATCH(N, 2, hipLaunchKernelGGL((k_adv_traces<NN, QQ>), dim3(agrid<NN>(nE)), dim3(256), 0, h->stream,
                                              h->vel, h->nodal, h->velTr, (int)nE));
        const int nsn = (int)(nE * 4 * h->n1);
        hipLaunchKernelGGL(k_adv_fvel, dim3((nsn + 255) / 256), dim3(256), 0, h->stream, h->velTr, h->pnode, h->fvel,
                           nsn, h->n1);
        SELF_HIP(hipGetLastError());
        SELF_HIP(hipStreamSynchronize(h->stream));
    }
    return SELF_OK;
}
SELF_CATCH_ALL

// field: 0 concentration, 1 tendency, 2 dc/dx, 3 dc/dy, 4 velocity
// (0:N,0:N,1:2), 5 relaxation field, 6 relaxation factor (zero if never set)
int self_adv2d_get_field(self_adv2d_t h, int field, double *data)
try {
    SELF_REQUIRE(h && data, SELF_ERR_ARG, "null argument");
    SELF_HIP(hipSetDevice(h->device));
    if (int rc = settle(h)) return rc;
    SELF_HIP(hipStreamSynchronize(h->stream));
    const size_t nE = h->nE, np = h->np;
    size_t nq = h->nq;
    const double *src = nullptr;
    switch (field) {
    case 0: src = h->c; break;
    case 1: src = h->tend; break;
    case 2: src = h->grad; break;
    case 3: src = h->grad + nq * nE * np; break;
    case 4: src = h->vel; nq = 2; break;
    case 5: src = h->relax; break;
    case 6: src = h->rFac; break;
    default: SELF_REQUIRE(false, SELF_ERR_ARG, "field %d", field);
    }
    if (!src) {  // a field never set holds zeros, as the reference's Build leaves it
        std::memset(data, 0, sizeof(double) * nq * nE * np);
        return SELF_OK;
    }
    return fields_to_host(src, data, nE, (int)nq, (int)np, h->stream);
}
SELF_CATCH_ALL

int self_adv2d_global_time_derivative(self_adv2d_t h, double t)
try {
    SELF_REQUIRE(h, SELF_ERR_ARG, "null handle");
    SELF_HIP(hipSetDevice(h->device));
    int rc = settle(h);
    if (!rc) rc = launch_c_traces(h, h->tr[h->cur]);
    if (rc) return rc;
    h->trValid = true;
    return stage(h, t, -1, 1);
}
SELF_CATCH_ALL

int self_adv2d_forward_step_rk3(self_adv2d_t h, double tn, int nSteps, double *elapsed_ms)
try {
    SELF_REQUIRE(h && nSteps >= 0, SELF_ERR_ARG, "bad arguments");
    SELF_HIP(hipSetDevice(h->device));
    int rc = SELF_OK;
    const bool resident = !h->runs.off && nSteps >= 1 && h->runs.ups.tries();
    if (!resident || elapsed_ms)
        if ((rc = settle(h))) return rc;
    if (!resident && !h->trValid) {
        if ((rc = launch_c_traces(h, h->tr[h->cur]))) return rc;
        h->trValid = true;
    }
    hipEvent_t e0 = nullptr, e1 = nullptr;
    if (elapsed_ms) {
        SELF_HIP(hipEventCreate(&e0));
        SELF_HIP(hipEventCreate(&e1));
        SELF_HIP(hipEventRecord(e0, h->stream));
    }
    int s = 0;
    while (resident && s < nSteps && !rc) {
        if (h->runs.pending.size() >= 64) rc = settle(h);
        if (rc || h->runs.ups.rest > 0) break;
        const int n = std::min(nSteps - s, kPersistMaxSteps);
        ADV_DISPATCH(h->N, h->nq, rc = (launch_steps<NN, QQ>(h, tn, s, n)));
        s += n;
    }
    if (!rc && s < nSteps) {
        rc = settle(h);
        if (!rc) rc = launched_steps(h, tn, s, nSteps);
    }
    if (elapsed_ms) {
        SELF_HIP(hipEventRecord(e1, h->stream));
        SELF_HIP(hipEventSynchronize(e1));
        float ms = 0;
        SELF_HIP(hipEventElapsedTime(&ms, e0, e1));
        *elapsed_ms = ms;
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        const int gaveUp = h->runs.ups.total;
        const auto t0 = std::chrono::steady_clock::now();
        if (!rc) rc = settle(h);
        if (h->runs.ups.total != gaveUp)  // the steps ran (again) in there
            *elapsed_ms += std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    }
    return rc;
}
SELF_CATCH_ALL

// WritePickup_Advection (AdvectionClass.f90:2040-2103)
int self_adv2d_write_pickup(self_adv2d_t h, const char *path)
try {
    SELF_REQUIRE(h && path, SELF_ERR_ARG, "null argument");
    const size_t nv = h->nE * h->np, q = (size_t)h->nq;
    std::vector<double> c(q * nv), relax(q * nv), rFac(q * nv), vel(2 * nv);
    int rc = self_adv2d_get_field(h, 0, c.data());
    if (!rc) rc = self_adv2d_get_field(h, 5, relax.data());
    if (!rc) rc = self_adv2d_get_field(h, 6, rFac.data());
    if (!rc) rc = self_adv2d_get_field(h, 4, vel.data());
    if (!rc) rc = self_adv2d_pickup_write(path, h->N, (int)h->nE, h->nq, c.data(), relax.data(), rFac.data(), vel.data());
    return rc;
}
SELF_CATCH_ALL

// ReadPickup_Advection (:2107-2171): solution, relaxation field and factor, velocity
int self_adv2d_read_pickup(self_adv2d_t h, const char *path)
try {
    SELF_REQUIRE(h && path, SELF_ERR_ARG, "null argument");
    const size_t nv = h->nE * h->np, q = (size_t)h->nq;
    std::vector<double> c(q * nv), relax(q * nv), rFac(q * nv), vel(2 * nv);
    int rc = self_adv2d_pickup_read(path, h->N, (int)h->nE, h->nq, c.data(), relax.data(), rFac.data(), vel.data());
    if (!rc) rc = self_adv2d_set_field(h, 0, c.data());
    if (!rc) rc = self_adv2d_set_field(h, 2, relax.data());
    if (!rc) rc = self_adv2d_set_field(h, 3, rFac.data());
    if (!rc) rc = self_adv2d_set_field(h, 1, vel.data());
    return rc;
}
SELF_CATCH_ALL

int self_adv2d_resident_counts(self_adv2d_t h, int *launches, int *gaveUp)
try {
    SELF_REQUIRE(h && launches && gaveUp, SELF_ERR_ARG, "null argument");
    if (int rc = settle(h)) return rc;
    *launches = h->runs.ups.launches;
    *gaveUp = h->runs.ups.total;
    return SELF_OK;
}
SELF_CATCH_ALL

int self_adv2d_synchronize(self_adv2d_t h)
try {
    SELF_REQUIRE(h, SELF_ERR_ARG, "null handle");
    SELF_HIP(hipStreamSynchronize(h->stream));
    return settle(h);
}
SELF_CATCH_ALL

}  // extern "C"
