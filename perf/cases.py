"""Workloads timed on the GPU, each through the framework's public classes.

Every case is what a driver program does between two outputs: it holds a
model whose state is on the device, advances it by `steps` RK3 steps (or
solves one elliptic problem) and fetches the result.  Sizes are those of the
repository's benchmark, tests and request stream, plus odd meshes and degrees
in between.  exact() gives the same result in 64 bits from plain torch code
that shares nothing with the framework: the discretisations restated on
structured meshes as dense products along each axis.
"""
import math

import numpy as np
import torch

RK_A = (0.0, -5.0 / 9.0, -153.0 / 128.0)
RK_G = (1.0 / 3.0, 15.0 / 16.0, 8.0 / 15.0)
GRAV, F0, LSW = 9.81, 1.0e-4, 1.0e6


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # a small request of the mixed stream (8..64 squared, N = 3, 5, 7; 200 steps): launch latency
        {"name": "sw_16x16_n3", "kind": "sw", "nX": 16, "nY": 16, "N": 3, "prec": "fp64", "drag": 0.0, "steps": 200},
        # the headline configuration, in the reference's arithmetic and in the mixed form
        {"name": "sw_64x64_n7", "kind": "sw", "nX": 64, "nY": 64, "N": 7, "prec": "fp64", "drag": 0.0, "steps": 500},
        {"name": "sw_64x64_n7_mixed", "kind": "sw", "nX": 64, "nY": 64, "N": 7, "prec": "mixed", "drag": 0.0,
         "steps": 500},
        # a basin-scale run on an odd mesh, even degree, with bottom drag: state beyond the caches of one XCD
        {"name": "sw_187x141_n6_drag", "kind": "sw", "nX": 187, "nY": 141, "N": 6, "prec": "fp64", "drag": 0.05,
         "steps": 100},
        # the 2-D advection-diffusion benchmark: 100 elements, 100 steps
        {"name": "adv2d_10x10_n7", "kind": "adv2d", "nX": 10, "nY": 10, "N": 7, "nq": 1, "warp": 0.0, "relax": False,
         "steps": 100},
        # several tracers relaxed toward a climatology on a curved odd mesh
        {"name": "adv2d_61x45_n4_q3", "kind": "adv2d", "nX": 61, "nY": 45, "N": 4, "nq": 3, "warp": 0.03,
         "relax": True, "steps": 100},
        # the 3-D advection benchmark: warped mesh, adaptive roll-off filter at every stage
        {"name": "adv3d_32x32x16_n7", "kind": "adv3d", "nX": 32, "nY": 32, "nZ": 16, "N": 7, "nq": 1, "steps": 100},
        # the reference's default degree and tracer count on an odd box
        {"name": "adv3d_19x13x11_n5_q2", "kind": "adv3d", "nX": 19, "nY": 13, "nZ": 11, "N": 5, "nq": 2, "steps": 100},
        # the hydrostatic model at the benchmark's degree: 504 columns of 12 layers
        {"name": "hpe_24x21x12_n7", "kind": "hpe", "nX": 24, "nY": 21, "nZ": 12, "N": 7, "steps": 100},
        # the elliptic solver: a small request of the stream, the benchmark, and FGMRES(30) with the FEM preconditioner
        {"name": "cgsem_16x16_n3", "kind": "cgsem", "nX": 16, "nY": 16, "N": 3, "method": "cgsem_pcg"},
        {"name": "cgsem_128x128_n7", "kind": "cgsem", "nX": 128, "nY": 128, "N": 7, "method": "cgsem_pcg"},
        {"name": "cgsem_45x33_n5_fgmres", "kind": "cgsem", "nX": 45, "nY": 33, "N": 5, "method": "pcgmres"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["sw", "sw", "adv2d", "adv3d", "hpe", "cgsem", "cgsem"])
    if kind == "sw":
        N = rng.randint(2, 10)
        top = 1.6e6 / (N + 1) ** 2
        nX = _log(rng, 6, math.sqrt(top))
        nY = _log(rng, 6, min(4 * nX, top / nX))
        nodes = nX * nY * (N + 1) ** 2
        return {"kind": kind, "nX": nX, "nY": nY, "N": N, "prec": rng.choice(["fp64", "mixed"]),
                "drag": rng.choice([0.0, 0.05]), "steps": max(40, min(500, int(1.2e8 / nodes)))}
    if kind == "adv2d":
        N = rng.randint(2, 8)
        nX = _log(rng, 5, 80)
        nY = _log(rng, 5, 80)
        nq = rng.randint(1, 4)
        return {"kind": kind, "nX": nX, "nY": nY, "N": N, "nq": nq, "warp": rng.choice([0.0, 0.03]),
                "relax": rng.choice([False, True]), "steps": 100}
    if kind == "adv3d":
        N = rng.randint(2, 7)
        top = 6.0e6 / (N + 1) ** 3
        nX = _log(rng, 4, min(48, top ** (1 / 3) * 1.3))
        nY = _log(rng, 4, min(48, math.sqrt(top / nX)))
        nZ = _log(rng, 3, max(4, min(32, top / (nX * nY))))
        return {"kind": kind, "nX": nX, "nY": nY, "nZ": nZ, "N": N, "nq": rng.randint(1, 2),
                "steps": max(20, min(100, int(2.0e8 / (nX * nY * nZ * (N + 1) ** 3))))}
    if kind == "hpe":
        N = rng.randint(2, 7)
        top = 2.5e6 / (N + 1) ** 3
        nX = _log(rng, 4, min(48, top ** (1 / 3) * 1.3))
        nY = _log(rng, 4, min(48, math.sqrt(top / nX)))
        nZ = _log(rng, 2, max(3, min(24, top / (nX * nY))))
        return {"kind": kind, "nX": nX, "nY": nY, "nZ": nZ, "N": N,
                "steps": max(20, min(100, int(2.0e8 / (nX * nY * nZ * (N + 1) ** 3))))}
    N = rng.randint(3, 8)
    nX = _log(rng, 8, 100)
    nY = _log(rng, 8, 100)
    return {"kind": "cgsem", "nX": nX, "nY": nY, "N": N, "method": rng.choice(["cgsem_pcg", "cgsem_pcg", "pcgmres"])}


# ------------------------------------------------------------ 1-D operators
def _lagrange(nodes, x):
    """Values at the points x of the Lagrange polynomials through nodes."""
    n = len(nodes)
    out = np.ones((len(x), n))
    for m in range(n):
        for k in range(n):
            if k != m:
                out[:, m] *= (x - nodes[k]) / (nodes[m] - nodes[k])
    return out


def _derivative(nodes):
    n = len(nodes)
    bw = np.array([1.0 / np.prod([nodes[m] - nodes[k] for k in range(n) if k != m]) for m in range(n)])
    D = np.zeros((n, n))
    for i in range(n):
        for j in range(n):
            if i != j:
                D[i, j] = bw[j] / bw[i] / (nodes[i] - nodes[j])
        D[i, i] = -D[i].sum()
    return D


class _Gauss:
    """Legendre-Gauss nodes, weights, strong and weak derivative matrices, end values."""

    def __init__(self, N):
        self.x, self.w = np.polynomial.legendre.leggauss(N + 1)
        if N == 3:  # the model's four-point rule lists its inner nodes in descending order
            self.x = self.x[[0, 2, 1, 3]]
        self.D = _derivative(self.x)
        self.Dw = -(self.D.T * self.w[None, :]) / self.w[:, None]
        self.l = _lagrange(self.x, np.array([-1.0, 1.0]))


def _gll(N):
    """Legendre-Gauss-Lobatto nodes and weights by Newton's method on (1 - x^2) P_N'."""
    c = np.zeros(N + 1)
    c[N] = 1.0
    P = np.polynomial.legendre.Legendre(c)
    x = -np.cos(np.pi * np.arange(N + 1) / N)
    for _ in range(60):
        x[1:-1] -= P.deriv(1)(x[1:-1]) / P.deriv(2)(x[1:-1])
    return x, 2.0 / (N * (N + 1) * P(x) ** 2)


def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _t(a):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=_dev())


def _along(a, M, dim):
    """M applied to a along one axis."""
    return (a.movedim(dim, -1) @ M.T).movedim(-1, dim)


def _unit(n, nodes):
    """Positions in [0, 1] of the nodes of n equal cells: (n, N+1)."""
    return (np.arange(n)[:, None] + 0.5 * (nodes[None, :] + 1.0)) / n


# ---------------------------------------------------------------- the inputs
def _sw_inputs(case, seed):
    """Geostrophic anomaly of the free surface over random Fourier bathymetry, [Y, X, field, j, i]."""
    g, rng = _Gauss(case["N"]), np.random.default_rng([seed, 1])
    x = LSW * _unit(case["nX"], g.x)[None, :, None, :]
    y = LSW * _unit(case["nY"], g.x)[:, None, :, None]
    h = 1000.0 + 0.0 * (x + y)
    for _ in range(8):
        m, n = rng.integers(-4, 5, 2)
        h = h + rng.uniform(0, 6.25) * np.cos(2 * np.pi * (m * x + n * y) / LSW + rng.uniform(0, 2 * np.pi))
    xc, yc = LSW * rng.uniform(0.35, 0.65, 2)
    wd = 1.0e5
    eta = rng.uniform(0.8, 1.2) * np.exp(-((x - xc) ** 2 + (y - yc) ** 2) / wd ** 2)
    u = (GRAV / F0) * 2.0 * (y - yc) / wd ** 2 * eta
    v = -(GRAV / F0) * 2.0 * (x - xc) / wd ** 2 * eta
    H = h + eta
    lam = np.max(np.maximum(np.abs(u), np.abs(v)) + np.sqrt(GRAV * H))
    dt = 0.5 * min(LSW / case["nX"], LSW / case["nY"]) / ((case["N"] + 1) ** 2 * lam)
    return np.stack([H * u, H * v, H], axis=2), h, float(dt)


def _blobs(rng, dist2, n, lo, hi):
    out = 0.0
    for _ in range(n):
        out = out + rng.uniform(0.5, 1.0) * np.exp(-dist2(rng.uniform(0.3, 0.7, 3)) / (2.0 * rng.uniform(lo, hi) ** 2))
    return out


def _geo2(case, s, p):
    """Warped unit square: positions and d(x, y)/d(s, p), [Y, X, j, i] for reference points s (i) and p (j)."""
    nX, nY, w, tp = case["nX"], case["nY"], case["warp"], 2 * np.pi
    a, b = _unit(nX, s)[None, :, None, :], _unit(nY, p)[:, None, :, None]
    S, Sa, Sb = np.sin(tp * a) * np.sin(tp * b), tp * np.cos(tp * a) * np.sin(tp * b), tp * np.sin(tp * a) * np.cos(tp * b)
    one = np.ones_like(S)
    return (a + w * S, b + w * S, (1 + w * Sa) * 0.5 / nX, w * Sb * 0.5 / nY * one, w * Sa * 0.5 / nX * one,
            (1 + w * Sb) * 0.5 / nY)


def _adv2d_inputs(case, seed):
    g, rng = _Gauss(case["N"]), np.random.default_rng([seed, 2])
    x, y = _geo2(case, g.x, g.x)[:2]
    c = np.stack([_blobs(rng, lambda q: (x - q[0]) ** 2 + (y - q[1]) ** 2, 2, 0.08, 0.15) for _ in range(case["nq"])],
                 axis=2)
    a = rng.uniform(0.05, 0.2)
    u = 1.0 + a * np.sin(2 * np.pi * y)
    v = 0.5 + a * np.sin(2 * np.pi * x)
    relax = 0.5 + 0.1 * c if case["relax"] else None
    n2, kappa = (case["N"] + 1) ** 2, 1.0e-3
    nm = max(case["nX"], case["nY"])
    dt = min(1.0e-4, 0.2 / (n2 * 2.0 * nm), 0.04 / (kappa * n2 * n2 * nm * nm))
    return c, u, v, relax, kappa, dt


WARP3, SIGN3, VEL3 = 0.05, (1, -1, 1), (1.0, 0.7, 0.3)


def _geo3(case, s, p, q):
    """Warped unit cube: positions [3] and covariant terms [3][3] (row: coordinate, column: direction), [Z, Y, X, k, j, i]."""
    n, tp = (case["nX"], case["nY"], case["nZ"]), 2 * np.pi
    r = (_unit(n[0], s)[None, None, :, None, None, :], _unit(n[1], p)[None, :, None, None, :, None],
         _unit(n[2], q)[:, None, None, :, None, None])
    sn, cs = [np.sin(tp * a) for a in r], [tp * np.cos(tp * a) for a in r]
    S = sn[0] * sn[1] * sn[2]
    dS = (cs[0] * sn[1] * sn[2], sn[0] * cs[1] * sn[2], sn[0] * sn[1] * cs[2])
    X = [r[d] + WARP3 * SIGN3[d] * S for d in range(3)]
    cov = [[(WARP3 * SIGN3[d] * dS[k] + (1.0 if k == d else 0.0)) * 0.5 / n[k] for k in range(3)] for d in range(3)]
    return X, cov


def _adv3d_inputs(case, seed):
    g, rng = _Gauss(case["N"]), np.random.default_rng([seed, 3])
    (x, y, z), _ = _geo3(case, g.x, g.x, g.x)
    c = np.stack([_blobs(rng, lambda q: (x - q[0]) ** 2 + (y - q[1]) ** 2 + (z - q[2]) ** 2, 3, 0.06, 0.12)
                  for _ in range(case["nq"])], axis=3)
    rate = sum(u * n for u, n in zip(VEL3, (case["nX"], case["nY"], case["nZ"])))
    return c, 0.5 / ((case["N"] + 1) ** 2 * rate)


HDEPTH, HBACK = 0.1, 1.0


def _hpe_inputs(case, seed):
    """Buoyancy anomaly of the first vertical mode and a weak current, [Z, Y, X, field u v b, k, j, i]."""
    g, rng = _Gauss(case["N"]), np.random.default_rng([seed, 4])
    x = _unit(case["nX"], g.x)[None, None, :, None, None, :]
    y = _unit(case["nY"], g.x)[None, :, None, None, :, None]
    z = HDEPTH * (_unit(case["nZ"], g.x)[:, None, None, :, None, None] - 1.0)
    b = _blobs(rng, lambda q: (x - q[0]) ** 2 + (y - q[1]) ** 2, 1, 0.08, 0.12) * 0.01 * np.cos(np.pi * z / HDEPTH)
    e = rng.uniform(0.5e-3, 1.0e-3)
    u = e * np.sin(np.pi * x) ** 2 * np.sin(2 * np.pi * y) + 0.0 * b
    v = e * np.sin(np.pi * y) ** 2 * np.sin(2 * np.pi * x) + 0.0 * b
    nm = max(case["nX"], case["nY"])
    dt = min(2.0e-3, 0.3 / ((case["N"] + 1) ** 2 * nm * 0.18), 0.3 * HDEPTH / ((case["N"] + 1) ** 2 * case["nZ"] * 0.2))
    return np.stack([u, v, b], axis=3), dt


def _cgsem_inputs(case, seed):
    """k = 1 + 0.5 sin sin and a source of 16 sine modes on the unit square, [Y, X, j, i]."""
    nodes, _ = _gll(case["N"])
    rng = np.random.default_rng([seed, 5])
    x, y = _unit(case["nX"], nodes)[None, :, None, :], _unit(case["nY"], nodes)[:, None, :, None]
    k = 1.0 + 0.5 * np.sin(2 * np.pi * x) * np.sin(2 * np.pi * y)
    f = 0.0 * k
    for _ in range(16):
        m, n = rng.integers(1, 9, 2)
        f = f + rng.standard_normal() / (m * m + n * n) * np.sin(m * np.pi * x) * np.sin(n * np.pi * y)
    return k, -f


def _flat(a, lead):
    """[Y, X, ...] (or [Z, Y, X, ...]) to the framework's element-first layout."""
    return np.ascontiguousarray(a.reshape((-1,) + a.shape[lead:]))


# --------------------------------------------------------- prepare, run, work
def prepare(case, seed):
    kind = case["kind"]
    if kind == "sw":
        from self_amd.shallow_water import ShallowWater, SWParams
        sol, h, dt = _sw_inputs(case, seed)
        m = ShallowWater(SWParams(polyDeg=case["N"], nXElem=case["nX"], nYElem=case["nY"], xScale=LSW, yScale=LSW,
                                  g=GRAV, f0=F0, dt=dt, linearDrag=case["drag"]), precision=case["prec"])
        m.SetBathymetry(_flat(np.stack([h, 0 * h, 0 * h], axis=2), 2))
        m.SetSolution(_flat(sol, 2))
        m.CalculateBathymetryGradient()
    elif kind == "adv2d":
        from self_amd.advection import Advection, AdvectionParams
        c, u, v, relax, kappa, dt = _adv2d_inputs(case, seed)
        m = Advection(AdvectionParams(polyDeg=case["N"], nXElem=case["nX"], nYElem=case["nY"], nTracers=case["nq"],
                                      dt=dt, kappa=kappa, warp=case["warp"]))
        m.SetSolution(_flat(c, 2))
        m.SetVelocity(_flat(u + 0 * c[:, :, 0], 2), _flat(v + 0 * c[:, :, 0], 2))
        if relax is not None:
            m.SetRelaxationField(_flat(relax, 2))
            m.SetRelaxationFactor(np.full_like(_flat(c, 2), 2.0))
    elif kind == "adv3d":
        from self_amd.advection3d import Advection3D, Advection3DParams
        c, dt = _adv3d_inputs(case, seed)
        m = Advection3D(Advection3DParams(polyDeg=case["N"], nXElem=case["nX"], nYElem=case["nY"], nZElem=case["nZ"],
                                          nTracers=case["nq"], dt=dt, warp=WARP3, warpSign=SIGN3))
        m.SetSolution(_flat(c, 3))
        m.SetVelocity(*[np.full_like(_flat(c[:, :, :, 0], 3), u) for u in VEL3])
    elif kind == "hpe":
        from self_amd.hydrostatic import HydrostaticParams, HydrostaticPrimitive
        s, dt = _hpe_inputs(case, seed)
        m = HydrostaticPrimitive(HydrostaticParams(polyDeg=case["N"], nXElem=case["nX"], nYElem=case["nY"],
                                                   nZElem=case["nZ"], dt=dt, zScale=HDEPTH))
        sol = np.zeros((m.nElems, 5) + s.shape[4:])
        sol[:, :3] = _flat(s, 3)
        bg = np.zeros_like(sol)
        bg[:, 2] = HBACK
        m.SetSolution(sol)
        m.SetBackgroundState(bg)
    else:
        from self_amd.krylov import CGsemElliptic2D, CGsemParams
        k, s = _cgsem_inputs(case, seed)
        m = CGsemElliptic2D(CGsemParams(polyDeg=case["N"], nXElem=case["nX"], nYElem=case["nY"], tolerance=1.0e-10,
                                        maximumIterates=20000))
        m.SetFluxCoefficient(_flat(k, 2))
        m.SetSource(_flat(s, 2))
        m.SetDirichletBoundaryCondition(0.0 * _flat(k, 2))
        if case["method"] == "pcgmres":
            m.SetPreconditioner(pcIterates=50, pcTolerance=1.0e-4, coefficient="flux")
        return {"kind": kind, "m": m, "case": case, "zero": 0.0 * _flat(k, 2)}
    return {"kind": kind, "m": m, "case": case}


def run(state):
    m, case = state["m"], state["case"]
    if state["kind"] == "cgsem":
        m.SetSolution(state["zero"])
        if case["method"] == "pcgmres":
            m.Solve("pcgmres", "fem", maxIters=40, mInner=30)
        else:
            m.Solve("cgsem_pcg", "jacobi")
        return m.GetSolution()
    if state["kind"] == "hpe":
        m.ForwardStepRK3(case["steps"])
    else:
        m.ForwardStepRK3(0.0, case["steps"])
    return m.GetSolution()


def work(case):
    """Inputs (state, static fields, geometry) read once and the state written once; operations of all steps."""
    N = case["N"]
    n1, nE = N + 1, case["nX"] * case["nY"] * case.get("nZ", 1)
    np2, np3 = n1 * n1, n1 ** 3
    if case["kind"] == "sw":
        read = nE * (np2 * 12 + 12 * n1)  # state, metrics, bathymetry gradient, vorticity; normals
        return {"bytes": 8.0 * (read + 3 * nE * np2),
                "flops": 3.0 * case["steps"] * nE * (np2 * (12 * n1 + 70) + 4 * n1 * (6 * n1 + 50))}
    if case["kind"] == "adv2d":
        nq, r = case["nq"], 2 if case["relax"] else 0
        read = nE * (np2 * (nq * (1 + r) + 7) + 12 * n1)
        return {"bytes": 8.0 * (read + nq * nE * np2),
                "flops": 3.0 * case["steps"] * nE * nq * (np2 * (12 * n1 + 40) + 4 * n1 * (6 * n1 + 30))}
    if case["kind"] == "adv3d":
        nq = case["nq"]
        read = nE * (np3 * (nq + 3 + 10) + 6 * np2 * 4)
        return {"bytes": 8.0 * (read + nq * nE * np3),
                "flops": 3.0 * case["steps"] * nE * nq * (np3 * (12 * n1 + 40) + 6 * np2 * (2 * n1 + 12))}
    if case["kind"] == "hpe":
        read = nE * (np3 * (3 + 1 + 10) + 6 * np2 * 4)
        return {"bytes": 8.0 * (read + 5 * nE * np3),
                "flops": 3.0 * case["steps"] * nE * (np3 * (22 * n1 + 60) + 6 * np2 * (10 * n1 + 20))}
    # what a solve needs is its iteration count (about 40 N max(nX, nY) with Jacobi: 5300 at 128x128, N = 7)
    its = 40 if case["method"] == "pcgmres" else 5.9 * N * max(case["nX"], case["nY"])
    return {"bytes": 8.0 * nE * np2 * 8, "flops": float(its * nE * np2 * (8 * n1 + 25))}


def tolerance(case):
    # about four times the distance to exact(), whose sums run in another order: a few thousand stages in 64 bits; the
    # mixed form's contractions in 32 bits (its gate); elliptic solutions that stop at a relative residual of 1e-10
    if case["kind"] == "sw":
        return {"rel": 1e-6, "max": 4e-5} if case["prec"] == "mixed" else {"rel": 4e-11, "max": 2e-9}
    if case["kind"] == "cgsem":
        return {"rel": 1e-9, "max": 1e-8}
    return {"rel": 2e-12, "max": 1e-10}


# ------------------------------------------------------------------- 64 bits
def exact(case, seed):
    return {"sw": _sw_exact, "adv2d": _adv2d_exact, "adv3d": _adv3d_exact, "hpe": _hpe_exact,
            "cgsem": _cgsem_exact}[case["kind"]](case, seed)


def _sw_exact(case, seed):
    g = _Gauss(case["N"])
    q, h, dt = _sw_inputs(case, seed)
    q, h, Dw, D = _t(q), _t(h), _t(g.Dw), _t(g.D)
    lL, lR, iw = _t(g.l[0]), _t(g.l[1]), _t(1.0 / g.w)
    ax, ay = 2.0 * case["nX"] / LSW, 2.0 * case["nY"] / LSW
    hx, hy = _along(h, D, 3) * ax, _along(h, D, 2) * ay
    drag = case["drag"] / h

    def face(a, b, n):  # flux through a face with normal along n (0: x, 1: y), state a before it and b behind
        cA, cB = torch.sqrt(GRAV * a[2]), torch.sqrt(GRAV * b[2])
        wA, wB = a[n] / a[2], b[n] / b[2]
        fac = torch.maximum(torch.maximum((wA + cA).abs(), (wA - cA).abs()),
                            torch.maximum((wB + cB).abs(), (wB - cB).abs()))
        F = [wA * a[f] + wB * b[f] - fac * (b[f] - a[f]) for f in range(2)] + [a[n] + b[n] - fac * (b[2] - a[2])]
        F[n] = F[n] + 0.5 * GRAV * (a[2] ** 2 + b[2] ** 2)
        return 0.5 * torch.stack(F)

    def tend(q):
        U, V, H = q[:, :, 0], q[:, :, 1], q[:, :, 2]
        pr = 0.5 * GRAV * H * H
        X = torch.stack([U * U / H + pr, U * V / H, U])
        Y = torch.stack([U * V / H, V * V / H + pr, V])
        w, e = torch.movedim(q @ lL, 2, 0), torch.movedim(q @ lR, 2, 0)
        qt = q.transpose(-1, -2)
        s, n = torch.movedim(qt @ lL, 2, 0), torch.movedim(qt @ lR, 2, 0)
        FE = face(e, torch.roll(w, -1, 2), 0)   # [f, Y, X, j]
        FN = face(n, torch.roll(s, -1, 1), 1)   # [f, Y, X, i]
        FW, FS = torch.roll(FE, 1, 2), torch.roll(FN, 1, 1)
        T = -ax * (X @ Dw.T + (FE[..., None] * lR - FW[..., None] * lL) * iw)
        T = T - ay * (_along(Y, Dw, 3) + (FN[..., None, :] * lR[:, None] - FS[..., None, :] * lL[:, None]) * iw[:, None])
        T[0] += F0 * V + GRAV * H * hx - drag * U
        T[1] += -F0 * U + GRAV * H * hy - drag * V
        return torch.movedim(T, 0, 2)

    G = torch.zeros_like(q)
    for _ in range(case["steps"]):
        for a, c in zip(RK_A, RK_G):
            G = a * G + tend(q)
            q = q + (c * dt) * G
    return q.reshape((-1,) + q.shape[2:]).cpu().numpy()


def _adv2d_exact(case, seed):
    g = _Gauss(case["N"])
    c, u, v, relax, kappa, dt = _adv2d_inputs(case, seed)
    c, u, v = _t(c), _t(u + 0 * c[:, :, 0]), _t(v + 0 * c[:, :, 0])
    relax = None if relax is None else _t(relax)
    Dw, lL, lR, iw = _t(g.Dw), _t(g.l[0]), _t(g.l[1]), _t(1.0 / g.w)
    xs, xp, ys, yp = [_t(a)[:, :, None] for a in _geo2(case, g.x, g.x)[2:]]
    J = xs * yp - xp * ys
    one = np.array([1.0])
    ge, gn = _geo2(case, one, g.x), _geo2(case, g.x, one)
    # area-weighted normals of the east face [Y, X, 1, j] and of the north face [Y, X, 1, i]
    nE = [_t(a)[:, :, None, :, 0] for a in (ge[5], -ge[3])]
    nN = [_t(a)[:, :, None, 0, :] for a in (-gn[4], gn[2])]

    def ends(a):
        at = a.transpose(-1, -2)
        return a @ lL, a @ lR, at @ lL, at @ lR

    def div(X, Y, FE, FN):  # weak divergence of contravariant fluxes with face fluxes
        FW, FS = torch.roll(FE, 1, 1), torch.roll(FN, 1, 0)
        return (X @ Dw.T + (FE[..., None] * lR - FW[..., None] * lL) * iw
                + _along(Y, Dw, 3) + (FN[..., None, :] * lR[:, None] - FS[..., None, :] * lL[:, None]) * iw[:, None]) / J

    uE, vE = (u @ lR)[:, :, None], (v @ lR)[:, :, None]
    uN, vN = (u.transpose(-1, -2) @ lR)[:, :, None], (v.transpose(-1, -2) @ lR)[:, :, None]
    wE, wN = uE * nE[0] + vE * nE[1], uN * nN[0] + vN * nN[1]
    u, v = u[:, :, None], v[:, :, None]

    def tend(c):
        w, e, s, n = ends(c)
        cE, cN = torch.roll(w, -1, 1), torch.roll(s, -1, 0)
        mE, mN = 0.5 * (e + cE), 0.5 * (n + cN)
        dx = div(yp * c, -ys * c, mE * nE[0], mN * nN[0])
        dy = div(-xp * c, xs * c, mE * nE[1], mN * nN[1])
        (xw, xe, xsn, xn), (yw, ye, ysn, yn) = ends(dx), ends(dy)
        gE = 0.5 * ((xe + torch.roll(xw, -1, 1)) * nE[0] + (ye + torch.roll(yw, -1, 1)) * nE[1])
        gN = 0.5 * ((xn + torch.roll(xsn, -1, 0)) * nN[0] + (yn + torch.roll(ysn, -1, 0)) * nN[1])
        FE = 0.5 * (wE * (cE + e) - wE.abs() * (cE - e)) - kappa * gE
        FN = 0.5 * (wN * (cN + n) - wN.abs() * (cN - n)) - kappa * gN
        X, Y = c * u - kappa * dx, c * v - kappa * dy
        T = -div(yp * X - xp * Y, -ys * X + xs * Y, FE, FN)
        return T if relax is None else T + (relax - c) * 2.0

    G = torch.zeros_like(c)
    for _ in range(case["steps"]):
        for a, b in zip(RK_A, RK_G):
            G = a * G + tend(c)
            c = c + (b * dt) * G
    return c.reshape((-1,) + c.shape[2:]).cpu().numpy()


def _cofactors(cov):
    """Cofactor rows of the covariant metric: area vectors of the s, p and q faces."""
    def cross(a, b):
        return (a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0])
    t = [[cov[r][k] for r in range(3)] for k in range(3)]
    return cross(t[1], t[2]), cross(t[2], t[0]), cross(t[0], t[1]), t


def _adv3d_exact(case, seed):
    N, g = case["N"], _Gauss(case["N"])
    c, dt = _adv3d_inputs(case, seed)
    c = _t(c)  # [Z, Y, X, f, k, j, i]
    _, cov = _geo3(case, g.x, g.x, g.x)
    rows, t = _cofactors(cov)[:3], _cofactors(cov)[3]
    J = _t(sum(a * b for a, b in zip(rows[0], t[0])))[:, :, :, None]
    a = [_t(sum(u * r for u, r in zip(VEL3, row)))[:, :, :, None] for row in rows]
    one = np.array([1.0])
    wn = []  # normal velocity times area on the east, north and top faces
    for d in range(3):
        pts = [g.x, g.x, g.x]
        pts[d] = one
        row = _cofactors(_geo3(case, *pts)[1])[d]
        wn.append(_t(sum(u * r for u, r in zip(VEL3, row)).squeeze(5 - d))[:, :, :, None])
    Dw, lL, lR, iw = _t(g.Dw), _t(g.l[0]), _t(g.l[1]), _t(1.0 / g.w)
    leg = np.polynomial.legendre.legvander(g.x, N)
    alpha = math.log(2.0) / 9.0  # cut-off mode 3
    nrm = (leg ** 2 * g.w[:, None]).sum(0)
    F1 = _t((leg * np.exp(-alpha * np.arange(N + 1) ** 2) / nrm) @ (leg.T * g.w[None, :]))
    w3 = _t(g.w[:, None, None] * g.w[None, :, None] * g.w[None, None, :])

    def tend(c):
        T = 0.0
        for d in range(3):  # axis of the nodes: 6 - d, axis of the elements: 2 - d
            x = c.movedim(6 - d, -1)
            w, e = x @ lL, x @ lR
            ex = torch.roll(w, -1, 2 - d)
            F = 0.5 * (wn[d] * (ex + e) - wn[d].abs() * (ex - e))
            FW = torch.roll(F, 1, 2 - d)
            x = (a[d] * c).movedim(6 - d, -1) @ Dw.T + (F[..., None] * lR - FW[..., None] * lL) * iw
            T = T - x.movedim(-1, 6 - d)
        return T / J

    E1 = E2 = None
    lim = [None, None, None]
    G = torch.zeros_like(c)
    for _ in range(case["steps"]):
        for st in range(3):
            cf = _along(_along(_along(c, F1, 6), F1, 5), F1, 4)
            e1, e2 = (cf * cf * J * w3).sum((4, 5, 6)), ((c - cf) ** 2 * J * w3).sum((4, 5, 6))
            if E1 is None:
                E1, E2 = torch.zeros_like(e1), torch.zeros_like(e2)
                lim = [torch.zeros_like(e1) for _ in range(3)]
            d1, d2, xi = e1 - E1, e2 - E2, e2 / e1
            E1, E2 = e1, e2
            new = ((d2 > 0) & (d1.abs() / d2 > 1.0)) | (d2 < 0)
            lim[st] = torch.where(new, xi, lim[st - 1] if st > 0 else lim[0])
            c = torch.where((xi > 1.05 * lim[st])[..., None, None, None], cf, c)
            G = RK_A[st] * G + tend(c)
            c = c + (RK_G[st] * dt) * G
    return c.reshape((-1,) + c.shape[3:]).cpu().numpy()


def _hpe_exact(case, seed):
    N, g = case["N"], _Gauss(case["N"])
    s, dt = _hpe_inputs(case, seed)
    u, v, b = [_t(s[:, :, :, f]) for f in range(3)]  # [Z, Y, X, k, j, i]
    Dw, D, lL, lR, iw = _t(g.Dw), _t(g.D), _t(g.l[0]), _t(g.l[1]), _t(1.0 / g.w)
    ax, ay, az = 2.0 * case["nX"], 2.0 * case["nY"], 2.0 * case["nZ"] / HDEPTH

    def integral(x0):  # S[k, m]: integral of the m-th Lagrange polynomial from x0 to node k
        gx, gw = np.polynomial.legendre.leggauss(N + 1)
        return np.stack([0.5 * (x - x0) * (gw @ _lagrange(g.x, 0.5 * (x - x0) * (gx + 1.0) + x0)) for x in g.x])
    Sd, Su = _t(integral(1.0) / az), _t(integral(-1.0) / az)

    def weak(F, dim, lo, hi):  # weak derivative along a node axis, face fluxes lo and hi without that axis
        x = F.movedim(dim, -1) @ Dw.T + (hi[..., None] * lR - lo[..., None] * lL) * iw
        return x.movedim(-1, dim)

    def diagnose(u, v, b):
        div = ax * _along(u, D, 5) + ay * _along(v, D, 4)
        p, w = torch.empty_like(b), torch.empty_like(b)
        base = torch.zeros_like(b[0][:, :, 0])
        for z in reversed(range(case["nZ"])):
            p[z] = base[:, :, None] + _along(b[z], Sd, 2)
            base = p[z].movedim(2, -1) @ lL
        base = torch.zeros_like(base)
        for z in range(case["nZ"]):
            w[z] = base[:, :, None] - _along(div[z], Su, 2)
            base = w[z].movedim(2, -1) @ lR
        return p, w

    def tend(u, v, b):
        p, w = diagnose(u, v, b)
        out = []
        for dim, cell, scale in ((5, 2, ax), (4, 1, ay)):
            x = p.movedim(dim, -1)
            lo, hi = x @ lL, x @ lR
            n = p.shape[cell]
            mid = 0.5 * (hi.narrow(cell, 0, n - 1) + lo.narrow(cell, 1, n - 1))
            FW = torch.cat([lo.narrow(cell, 0, 1), mid], cell)
            FE = torch.cat([mid, hi.narrow(cell, n - 1, 1)], cell)
            out.append(-scale * weak(p, dim, FW, FE))
        bz, wz = b.movedim(3, -1), w.movedim(3, -1)
        bl, bh, wl, wh = bz @ lL, bz @ lR, wz @ lL, wz @ lR
        zero = torch.zeros_like(bl[:1])
        b0, w0 = torch.cat([zero, bh]), torch.cat([wl[:1], wh])   # below each face; the sea floor mirrors w
        b1, w1 = torch.cat([bl, zero]), torch.cat([wl, zero])     # above each face; nothing above the lid
        F = 0.5 * (HBACK * (w0 + w1) - torch.maximum(w0.abs(), w1.abs()) * (b1 - b0))
        out.append(-az * weak(HBACK * w, 3, F[:-1], F[1:]))
        return out, w, p

    G = [torch.zeros_like(b) for _ in range(3)]
    q = [u, v, b]
    for _ in range(case["steps"]):
        for a, c in zip(RK_A, RK_G):
            T, w, p = tend(*q)
            G = [a * x + y for x, y in zip(G, T)]
            q = [x + (c * dt) * y for x, y in zip(q, G)]
    q = torch.stack(q + [w, p], 3)  # w and p as the last stage diagnosed them
    return q.reshape((-1,) + q.shape[3:]).cpu().numpy()


def _cgsem_exact(case, seed):
    N, nX, nY = case["N"], case["nX"], case["nY"]
    nodes, wt = _gll(N)
    k, s = _cgsem_inputs(case, seed)
    D = _t(_derivative(nodes))
    ww = wt[:, None] * wt[None, :]
    hx, hy = 0.5 / nX, 0.5 / nY
    kx, ky = _t(k * ww * hy / hx), _t(k * ww * hx / hy)
    ix = (np.arange(nX)[:, None] * N + np.arange(N + 1)[None, :])[None, :, None, :]
    iy = (np.arange(nY)[:, None] * N + np.arange(N + 1)[None, :])[:, None, :, None]
    cols = nX * N + 1
    idx = torch.as_tensor((iy * cols + ix).reshape(-1), device=_dev())
    inner = torch.zeros((nY * N + 1, cols), dtype=torch.float64, device=_dev())
    inner[1:-1, 1:-1] = 1.0
    inner = inner.reshape(-1)
    shape = (nY, nX, N + 1, N + 1)

    def assemble(l):
        return torch.zeros_like(inner).index_add_(0, idx, l.reshape(-1)) * inner

    def A(x):
        l = x[idx].reshape(shape)
        return assemble((kx * (l @ D.T)) @ D + _along(ky * _along(l, D, 2), D.T, 2))

    D2 = D * D
    diag = assemble(kx @ D2 + _along(ky, D2.T, 2))
    P = torch.where(inner > 0, 1.0 / torch.where(diag > 0, diag, torch.ones_like(diag)), torch.zeros_like(diag))
    rhs = assemble(_t(-s * ww * hx * hy))
    x, r = torch.zeros_like(rhs), rhs.clone()
    z = P * r
    p, rz, stop = z.clone(), r @ z, 1e-13 * float(torch.linalg.norm(rhs))
    for it in range(4 * (nX + nY) * N + 2000):
        Ap = A(p)
        al = rz / (p @ Ap)
        x = x + al * p
        r = r - al * Ap
        z = P * r
        new = r @ z
        p, rz = z + (new / rz) * p, new
        if it % 50 == 49 and float(torch.linalg.norm(r)) < stop:
            break
    return x[idx].reshape((-1,) + shape[2:]).cpu().numpy()
