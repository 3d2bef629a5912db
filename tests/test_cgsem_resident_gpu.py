"""The CGSEM CG as one launch per solve against the launched iterations that a
launch whose first unsuccessful poll gives up falls back to: every degree, one,
two and four nodes a thread, ragged last workgroups, curved elements,
prescribed boundary values, no preconditioner, a start at the solution, and
sizes past the device's (which stay with the launches of large problems).

The two sum in one order and are bitwise equal (the bounds of the first two
tests are those of any order: 12 iterations amplify 1e-16 by far less than 1e4
on these well-scaled problems, so 1e-12 relative; solutions to a relative
residual of 1e-11 differ by at most that times the condition number, < 1e4 here
after the diagonal's scaling: 1e-7).  The operator is checked against another
kernel's: the recursion's residual is that of the solution (Residual), up to
the rounding of 12 iterations."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


def _model(N, nX, nY, warp=0.0, boundary=False):
    from self_amd.krylov import CGsemElliptic2D, CGsemParams
    m = CGsemElliptic2D(CGsemParams(polyDeg=N, nXElem=nX, nYElem=nY, warp=warp))
    x, y = m.mesh.x, m.mesh.y
    rng = np.random.default_rng(N + nX)
    m.SetFluxCoefficient(1.0 + 0.5 * np.sin(2 * np.pi * x) * np.sin(2 * np.pi * y))
    m.SetSource(np.cos(3 * x) * (1.0 + y) + 0.1 * rng.standard_normal(x.shape))
    m.SetDirichletBoundaryCondition(np.cos(2 * x + y) if boundary else 0 * x)
    return m


def _solve(m, precond, tol, iters, start=None):
    m.SetSolution(np.zeros_like(m.mesh.x) if start is None else start)
    io, it, _ = m.Solve("cgsem_pcg", precond, tolerance=tol, maxIters=iters)
    return m.GetSolution(), it, io, m.resi.copy()


SHAPES = [(2, 7, 9), (3, 4, 4), (3, 21, 13), (4, 11, 6), (5, 3, 2), (5, 30, 17), (6, 8, 8), (7, 5, 7),
          (7, 63, 57), (8, 9, 5), (9, 6, 6), (10, 4, 5), (11, 5, 3), (7, 80, 61), (3, 150, 131), (5, 122, 101),
          (7, 128, 127), (10, 75, 60), (7, 130, 128), (2, 23, 19)]


def _workgroups(N, nX, nY):  # at one node a thread
    return -(-nX * nY // (1024 // (N + 1) ** 2))


def _counted(m, launches, gaveUp, several):
    n, g = m.ResidentCounts()
    # a problem of one workgroup may find its messages at the first poll
    assert n == launches and (g == gaveUp or not several), (n, g)


@pytest.mark.parametrize("N,nX,nY", SHAPES)
def test_one_launch_follows_the_launched_iterations(gpu_lib, N, nX, nY, monkeypatch):
    m = _model(N, nX, nY, warp=0.03 if nX < 40 else 0.0, boundary=True)
    fits = nX * nY * (N + 1) ** 2 <= 1 << 20
    for k, precond in enumerate(("jacobi", "none")):
        a, ia, _, ra = _solve(m, precond, 1e-300, 12)
        monkeypatch.setenv("SELF_AMD_SPIN_LIMIT", "0")
        b, ib, _, rb = _solve(m, precond, 1e-300, 12)
        monkeypatch.delenv("SELF_AMD_SPIN_LIMIT")
        _counted(m, 2 * k + 2 if fits else 0, k + 1 if fits else 0, _workgroups(N, nX, nY) > 1)
        assert ia == ib == 12
        assert rel_l2(a, b) < 1e-12
        assert np.allclose(ra[:13], rb[:13], rtol=1e-10, atol=0)
        assert abs(np.linalg.norm(m.Residual()) - rb[12]) < 1e-12 * rb[0]
    m.Trash()


@pytest.mark.parametrize("N,nX,nY", [(2, 7, 9), (3, 21, 13), (5, 30, 17), (7, 33, 31), (10, 4, 5)])
def test_solutions_and_stop(gpu_lib, N, nX, nY, monkeypatch):
    m = _model(N, nX, nY, warp=0.03, boundary=True)
    a, ia, ioa, ra = _solve(m, "jacobi", 1e-11, 20000)
    again, ic, _, _ = _solve(m, "jacobi", 1e-11, 20000)
    assert ic == ia and np.array_equal(a, again)  # the same bits every time
    monkeypatch.setenv("SELF_AMD_SPIN_LIMIT", "0")
    b, ib, iob, _ = _solve(m, "jacobi", 1e-11, 20000)
    monkeypatch.delenv("SELF_AMD_SPIN_LIMIT")
    _counted(m, 3, 1, _workgroups(N, nX, nY) > 1)
    assert ioa == iob and abs(ia - ib) <= 2 + ib // 100
    assert ra[ia] / ra[0] < 1e-11 <= ra[ia - 1] / ra[0]
    assert rel_l2(a, b) < 1e-7
    # begun at the solution: few iterations, and the form is still taken
    c, it, _, _ = _solve(m, "jacobi", 1e-3, 100, start=a)
    assert np.isfinite(c).all() and it <= 100
    _counted(m, 4, 1, _workgroups(N, nX, nY) > 1)
    m.Trash()


def test_nothing_to_solve(gpu_lib):
    """A zero source from the zero solution: the loop ends before its first iteration."""
    m = _model(7, 4, 3)
    m.SetSource(0 * m.mesh.x)
    u, it, _, _ = _solve(m, "jacobi", 1e-10, 50)
    assert it == 0 and not u.any()
    m.Trash()


@pytest.mark.parametrize("N,nX,nY", [s for s in SHAPES if s[1] * s[2] * (s[0] + 1) ** 2 <= 1 << 20])
def test_a_solve_that_gave_up_has_the_same_bits(gpu_lib, N, nX, nY, monkeypatch):
    """A result must not depend on what else the device does: the launched
    iterations of a problem of a resident shape sum in the resident order."""
    m = _model(N, nX, nY, warp=0.03 if nX < 40 else 0.0, boundary=True)
    for precond, tol, iters in (("jacobi", 1e-300, 40), ("none", 1e-300, 9), ("jacobi", 0.3, 200)):
        a, ia, ioa, ra = _solve(m, precond, tol, iters)
        monkeypatch.setenv("SELF_AMD_SPIN_LIMIT", "0")
        b, ib, iob, rb = _solve(m, precond, tol, iters)
        monkeypatch.delenv("SELF_AMD_SPIN_LIMIT")
        assert (ia, ioa) == (ib, iob) and np.array_equal(a, b) and np.array_equal(ra, rb)
    m.Trash()


def test_a_batch_that_gave_up_has_the_single_solves_bits(gpu_lib, monkeypatch):
    from self_amd.krylov import SolveBatched
    shapes = [(7, 33, 31), (3, 21, 13), (5, 30, 17), (7, 80, 61), (2, 23, 19)]
    ms = [_model(*s, boundary=True) for s in shapes]
    want = [_solve(m, "jacobi", 1e-9, 5000)[:2] for m in ms]
    for limit in ("2000", "0"):
        monkeypatch.setenv("SELF_AMD_SPIN_LIMIT", limit)
        for m in ms:
            m.SetSolution(np.zeros_like(m.mesh.x))
        _, its, _ = SolveBatched(ms, precond="jacobi", tolerance=1e-9, maxIters=5000)
        for m, i, (u, it) in zip(ms, its, want):
            assert i == it and np.array_equal(m.GetSolution(), u)
    monkeypatch.delenv("SELF_AMD_SPIN_LIMIT")
    assert [m.ResidentCounts()[1] for m in ms] == [1] * len(ms)
    for m in ms:
        m.Trash()
