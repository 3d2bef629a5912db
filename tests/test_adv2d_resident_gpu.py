"""Several advection-diffusion RK3 steps in one launch against the launches of
a model too large for it: the same expressions in the same order, so bitwise
equal.  The launched steps come from the fallback of a launch whose first
unsuccessful poll gives up.  Every degree and tracer count, walls, inflow
(time-dependent), warp and relaxation, several launches in flight."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _model(N, nX, nY, nq, periodic=True, warp=0.0, relax=False, inflow=False, dt=2e-5):
    from self_amd.advection import Advection, AdvectionParams
    p = AdvectionParams(polyDeg=N, nXElem=nX, nYElem=nY, nTracers=nq, dt=dt, kappa=2e-3, warp=warp,
                        periodicX=periodic, periodicY=periodic)
    edges = None
    if inflow:
        edges = Advection(p).mesh.edges.copy()
        wall = np.flatnonzero(edges[:, 2] < 0)
        edges[wall[::2], 2] = -103
        edges[wall[1::3], 2] = -104
    m = Advection(p, edges=edges)
    x, y = m.mesh.x, m.mesh.y
    c = np.stack([np.exp(-((x - 0.4) ** 2 + (y - 0.5 - 0.1 * f) ** 2) / 0.03) for f in range(nq)], axis=1)
    m.SetSolution(c)
    m.SetVelocity(1.0 + 0.3 * np.sin(2 * np.pi * y), 0.5 - 0.2 * np.cos(2 * np.pi * x))
    if relax:
        m.SetRelaxationField(0.3 + 0 * c)
        m.SetRelaxationFactor(5.0 + 0 * c)
    return m


CASES = [dict(N=N, nX=5 + N % 3, nY=4, nq=1 + N % 4) for N in range(1, 9)] + [
    dict(N=7, nX=10, nY=10, nq=1, warp=0.03),
    dict(N=7, nX=6, nY=7, nq=2, periodic=False, relax=True),
    dict(N=3, nX=13, nY=9, nq=4, periodic=False, inflow=True),
    dict(N=4, nX=31, nY=17, nq=3, relax=True, warp=0.02),
    dict(N=2, nX=9, nY=11, nq=2, periodic=False, inflow=True),
    dict(N=5, nX=60, nY=50, nq=1),
    dict(N=1, nX=13, nY=12, nq=3, warp=0.02),
    dict(N=2, nX=12, nY=9, nq=4, relax=True),
]


def _workgroups(case):
    return -(-case["nX"] * case["nY"] // (256 // (case["N"] + 1) ** 2))


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(v) for v in c.values()))
def test_resident_steps_equal_launches(gpu_lib, case, monkeypatch):
    a, b = _model(**case), _model(**case)
    t = 0.25
    for n in (1, 5, 2):  # in flight together
        a.ForwardStepRK3(t, n)
        t += n * 2e-5
    got = a.GetSolution()
    monkeypatch.setenv("SELF_AMD_SPIN_LIMIT", "0")
    t = 0.25
    for n in (1, 5, 2):
        b.ForwardStepRK3(t, n)
        t += n * 2e-5
    want = b.GetSolution()
    monkeypatch.delenv("SELF_AMD_SPIN_LIMIT")
    assert np.isfinite(want).all() and not np.array_equal(want, _model(**case).GetSolution())
    assert np.array_equal(got, want)
    # a model of one workgroup may find its messages at the first poll
    assert a.ResidentCounts() == (3, 0)
    if _workgroups(case) > 1:
        assert b.ResidentCounts() == (3, 1)
    b.ForwardStepRK3(t, 3)  # the form is taken up again
    a.ForwardStepRK3(t, 3)
    assert np.array_equal(a.GetSolution(), b.GetSolution())
    assert b.ResidentCounts() == (4, 1 if _workgroups(case) > 1 else b.ResidentCounts()[1])
    a.GlobalTimeDerivative(t)
    b.GlobalTimeDerivative(t)
    assert np.array_equal(a.GetTendency(), b.GetTendency())
    a.Trash()
    b.Trash()


@pytest.mark.parametrize("case", [CASES[14], CASES[2], CASES[8], CASES[10], CASES[11]],
                         ids=lambda c: "-".join(str(v) for v in c.values()))
def test_gradient_after_steps(gpu_lib, case, monkeypatch):
    """GetGradient after ForwardStepRK3 is the last stage's, as the launched
    stages leave it: not that of an earlier time derivative."""
    a, b = _model(**case), _model(**case)
    monkeypatch.setenv("SELF_AMD_SPIN_LIMIT", "0")
    for n in (1, 4):
        b.ForwardStepRK3(0.1, n)
        b.Synchronize()
    want = b.GetGradient()
    monkeypatch.delenv("SELF_AMD_SPIN_LIMIT")
    assert _workgroups(case) == 1 or b.ResidentCounts() == (2, 2)
    a.GlobalTimeDerivative(0.1)
    before = a.GetGradient()
    for n in (1, 4):
        a.ForwardStepRK3(0.1, n)
    assert a.ResidentCounts() == (2, 0)
    for g, w, o in zip(a.GetGradient(), want, before):
        assert np.isfinite(w).all() and np.array_equal(g, w) and not np.array_equal(g, o)
    a.Trash()
    b.Trash()


def test_tags_come_round_after_a_launch_gave_up(gpu_lib, monkeypatch):
    """65536 steps are a multiple of the 65536 stages after which a message's
    tag is the same again: the first messages of a launch that gave up must not
    be taken for those of the launch after it.  More steps than one launch takes
    too, with an inflow that depends on the time."""
    case = dict(N=2, nX=9, nY=11, nq=1, periodic=False, inflow=True, dt=1e-8)
    a, b = _model(**case), _model(**case)
    b.ForwardStepRK3(0.2, 65536 + 3)
    b.ForwardStepRK3(0.3, 2)
    monkeypatch.setenv("SELF_AMD_SPIN_LIMIT", "0")
    a.ForwardStepRK3(0.2, 65536 + 3)
    a.Synchronize()
    monkeypatch.delenv("SELF_AMD_SPIN_LIMIT")
    assert a.ResidentCounts() == (2, 1)  # the second returned at once
    a.ForwardStepRK3(0.3, 2)
    want = b.GetSolution()
    assert np.isfinite(want).all() and np.array_equal(a.GetSolution(), want)
    a.Trash()
    b.Trash()
