"""Several RK3 steps in one launch, its workgroups waiting for each other's
traces, against one launch per stage: the same expressions in the same order,
so the states are bitwise equal.  Degrees on and off the matrix-core path,
meshes of one and of many workgroups with a ragged last one, walls, warp, drag,
relaxation, the examples' class and ensembles.  A launch whose first
unsuccessful poll gives up must leave the state to the ordinary launches."""
import numpy as np
import pytest

from sw2d_cases import smooth_state

pytestmark = pytest.mark.gpu


def _model(N, nX, nY, precision, members=1, periodic=True, warp=0.0, drag=0.0, relax=False, variant=0):
    from self_amd.shallow_water import ShallowWater, SWParams
    dt = 2e-4 * min(1.0, 5.0 / max(nX, nY))
    p = SWParams(polyDeg=N, nXElem=nX, nYElem=nY, xScale=2.0, yScale=3.0, dt=dt, linearDrag=drag,
                 periodicX=periodic, periodicY=periodic, warp=warp)
    m = ShallowWater(p, precision=precision, mixedGuard=0)
    x, y = m.mesh.x, m.mesh.y
    U, V, H, h, f = smooth_state(x, y, 2.0, 3.0)
    sol = np.stack([U, V, H], axis=1)
    m.SetVariant(variant)
    m.SetBathymetry(np.stack([h, 0 * h, 0 * h], axis=1))
    m.SetPlanetaryVorticity(f)
    m.CalculateBathymetryGradient()
    if relax:
        m.SetRelaxationField(np.stack([0 * U, 0 * V, h, 0.5 + 0 * h], axis=1))
    if members > 1:
        m.SetMembers(members)
        for k in range(members):
            m.SetMemberSolution(k, sol * (1.0 + 1e-3 * k))
            m.SetMemberTimeStep(k, dt * (1.0 - 0.1 * k))
    else:
        m.SetSolution(sol)
    return m


def _states(m, members):
    return [m.GetMemberSolution(k) for k in range(members)] if members > 1 else [m.GetSolution()]


CASES = [
    dict(N=7, nX=3, nY=3, precision="fp64"),
    dict(N=7, nX=13, nY=5, precision="fp64", periodic=False, warp=0.03, drag=0.1),
    dict(N=7, nX=9, nY=7, precision="mixed", relax=True),
    dict(N=7, nX=5, nY=4, precision="mixed", members=3),
    dict(N=3, nX=5, nY=7, precision="fp64", warp=0.03),
    dict(N=3, nX=11, nY=9, precision="mixed", periodic=False, members=2),
    dict(N=1, nX=9, nY=8, precision="fp64"),
    dict(N=2, nX=7, nY=5, precision="mixed", periodic=False),
    dict(N=4, nX=6, nY=5, precision="fp64", variant=1),
    dict(N=5, nX=8, nY=3, precision="fp64", members=2, relax=True),
    dict(N=6, nX=4, nY=4, precision="mixed", warp=0.02),
    dict(N=8, nX=7, nY=3, precision="fp64", periodic=False),
    dict(N=10, nX=5, nY=3, precision="fp64", drag=0.2),
    dict(N=11, nX=3, nY=4, precision="mixed"),
    dict(N=7, nX=64, nY=64, precision="fp64"),   # every workgroup the device holds
    dict(N=7, nX=65, nY=64, precision="fp64"),   # one too many: not this form
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(v) for v in c.values()))
def test_resident_steps_equal_stage_launches(gpu_lib, case):
    members = case.get("members", 1)
    a, b = _model(**case), _model(**case)
    b.SetGraph(False)
    for n in (2, 5, 1, 4):
        b.ForwardStepRK3(0.0, n)
    want = _states(b, members)
    for n in (2, 5):  # two launches in flight
        a.ForwardStepRK3(0.0, n)
    a.ForwardStepRK3(0.0, 1)
    a.ForwardStepRK3(0.0, 4)
    got = _states(a, members)
    assert all(np.isfinite(w).all() for w in want)
    for g, w in zip(got, want):
        assert np.array_equal(g, w)
    assert b.ResidentCounts() == (0, 0)
    assert a.ResidentCounts() == ((0, 0) if case["nX"] == 65 else (3, 0))  # every call of two steps or more
    a.Trash()
    b.Trash()


@pytest.mark.parametrize("case", [CASES[1], CASES[5], CASES[9]], ids=["N7", "N3-ensemble", "N5-ensemble"])
def test_steps_run_again_where_a_launch_gives_up(gpu_lib, case, monkeypatch):
    members = case.get("members", 1)
    a, b = _model(**case), _model(**case)
    b.SetGraph(False)
    for n in (3, 4, 2):
        b.ForwardStepRK3(0.0, n)
    a.ForwardStepRK3(0.0, 3)
    monkeypatch.setenv("SELF_AMD_SPIN_LIMIT", "0")
    a.ForwardStepRK3(0.0, 4)
    monkeypatch.delenv("SELF_AMD_SPIN_LIMIT")
    a.ForwardStepRK3(0.0, 2)  # returns at once behind the one that gave up
    for g, w in zip(_states(a, members), _states(b, members)):
        assert np.array_equal(g, w)
    assert a.ResidentCounts() == (3, 1)
    a.ForwardStepRK3(0.0, 6)  # and the form is taken up again
    b.ForwardStepRK3(0.0, 6)
    for g, w in zip(_states(a, members), _states(b, members)):
        assert np.array_equal(g, w)
    assert a.ResidentCounts() == (4, 1)
    a.Trash()
    b.Trash()


def test_the_form_rests_after_four_launches_in_a_row_gave_up(gpu_lib, monkeypatch):
    case = CASES[4]
    a, b = _model(**case), _model(**case)
    b.SetGraph(False)

    def step(n):
        for _ in range(n):
            a.ForwardStepRK3(0.0, 2)
            b.ForwardStepRK3(0.0, 2)

    monkeypatch.setenv("SELF_AMD_SPIN_LIMIT", "0")
    for k in range(3):
        step(1)
        assert a.ResidentCounts() == (k + 1, k + 1)
    monkeypatch.delenv("SELF_AMD_SPIN_LIMIT")
    step(1)  # one that finishes: the count begins again
    assert a.ResidentCounts() == (4, 3)
    monkeypatch.setenv("SELF_AMD_SPIN_LIMIT", "0")
    for k in range(4):
        step(1)
        assert a.ResidentCounts() == (k + 5, k + 4)
    monkeypatch.delenv("SELF_AMD_SPIN_LIMIT")
    step(256)
    assert a.ResidentCounts() == (8, 7)
    step(1)
    assert a.ResidentCounts() == (9, 7)
    assert np.array_equal(a.GetSolution(), b.GetSolution())
    a.Trash()
    b.Trash()


def test_models_in_flight_together_equal_alone(gpu_lib):
    """Four models of one thread, each on its own stream, their launches in
    flight together (two of them fill the device)."""
    cases = [CASES[14], CASES[1], dict(CASES[14], precision="mixed"), CASES[4]]
    ms = [_model(**c) for c in cases]
    for _ in range(3):
        for m in ms:
            m.ForwardStepRK3(0.0, 4)
    got = [m.GetSolution() for m in ms]
    for c, m, g in zip(cases, ms, got):
        m.Trash()
        w = _model(**c)
        w.SetGraph(False)
        for _ in range(3):
            w.ForwardStepRK3(0.0, 4)
        assert np.array_equal(g, w.GetSolution())
        w.Trash()


def test_tags_come_round_after_a_launch_gave_up(gpu_lib, monkeypatch):
    """65536 steps are a multiple of the 65536 stages after which a message's
    tag is the same again: the first messages of a launch that gave up must not
    be taken for those of the launch after it."""
    case = dict(N=3, nX=5, nY=7, precision="fp64", warp=0.03)
    a, b = _model(**case), _model(**case)
    for m in (a, b):
        gpu_lib.check(gpu_lib.lib().self_sw2d_set_params(m._h, 1.0, 1e-7, 0.0))
    b.ForwardStepRK3(0.0, 65536)
    b.ForwardStepRK3(0.0, 2)
    monkeypatch.setenv("SELF_AMD_SPIN_LIMIT", "0")
    a.ForwardStepRK3(0.0, 65536)
    a.Synchronize()
    monkeypatch.delenv("SELF_AMD_SPIN_LIMIT")
    assert a.ResidentCounts() == (1, 1)
    a.ForwardStepRK3(0.0, 2)
    want = b.GetSolution()
    assert np.isfinite(want).all() and np.array_equal(a.GetSolution(), want)
    a.Trash()
    b.Trash()


def test_tuning_keeps_resident_and_launched_models_apart(gpu_lib, tmp_path):
    """64x64 elements at N = 7 fit the device, 65x64 of the same size class do
    not: neither takes the other's choice, nor one written before there were
    resident steps."""
    from self_amd import shallow_water as SW
    SW.clear_tuning_table()
    big, fit = _model(N=7, nX=65, nY=64, precision="fp64"), _model(N=7, nX=64, nY=64, precision="fp64")
    big.Autotune(4)
    assert [t["kind"] for t in SW.tuning_table()] == ["sw2d_launched"]
    fit.Autotune(4)
    assert sorted(t["kind"] for t in SW.tuning_table()) == ["sw2d", "sw2d_launched"]
    n = fit.ResidentCounts()[0]
    assert n >= 2  # a trial's
    fit.Autotune(4)  # from the table
    assert fit.ResidentCounts() == (n, 0)
    path = tmp_path / "t.txt"
    path.write_text("sw2d 2 7 0 12 2 0 0 0 0.05\n")
    SW.load_tuning_table(str(path))
    fit.Autotune(4)
    assert fit.ResidentCounts()[0] > n
    kept = {t["kind"]: t["config"] for t in SW.tuning_table()}
    assert kept["sw2d"][:3] == [1, 1, 1]
    SW.clear_tuning_table()
    big.Trash()
    fit.Trash()
