"""Hydrostatic primitive equations, N = 7 on the matrix cores, against the
oracle where the column loop and the face branches have edges: one layer (the
loop's first iteration is its last), one column, walls on every side above the
sea floor, a warped mesh, pressure given instead of diagnosed.

Tolerance: as the oracle comparison of the other orders, 1e-12 for one time
derivative (sums of at most 8 layers x 8 products, 64 * 2^-53 = 7e-15 relative
to the largest term, and the cancellation of the column sums), 1e-11 after
steps.
"""
import numpy as np
import pytest

from conftest import rel_l2
from test_hpe_gpu import _pair

pytestmark = pytest.mark.gpu

CASES = [
    dict(N=7, n=(1, 1, 1), periodic=(True, True), warp=0.0, dp=True),
    dict(N=7, n=(2, 1, 1), periodic=(False, False), warp=0.02, dp=True),
    dict(N=7, n=(1, 2, 5), periodic=(True, False), warp=0.03, dp=False),
    dict(N=7, n=(2, 2, 4), periodic=(False, True), warp=0.0, dp=True),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c["n"])) + ("" if c["dp"] else "-noP"))
def test_derivative_and_steps_match_the_oracle(gpu_lib, case):
    orc, gpu = _pair(case, dt=2e-3)
    orc.call("global_time_derivative")
    gpu.GlobalTimeDerivative()
    assert rel_l2(gpu.GetDivU().ravel(), orc.divU) < 1e-12
    so, sg = orc.view(orc.sol, 5), gpu.GetSolution()
    for f in (3, 4):
        assert rel_l2(sg[:, f], so[:, f]) < 1e-12, f
    to, tg = orc.view(orc.tend, 3), gpu.GetTendency()
    for f in range(3):
        assert rel_l2(tg[:, f], to[:, f]) < 1e-12, f
    for _ in range(3):
        orc.call("forward_step_rk3")
    gpu.ForwardStepRK3(3)
    orc.G[:] = 0.0
    gpu.SetPreviousTendency(np.zeros((orc.nElems, 3) + so.shape[2:]))
    for _ in range(2):
        orc.call("forward_step_ab2")
    gpu.ForwardStepAB2(2)
    so, sg = orc.view(orc.sol, 5), gpu.GetSolution()
    for f in range(3):
        assert rel_l2(sg[:, f], so[:, f]) < 1e-11, f


@pytest.mark.parametrize("N", [4, 7])
def test_kernel_times_are_of_the_kernels_a_step_runs(gpu_lib, N):
    """KernelTimes advances the model as that many steps do, bit for bit: it
    times the same kernels."""
    case = dict(N=N, n=(2, 2, 3), periodic=(False, True), warp=0.02, dp=True)
    _, a = _pair(case, dt=2e-3)
    _, b = _pair(case, dt=2e-3)
    a.ForwardStepRK3(3)
    assert min(b.KernelTimes(3)) > 0.0
    assert np.array_equal(a.GetSolution(), b.GetSolution())
