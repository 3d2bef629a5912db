"""3-D advection, N = 7 FP64 stage on the matrix cores (contractions, face
traces and adaptive filter), and the general stage's row-summed filter
energies, against the oracle where the workgroup layout has edges: one
element, boundary faces of every kind, two tracers, the last workgroup partly
filled (N = 3: two elements a workgroup or more).

Tolerance: a stage sums at most 3 x 8 products per node and 512 energies; with
O(1) data three steps of three stages stay within 9 * (24 + 512) * 2^-53 =
5.4e-13 of the oracle in any summation order, so 1e-12.
"""
import pytest

from test_adv3d_gpu import _cmp, _pair

pytestmark = pytest.mark.gpu

CASES = [
    dict(N=7, n=(1, 1, 1), nq=1, periodic=(True, True, True), warp=0.0),
    dict(N=7, n=(2, 1, 3), nq=2, periodic=(False, True, False), warp=0.03, inflow=True, relax=True),
    dict(N=7, n=(3, 2, 1), nq=1, periodic=(False, False, False), warp=0.02, inflow=True),
    dict(N=7, n=(2, 2, 2), nq=2, periodic=(True, True, True), warp=0.05, filter=False),
    dict(N=3, n=(3, 1, 1), nq=1, periodic=(False, True, True), warp=0.0),
    dict(N=6, n=(1, 2, 1), nq=2, periodic=(True, False, True), warp=0.0, relax=True),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"N{c['N']}-{'x'.join(map(str, c['n']))}-q{c['nq']}")
def test_three_steps_match_the_oracle(gpu_lib, case):
    orc, m = _pair(case)
    for s in range(3):
        orc.forward_step_rk3(0.2 + s * 2e-3)
    m.ForwardStepRK3(0.2, 3)
    _cmp(m.GetSolution(), orc.c, case["nq"], 1e-12)
    m.Trash()
