"""The FEM preconditioner's iterations as a graph: replays give the bits of a
fresh solver's first application, on other right-hand sides too, with solves
(another state ends those) in FP64 and FP32 between them, and after the
preconditioner is built again with other settings.  Sizes: less than one
workgroup of rows, just under and over one workgroup, more rows than the grid's
threads (the strided loop), and no iteration at all, which returns the
right-hand side.  The values themselves are compared with the oracle's.

Tolerance: as the oracle comparison of a fixed short CG sequence, 1e-12.
"""
import numpy as np
import pytest

from conftest import rel_l2
from oracle import pyoracle as po
from test_cgsem_pc_gpu import _model

pytestmark = pytest.mark.gpu


def _rhs(o, g, N, seed):
    b = o.unmask(o.mask(np.random.default_rng(seed).standard_normal(o.solution.size)))
    return b, b.reshape(g.nElems, N + 1, N + 1)


# interior nodes: 9, 255, 273, 131769 (more than 512 workgroups of 256), 88
@pytest.mark.parametrize("N,nX,nY,its", [(2, 2, 2, 4), (2, 8, 9, 3), (2, 11, 7, 3), (4, 91, 91, 2), (3, 4, 3, 0)])
def test_replays_equal_a_fresh_application_and_the_oracle(gpu_lib, N, nX, nY, its):
    g, h = _model(N, nX, nY), _model(N, nX, nY)
    o = po.CGSEM2D(N, nX, nY, tolerance=1e-10, maxIters=10)
    for m in (g, h):
        m.SetPreconditioner(pcIterates=its, pcTolerance=1e-30)
    o.build_preconditioner(g.mesh.x.ravel(), g.mesh.y.ravel(), pcTolerance=1e-30, pcIterates=its)
    zero = np.zeros((g.nElems, N + 1, N + 1))
    bo, b = _rhs(o, g, N, 1)
    g.SetSource(b)
    g.SetDirichletBoundaryCondition(zero)
    first, n = g.ApplyPreconditioner(b)
    assert n == its
    assert rel_l2(first.ravel(), o.precondition(bo)[0] if its else bo) < 1e-12
    for rep in range(3):
        if its:
            g.SetSolution(zero)
            g.Solve("pcgmres", "fem", maxIters=1, mInner=3)
            g.SetSolution(zero)
            g.SolveGMRESMixed(maxCycles=1, mInner=3)
        b2 = _rhs(o, g, N, 5 + rep)[1]
        assert np.array_equal(g.ApplyPreconditioner(b2)[0], h.ApplyPreconditioner(b2)[0])
        assert np.array_equal(g.ApplyPreconditioner(b)[0], first)
    for m in (g, h):
        m.SetPreconditioner(pcIterates=its + 2, pcTolerance=1e-30)
    x, n = g.ApplyPreconditioner(b)
    assert n == its + 2 and np.array_equal(x, h.ApplyPreconditioner(b)[0])
    g.Trash()
    h.Trash()


def test_iterations_past_the_graph_s_bound(gpu_lib):
    """8192 iterations are a graph, 8193 launches: the same bits, early end and all."""
    g, h = _model(3, 9, 8), _model(3, 9, 8)
    g.SetPreconditioner(pcIterates=8192, pcTolerance=0.2)
    h.SetPreconditioner(pcIterates=8193, pcTolerance=0.2)
    b = np.sin(5 * g.mesh.x) * (1 + g.mesh.y)
    for _ in range(3):
        (x, n), (y, m) = g.ApplyPreconditioner(b), h.ApplyPreconditioner(b)
        assert 0 < n == m < 400 and np.array_equal(x, y)
    g.Trash()
    h.Trash()
