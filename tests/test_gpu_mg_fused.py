"""GPU: pre-smoothing and restriction in one launch, at the grids where its tiles
(16x8 and 4x4x4 fine nodes) begin and end: the V-cycle against its FP64 oracle at
FP32 tolerance, and solves with the PCG update inside it against the FP64 path."""
import numpy as np
import pytest

from conftest import relerr, rng
from test_gpu_mg import node_major, node_mask

pytestmark = pytest.mark.gpu

GRIDS = [((2, 2), None), ((14, 6), None), ((16, 8), (1.0, 0.5)), ((30, 14), None),
         ((34, 18), None), ((2, 2, 2), None), ((4, 2, 6), None), ((6, 4, 4), (1.0, 2.0, 0.5)),
         ((8, 6, 10), None), ((12, 14, 2), None), ((24, 12, 12), (1.0, 1.5, 0.75))]


@pytest.mark.parametrize("case", range(len(GRIDS)))
def test_vcycle_and_solve(T, O, gpu, case):
    from oracle import mg_oracle
    nels, sizes = GRIDS[case]
    prob = T.PointLoadCantilever(nels, sizes=sizes)
    s = T.FEASolver(T.HIPMatrixFreeSolver, prob, xmin=1e-3, penalty=T.PowerPenaltyFun(3.0),
                    abstol=0.0, reltol=1e-9, cg_max_iter=2000, precision="mixed_mg")
    g = rng(60 + case)
    s.vars = g.uniform(0.1, 1.0, prob.ncells)
    fixed = prob.fixed.astype(bool)
    r = g.standard_normal(prob.ndofs)
    r[fixed] = 0.0
    z = s.mg_apply(r)
    h = list(sizes) if sizes else [1.0] * len(nels)
    md = O.Oracle(O.Cantilever(tuple(nels)), xmin=1e-3, p=3.0, h=tuple(h)).meandiag
    M = mg_oracle.MGOracle(tuple(nels), 1e-3 + (1 - 1e-3) * s.vars**3, node_mask(prob), md, h=h)
    w, _ = s.mg_weights()
    M.omega = [float(v) for v in w]
    idx = node_major(prob)
    assert relerr(z[idx], M.apply(r[idx])) < 1e-5
    assert np.all(z[fixed] == 0.0)
    s()
    assert s.converged
    u = s.u.copy()
    s(precision="fp64")
    assert relerr(u, s.u) < 1e-6
