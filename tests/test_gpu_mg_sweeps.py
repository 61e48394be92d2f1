"""GPU: the matrix of a coarsest multigrid level of sweeps against the sweeps it
stands for, at level sizes around its limits (one and two nodes or cells a
thread, prescribed columns, 2D and 3D, cubes and boxes)."""
import numpy as np
import pytest

from conftest import relerr, rng

pytestmark = pytest.mark.gpu

# fine grid, cell sizes; coarsest: 21x7x7 (1408 nodes), 13x9x5 (840 nodes, 585
# cells), 25x7x7 box cells (1664 nodes, 1225 cells), 2D 39x29 (1131 cells), 31x13
CASES = [((42, 14, 14), None), ((26, 18, 10), None), ((50, 14, 14), (1.0, 1.5, 0.75)),
         ((78, 58), None), ((62, 26), (1.0, 0.5))]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_sweeps_as_matrix(T, gpu, monkeypatch, case):
    monkeypatch.setenv("TOHIP_MG_WADAPT", "0")  # the same smoother in both
    nels, sizes = CASES[case]
    prob = T.PointLoadCantilever(nels, sizes=sizes)
    s = T.FEASolver(T.HIPMatrixFreeSolver, prob, penalty=T.PowerPenaltyFun(3.0), abstol=0.0,
                    reltol=1e-9, cg_max_iter=2000, precision="mixed_mg")
    g = rng(40 + case)
    fixed = prob.fixed.astype(bool)
    for _ in range(2):  # a second design: the matrix follows the operator
        s.vars = g.uniform(0.1, 1.0, prob.ncells)
        r = g.standard_normal(prob.ndofs)
        r[fixed] = 0.0
        z = s.mg_apply(r)  # the sweeps
        assert np.all(z[fixed] == 0.0)
        # one iteration from zero on the load r: u = alpha M r, by the matrix
        s(rhs=r, precision="fp64_mg", maxiter=1, reltol=1e-30)
        # 30 FP32 sweeps against a row sum of FP32 products: the V-cycle's bound
        assert relerr(s.u / np.linalg.norm(s.u), z / np.linalg.norm(z)) < 1e-5
        s()
        assert s.converged
        # the solves' matrix does not show in one application
        assert np.array_equal(s.mg_apply(r, refresh=False), z)
        u, it = s.u.copy(), s.last_iters
        s(precision="fp64")
        assert relerr(u, s.u) < 1e-6
        s()
        assert s.last_iters == it and np.array_equal(s.u, u)
