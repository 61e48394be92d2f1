"""GPU tests of the one-launch PCG iteration at the sizes where its tiles and
chunks begin and end (15 output nodes a tile, 16 cells, chunks of planes), and
where its residual sums cannot be formed by subtraction."""
import numpy as np
import pytest

from conftest import relerr

pytestmark = pytest.mark.gpu

HEAT = [(1, 1), (14, 14), (15, 16), (29, 31), (44, 3), (1, 1, 1), (14, 15, 2), (16, 13, 5),
        (30, 15, 9), (3, 44, 17)]


@pytest.mark.parametrize("nels", HEAT)
def test_heat_tiles(T, gpu, nels):
    from oracle import heat_oracle as H
    sizes = (1.0, 0.7, 1.6)[:len(nels)]
    kw = dict(Tleft=1.0, Tright=None, heatflux={"top": 1.0}, cload={2: 0.5})
    prob = T.HeatConductionProblem(nels, sizes, 1.3, **kw)
    P = H.HeatProblem(nels, sizes, 1.3, **kw)
    s = T.FEASolver(T.HIPMatrixFreeSolver, prob, xmin=0.01, penalty=T.PowerPenaltyFun(3.0),
                    abstol=0.0, reltol=1e-13, cg_max_iter=20000)
    g = np.random.default_rng(sum(nels))
    x = g.uniform(0.2, 1.0, prob.ncells)
    s.set_densities(x)
    K = P.assemble(0.01 + 0.99 * x**3)
    free = ~P.fixed
    v = g.standard_normal(prob.ndofs)
    # every node a sum of at most 27 terms: a few roundings of its largest
    assert relerr(s.matvec(v)[free], K[free][:, free] @ v[free]) < 1e-14
    s()
    Te, _ = P.solve(x, 3.0, 0.01)
    assert s.converged
    # ||r|| <= 1e-13 ||r0|| times the condition numbers here (below 1e4)
    assert relerr(s.u, Te) < 1e-9
    # a warm start from the solution stops at once or stays there
    s(initially_zero=False)
    assert relerr(s.u, Te) < 1e-9


def test_heat_maxiter_and_zero_load(T, gpu):
    prob = T.HeatTree((33, 18))
    s = T.FEASolver(T.HIPMatrixFreeSolver, prob, abstol=0.0, reltol=1e-12)
    for n in (0, 1, 2, 7, 8, 9):  # converges after ny = 18
        s(maxiter=n)
        assert s.last_iters == n and not s.converged
    s(rhs=np.zeros(prob.ndofs))
    assert s.last_iters == 0 and s.converged and not np.any(s.lhs)


# 2D; 3D by planes (at most 256 of them over all columns) and marching chunks
# (the last two), cubes and boxes, tiles of 15 nodes cut at every remainder
ELASTIC = [((1, 2), None), ((14, 14), (1.0, 0.5)), ((15, 16), None), ((61, 30), (1.0, 1.5)),
           ((1, 2, 2), None), ((14, 14, 2), None), ((15, 16, 4), (1.0, 1.5, 0.75)),
           ((29, 14, 8), None), ((17, 46, 44), None), ((31, 44, 22), (1.0, 0.5, 1.25))]


@pytest.mark.parametrize("case", range(len(ELASTIC)))
def test_elastic_tiles(T, O, gpu, case):
    nels, h = ELASTIC[case]
    prob = T.PointLoadCantilever(nels, sizes=h)
    s = T.FEASolver(T.HIPMatrixFreeSolver, prob, penalty=T.PowerPenaltyFun(3.0), abstol=0.0,
                    reltol=1e-12, cg_max_iter=20000)
    orc = O.Oracle(O.Cantilever(tuple(nels)), p=3.0, h=h)
    x = np.random.default_rng(case).uniform(0.5, 1.0, prob.ncells)
    s.vars = x
    orc.set_vars(x)
    s()
    assert s.converged
    free = ~prob.fixed.astype(bool)
    # the true residual of the recursive 1e-12: its drift on 1 : 2 boxes is a few 1e-10
    f = prob.f
    assert np.linalg.norm((f - orc.matvec(s.u))[free]) <= 1e-9 * np.linalg.norm(f)
    u, it = s.u.copy(), s.last_iters
    # the same solve again: the same bits; a warm start from its answer: at once
    s()
    assert s.last_iters == it and np.array_equal(s.u, u)
    s(initially_zero=False, reltol=1.0)
    assert s.last_iters == 0 and np.array_equal(s.u, u)
    for n in (0, 1, 2, 3):
        if n < it:
            s(maxiter=n)
            assert s.last_iters == n and not s.converged


# rows of one to 27 neighbours; node counts at the remainders of 32 (64 in 2D) a workgroup
CSR = [(1, 2), (7, 8), (15, 2), (30, 32), (1, 2, 2), (3, 2, 2), (7, 4, 4), (9, 6, 8), (20, 10, 12)]


@pytest.mark.parametrize("nels", CSR)
@pytest.mark.parametrize("jacobi", [False, True])
def test_assembled_product_and_solve(T, O, gpu, nels, jacobi):
    from topopt_jl_amd._lib import dptr
    prob = T.PointLoadCantilever(nels)
    s = T.FEASolver(T.HIPCGAssemblySolver, prob, xmin=1e-3, penalty=T.PowerPenaltyFun(3.0),
                    cg_max_iter=20000, preconditioner="jacobi" if jacobi else None)
    orc = O.Oracle(O.Cantilever(tuple(nels)), xmin=1e-3, p=3.0)
    g = np.random.default_rng(prob.ncells)
    x = g.uniform(0.5, 1.0, prob.ncells)
    s.vars = x
    orc.set_vars(x)
    Ke, _ = orc.assembled()
    v = g.standard_normal(prob.ndofs)
    s.set_densities(x)
    y = np.empty_like(v)
    assert s.lib.tohip_csr_matvec(s.ctx.ptr, dptr(v), dptr(y)) == 0
    free = ~prob.fixed.astype(bool)
    assert relerr(y[free], (Ke @ v)[free]) < 1e-14  # sums of at most 81 terms
    s(abstol=0.0, reltol=1e-11)
    assert s.converged
    b = np.where(free, prob.f, 0.0)
    assert np.linalg.norm(b - Ke @ s.u) <= 1e-9 * np.linalg.norm(b)
    it = s.last_iters
    for n in (0, 1, 2):
        if n < it:
            s(abstol=0.0, reltol=1e-11, maxiter=n)
            assert s.last_iters == n and not s.converged
