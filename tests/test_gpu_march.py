"""GPU: the FP32 passes by marching columns on small grids (TOHIP_MARCH_MINCELLS), at
the sizes where their columns (15 and 14 nodes), cells (16) and chunks of planes begin
and end: the V-cycle against its FP64 oracle at FP32 tolerance, the prolongation while
staging against the separate pass, and solves against the FP64 path."""
import numpy as np
import pytest

from conftest import relerr, rng
from test_gpu_mg import node_major, node_mask

pytestmark = pytest.mark.gpu

GRIDS = [((2, 2, 2), None), ((14, 4, 6), None), ((16, 14, 2), (1.0, 1.5, 0.75)),
         ((12, 28, 4), None), ((30, 30, 8), None), ((44, 12, 12), (1.0, 2.0, 0.5)),
         ((28, 16, 20), None)]


def _solver(T, nels, sizes, g, **kw):
    prob = T.PointLoadCantilever(nels, sizes=sizes)
    s = T.FEASolver(T.HIPMatrixFreeSolver, prob, xmin=1e-3, penalty=T.PowerPenaltyFun(3.0),
                    abstol=0.0, reltol=1e-9, cg_max_iter=20000, **kw)
    s.vars = g.uniform(0.1, 1.0, prob.ncells)
    return prob, s


@pytest.mark.parametrize("case", range(len(GRIDS)))
def test_vcycle_and_solves(T, O, gpu, monkeypatch, case):
    from oracle import mg_oracle
    monkeypatch.setenv("TOHIP_MARCH_MINCELLS", "1")
    nels, sizes = GRIDS[case]
    g = rng(80 + case)
    prob, s = _solver(T, nels, sizes, g)
    fixed = prob.fixed.astype(bool)
    r = g.standard_normal(prob.ndofs)
    r[fixed] = 0.0
    z = s.mg_apply(r)
    h = list(sizes) if sizes else [1.0] * 3
    md = O.Oracle(O.Cantilever(tuple(nels)), xmin=1e-3, p=3.0, h=tuple(h)).meandiag
    M = mg_oracle.MGOracle(tuple(nels), 1e-3 + (1 - 1e-3) * s.vars**3, node_mask(prob), md, h=h)
    M.omega = [float(v) for v in s.mg_weights()[0]]
    idx = node_major(prob)
    assert relerr(z[idx], M.apply(r[idx])) < 1e-5
    assert np.all(z[fixed] == 0.0)
    monkeypatch.setenv("TOHIP_ZM_PROL", "0")
    assert np.array_equal(s.mg_apply(r, refresh=False), z)
    monkeypatch.delenv("TOHIP_ZM_PROL")
    s(precision="fp64")
    u = s.u.copy()
    for prec in ("mixed_mg", "mixed"):
        s(precision=prec)
        assert s.converged
        assert relerr(s.u, u) < 1e-6


@pytest.mark.parametrize("nels,sizes", [((120, 88, 14), None), ((200, 124, 16), (1.0, 1.2, 0.9))])
def test_above_the_line(T, gpu, nels, sizes):
    """The rule's own line (2^17 cells), chunks of two and of more planes."""
    g = rng(90)
    prob, s = _solver(T, nels, sizes, g, precision="mixed_mg")
    s()
    assert s.converged
    u = s.u.copy()
    s(precision="fp64")
    assert relerr(u, s.u) < 1e-6
