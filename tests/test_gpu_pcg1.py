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


# More work than workgroups at once (768 in 2D and for heat, 512 in 3D): two columns of
# tiles, the second one node wide, and a long ragged side
STRIDED = [((15, 8000), None), ((15, 5800), (1.0, 1.5)), ((15, 3880, 2), None),
           ((15, 4100, 2), (1.0, 1.5, 0.75))]


@pytest.mark.parametrize("case", range(len(STRIDED)))
def test_strided_elastic(T, O, gpu, case):
    """The iterates after 0 .. 9 iterations against the oracle's.  The load on the
    prescribed DOFs goes in the first one, which leaves r.z a millionth of what it was:
    the launch that applies the update alone."""
    from topopt_jl_amd._lib import dptr
    import ctypes as C
    nels, h = STRIDED[case]
    prob = T.PointLoadCantilever(nels, sizes=h)
    s = T.FEASolver(T.HIPMatrixFreeSolver, prob, penalty=T.PowerPenaltyFun(3.0))
    orc = O.Oracle(O.Cantilever(tuple(nels)), p=3.0, h=h)
    g = np.random.default_rng(case)
    x = g.uniform(0.5, 1.0, prob.ncells)
    s.set_densities(x)
    orc.set_vars(x)
    fixed = prob.fixed.astype(bool)
    b = np.where(fixed, 1e3, 1e-3) * g.standard_normal(prob.ndofs)
    z = orc.jacobi_diag() ** -1 * b
    z1 = b - (b @ z) / (z @ orc.matvec(z)) * orc.matvec(z)
    assert z1 @ (z1 / orc.jacobi_diag()) < 5e-4 * (b @ z)  # due below 1e-3
    for n in (0, 1, 2, 9):
        u, again = np.zeros(prob.ndofs), np.zeros(prob.ndofs)
        it, res = C.c_int64(), C.c_double()
        for v in (u, again):
            assert s.lib.tohip_solve(s.ctx.ptr, dptr(b), dptr(v), 0.0, 1e-30, n, 1, 0,
                                     C.byref(it), C.byref(res)) == 1  # not converged
        assert it.value == n and np.array_equal(u, again)
        ue, ite, rese = orc.pcg(b, reltol=1e-30, maxiter=n)
        assert ite == n
        # 1e-16 over the part of the residual that the first iteration leaves
        assert relerr(u, ue) < 1e-9 and abs(res.value - rese) < 1e-9 * np.linalg.norm(b)


@pytest.mark.parametrize("nels", [(15, 8000), (421, 420), (15, 5791, 2)])
def test_strided_heat(T, gpu, nels):
    """As above: the guess at the prescribed nodes goes in the first iteration."""
    import ctypes as C
    import scipy.sparse as sp
    from oracle import heat_oracle as H
    from topopt_jl_amd._lib import dptr
    sizes = (1.0, 0.7, 1.6)[:len(nels)]
    prob = T.HeatConductionProblem(nels, sizes, 1.3, Tleft=0.0, Tright=None)
    s = T.FEASolver(T.HIPMatrixFreeSolver, prob, xmin=0.01, penalty=T.PowerPenaltyFun(3.0))
    g = np.random.default_rng(sum(nels))
    x = g.uniform(0.3, 1.0, prob.ncells)
    s.set_densities(x)
    dofs = (np.asarray(prob.cell_dofs).T - 1).astype(np.int64)
    Ke, rho, nc = H.heat_ke(len(nels), sizes, 1.3), 0.01 + 0.99 * x**3, dofs.shape[1]
    K = sp.csr_matrix(((rho[:, None, None] * Ke).ravel(),
                       (np.repeat(dofs, nc, axis=1).ravel(), np.tile(dofs, (1, nc)).ravel())))
    fixed = prob.fixed.astype(bool)
    md = np.trace(Ke) * prob.ncells
    diag = np.where(fixed, md, K.diagonal())
    A = lambda v: np.where(fixed, md * v, K @ np.where(fixed, 0.0, v))
    v = g.standard_normal(prob.ndofs)
    assert relerr(s.matvec(v), A(v)) < 1e-14
    b = np.where(fixed, 0.0, g.standard_normal(prob.ndofs))
    u0 = np.where(fixed, 1.0, 0.0)
    u, p, rho_prev = u0.copy(), 0.0, 1.0
    r = b - A(u)
    for n in range(10):
        if n in (0, 1, 2, 9):
            t, it, res = u0.copy(), C.c_int64(), C.c_double()
            assert s.lib.tohip_heat_solve(s.ptr, dptr(b), dptr(t), 0.0, 1e-30, n, 0, 0,
                                          C.byref(it), C.byref(res)) == 1
            assert it.value == n and relerr(t, u) < 1e-9
            assert abs(res.value - np.linalg.norm(r)) < 1e-9 * np.linalg.norm(A(u0))
        z = r / diag
        rz = r @ z
        if n == 1:
            assert rz < 5e-4 * rho_prev  # an update alone is due below 1e-3
        p = z + rz / rho_prev * p
        q = A(p)
        a = rz / (p @ q)
        u, r, rho_prev = u + a * p, r - a * q, rz


def test_iteration_time_grows_with_the_grid(T, gpu):
    """FP64 elasticity and heat: 1000x990 against 640x320 cells, 4.8 times the nodes.
    Every workgroup sums every workgroup's partials, so that an iteration of one
    workgroup a tile took 7.5 and 8 times as long."""
    import time
    from topopt_jl_amd import _lib
    import ctypes as C

    def per_iteration(run):
        best = []
        for n in (64, 320):
            run(n)
            t = []
            for _ in range(5):
                t0 = time.perf_counter()
                run(n)
                t.append(time.perf_counter() - t0)
            best.append(min(t))
        return best[1] - best[0]

    el, he = [], []
    for nels in ((640, 320), (1000, 990)):
        nn = (nels[0] + 1) * (nels[1] + 1)
        fixed = np.repeat(np.arange(nn) % (nels[0] + 1) == 0, 2).astype(np.uint8)
        c = _lib.Context(2, nels, np.ones(2), 1.0, 0.3, 1e-3, 3.0, True, None, fixed)
        g = np.random.default_rng(nn)
        assert c.lib.tohip_set_densities(c.ptr, _lib.dptr(g.uniform(0.3, 1, c.ncells))) == 0
        assert c.lib.tohip_set_load(c.ptr, _lib.dptr(g.standard_normal(c.ndofs))) == 0
        it, res = C.c_int64(), C.c_double()
        el.append(per_iteration(lambda n: c.lib.tohip_solve(
            c.ptr, None, None, 0.0, 1e-30, n, 1, 0, C.byref(it), C.byref(res))))
        prob = T.HeatConductionProblem(nels, (1.0, 1.0), 1.0, Tleft=1.0)
        s = T.FEASolver(T.HIPMatrixFreeSolver, prob, abstol=0.0, reltol=1e-30)
        b = g.standard_normal(prob.ndofs)
        he.append(per_iteration(lambda n: s(rhs=b, maxiter=n)))
    assert el[1] < 4.8 * el[0], (el[0] / 256, el[1] / 256)
    assert he[1] < 4.8 * he[0], (he[0] / 256, he[1] / 256)


def test_heat_rows_past_32_bit_offsets(T, gpu):
    """A grid whose 17 rows of a column span 4 GiB: 31,580,641 x 1 cells.  Operator and
    three iterations on loads in three windows (the last one at the far end), against the
    windows alone."""
    import ctypes as C
    import scipy.sparse as sp
    from oracle import heat_oracle as H
    from topopt_jl_amd import _lib
    nx, wn = 31580641, 40
    NX, n = nx + 1, 2 * (nx + 1)
    assert NX * 17 * 8 >= 2**32
    lib = T.load_library()
    ptr, order = C.c_void_p(), np.arange(1, n + 1)
    fixed = np.zeros(n, np.uint8)
    fixed[0] = 1
    h = np.array([1.0, 0.7])
    assert lib.tohip_heat_create(C.byref(ptr), 2, _lib.i64ptr(np.array([nx, 1])), _lib.dptr(h), 1.3,
                                 1e-3, 3.0, 1, _lib.i64ptr(order), _lib.u8ptr(fixed), None) == 0
    del order, fixed
    try:
        Ke = H.heat_ke(2, tuple(h), 1.3)  # densities are 1 from the start
        c = np.arange(wn)
        dofs = np.stack([c, c + 1, c + wn + 2, c + wn + 1], 1)  # window nodes, x fastest
        K = sp.csr_matrix((np.tile(Ke.ravel(), wn), (np.repeat(dofs, 4, axis=1).ravel(),
                                                     np.tile(dofs, (1, 4)).ravel()))).toarray()
        starts = (1000, 2**24 - 20, nx - wn)
        at = [np.concatenate([s + np.arange(wn + 1), NX + s + np.arange(wn + 1)]) for s in starts]
        g = np.random.default_rng(0)
        b, loads = np.zeros(n), []
        for k, idx in enumerate(at):
            f = np.zeros(2 * (wn + 1))
            # away from the window's ends, and at the grid's own
            on = np.arange(wn - 9, wn + 1) if k == 2 else np.arange(15, 25)
            f[np.concatenate([on, wn + 1 + on])] = g.standard_normal(20)
            b[idx] = f
            loads.append(f)
        y = np.empty(n)
        assert lib.tohip_heat_matvec(ptr, _lib.dptr(b), _lib.dptr(y)) == 0
        for idx, f in zip(at, loads):
            assert np.linalg.norm(y[idx] - K @ f) < 1e-14 * np.linalg.norm(K @ f)
            y[idx] = 0.0
        assert not y.any()
        u, it, res = np.zeros(n), C.c_int64(), C.c_double()
        assert lib.tohip_heat_solve(ptr, _lib.dptr(b), _lib.dptr(u), 0.0, 1e-30, 3, 1, 0,
                                    C.byref(it), C.byref(res)) == 1
        r, p = np.stack(loads), 0.0  # a row a window
        x, diag, rho_prev = np.zeros_like(r), K.diagonal(), 1.0
        for _ in range(3):
            z = r / diag
            rho = (r * z).sum()
            p = z + rho / rho_prev * p
            q = p @ K
            a = rho / (p * q).sum()
            x, r, rho_prev = x + a * p, r - a * q, rho
        assert it.value == 3
        for idx, v in zip(at, x):
            assert np.linalg.norm(u[idx] - v) < 1e-12 * np.linalg.norm(v)
            u[idx] = 0.0
        assert not u.any()
    finally:
        lib.tohip_heat_destroy(ptr)
