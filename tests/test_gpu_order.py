"""GPU tests of the caller's DOF order at the entry points: a context with a
shuffled order against one in the library's own, bit for bit, and refused values on
both sides of the lengths where the check (2^16) and the way back to the caller's order
(2^15) move from the host to the device."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GRIDS = [(1, 1), (13, 7), (180, 180), (181, 181), (3, 2, 2), (28, 27, 27), (127, 127), (128, 127)]


def _contexts(T, nels):
    from topopt_jl_amd import _lib
    dim = len(nels)
    node = np.indices([n + 1 for n in nels[::-1]])[::-1].reshape(dim, -1)  # x fastest
    nn = node.shape[1]
    g = np.random.default_rng(nn)
    order = g.permutation(dim * nn) + 1          # caller's 1-based DOF of (node, d)
    fixed = np.repeat(node[0] == 0, dim).astype(np.uint8)
    fixed_p = np.empty_like(fixed)
    fixed_p[order - 1] = fixed
    own = _lib.Context(dim, nels, np.ones(dim), 1.0, 0.3, 1e-3, 3.0, True, None, fixed)
    shuf = _lib.Context(dim, nels, np.ones(dim), 1.0, 0.3, 1e-3, 3.0, True,
                        order.reshape(nn, dim).T, fixed_p)
    return _lib, own, shuf, order - 1, g


@pytest.mark.parametrize("nels", GRIDS)
def test_shuffled_order(T, gpu, nels):
    _lib, own, shuf, order, g = _contexts(T, nels)
    lib, ptr = own.lib, _lib.dptr
    x = g.uniform(0.3, 1.0, own.ncells)
    f, u0 = g.standard_normal(own.ndofs), g.standard_normal(own.ndofs)
    out = {}
    for c in (own, shuf):
        def there(v):
            w = np.empty_like(v)
            if c is own:
                return v.copy()
            w[order] = v
            return w
        assert lib.tohip_set_densities(c.ptr, ptr(x)) == 0
        got = []
        y = np.empty(c.ndofs)
        assert lib.tohip_matvec(c.ptr, ptr(there(u0)), ptr(y)) == 0
        got.append(y)
        it, res = C.c_int64(), C.c_double()
        for zero in (0, 1):
            u = there(u0)
            assert lib.tohip_solve(c.ptr, ptr(there(f)), ptr(u), 0.0, 1e-30, 5, zero, 0,
                                   C.byref(it), C.byref(res)) >= 0
            got.append(u)
            u = there(u0)
            assert lib.tohip_csr_solve(c.ptr, ptr(there(f)), ptr(u), 0.0, 1e-30, 5, zero, 1, 1,
                                       C.byref(it), C.byref(res)) >= 0
            got.append(u)
        # the load kept on the device: prescribed DOFs zeroed
        assert lib.tohip_set_load(c.ptr, ptr(there(f))) == 0
        assert lib.tohip_solve(c.ptr, None, None, 0.0, 1e-30, 5, 1, 0, C.byref(it),
                               C.byref(res)) >= 0
        u = np.empty(c.ndofs)
        assert lib.tohip_get_u(c.ptr, ptr(u)) == 0
        got.append(u)
        out[c] = [v if c is own else v[order] for v in got]
    for a, b in zip(out[own], out[shuf]):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("nels", GRIDS[2:4])
@pytest.mark.parametrize("bad", [np.nan, -np.inf])
def test_refused_values(T, gpu, nels, bad):
    """A refused load or guess leaves the load and the displacement as they were."""
    _lib, _, c, order, g = _contexts(T, nels)
    lib, ptr = c.lib, _lib.dptr
    assert lib.tohip_set_densities(c.ptr, ptr(np.full(c.ncells, 0.5))) == 0
    f = g.standard_normal(c.ndofs)
    it, res = C.c_int64(), C.c_double()

    def solve(f, u, zero=1):
        return lib.tohip_solve(c.ptr, f, u, 0.0, 1e-30, 5, zero, 0, C.byref(it), C.byref(res))

    assert lib.tohip_set_load(c.ptr, ptr(f)) == 0
    assert solve(None, None) >= 0
    u, now = np.empty(c.ndofs), np.empty(c.ndofs)
    assert lib.tohip_get_u(c.ptr, ptr(u)) == 0
    for at in (0, c.ndofs - 1):
        b = f.copy()
        b[at] = bad
        assert lib.tohip_set_load(c.ptr, ptr(b)) == _lib.TOHIP_ERR_ARG
        assert solve(ptr(b), None) == _lib.TOHIP_ERR_ARG
        assert solve(ptr(f), ptr(b), 0) == _lib.TOHIP_ERR_ARG
        for args in ((b, f, 1), (f, b, 0)):
            assert lib.tohip_csr_solve(c.ptr, ptr(args[0]), ptr(args[1].copy()), 0.0, 1e-30, 5,
                                       args[2], 1, 1, C.byref(it),
                                       C.byref(res)) == _lib.TOHIP_ERR_ARG
        assert lib.tohip_get_u(c.ptr, ptr(now)) == 0 and np.array_equal(now, u)
    assert solve(None, None) >= 0
    assert lib.tohip_get_u(c.ptr, ptr(now)) == 0 and np.array_equal(now, u)


@pytest.mark.parametrize("nels", [(12, 9), (255, 254), (256, 255), (40, 40, 39), (181, 179), (181, 180)])
def test_heat_values(T, gpu, nels):
    """Heat: refused values on both sides of the rule; the temperature comes back in
    the order it was given (no iterations: the guess with its prescribed values)."""
    prob = T.HeatConductionProblem(nels, (1.0,) * len(nels), 1.0, Tleft=1.0)
    s = T.FEASolver(T.HIPMatrixFreeSolver, prob, abstol=0.0, reltol=1e-30)
    g = np.random.default_rng(sum(nels))
    s.set_densities(np.full(prob.ncells, 0.5))
    t0 = g.standard_normal(prob.ndofs)
    s.u = t0.copy()
    s(initially_zero=False, maxiter=0)
    assert np.array_equal(s.u, t0)
    free = np.flatnonzero(~prob.fixed.astype(bool))  # prescribed ones are zeroed before
    for at in (free[0], free[-1]):
        b = np.zeros(prob.ndofs)
        b[at] = np.inf
        with pytest.raises(T.TohipError, match="non-finite"):
            s(rhs=b)
        s.u = b
        with pytest.raises(T.TohipError, match="non-finite"):
            s(initially_zero=False)
        s.u = t0.copy()
