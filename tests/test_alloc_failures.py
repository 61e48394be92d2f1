"""CPU: device allocations that fail, in calls that are then made again.  The library
runs on a stub of the HIP runtime in a process of its own, loaded before it with its
symbols global."""
import json
import os
import subprocess
import sys
import textwrap

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SETUP = textwrap.dedent("""
    import ctypes as C, json, sys
    import numpy as np
    stub = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
    stub.stub_live.restype = stub.stub_bytes.restype = stub.stub_count.restype = C.c_long
    stub.stub_fail_in.argtypes = [C.c_long]
    sys.path.insert(0, sys.argv[2])
    import _pkg
    T = _pkg.load_package()
    from topopt_jl_amd import _lib
    nels = json.loads(sys.argv[3])
    dim = len(nels)

    def context():
        nn = int(np.prod([n + 1 for n in nels]))
        fixed = np.repeat(np.arange(nn) % (nels[0] + 1) == 0, dim).astype(np.uint8)
        return _lib.Context(dim, nels, np.ones(dim), 1.0, 0.3, 1e-3, 3.0, True, None, fixed)

    c = context()
    L, x = c.lib, np.full(c.ncells, 0.5)
    r, z = np.ones(c.ndofs), np.empty(c.ndofs)
""")

ERROR = SETUP + textwrap.dedent("""
    assert L.tohip_set_densities(c.ptr, _lib.dptr(x)) == 0
    stub.stub_fail_in(1)
    assert L.tohip_mg_apply(c.ptr, _lib.dptr(r), _lib.dptr(z)) == _lib.TOHIP_ERR_HIP
    assert "out of memory" in L.tohip_last_error(c.ptr).decode()
    assert L.tohip_set_densities(c.ptr, _lib.dptr(x)) == 0
    stub.stub_fail_in(3)
    try:
        T.FEASolver(T.HIPMatrixFreeSolver, T.HeatTree(nels))
        raise SystemExit("created")
    except T.TohipError:
        pass
    assert L.tohip_set_densities(c.ptr, _lib.dptr(x)) == 0
    assert L.tohip_mg_apply(c.ptr, _lib.dptr(r), _lib.dptr(z)) == 0
    T.FEASolver(T.HIPMatrixFreeSolver, T.HeatTree(nels))
""")

SWEEP = SETUP + textwrap.dedent("""

    def held():
        b = C.c_int64()
        assert L.tohip_memory(c.ptr, C.byref(b), None, None) == 0
        return b.value

    assert L.tohip_set_densities(c.ptr, _lib.dptr(x)) == 0
    base, k, rows = stub.stub_bytes() - held(), 0, []
    while True:
        k += 1
        stub.stub_fail_in(k)
        rc = L.tohip_mg_apply(c.ptr, _lib.dptr(r), _lib.dptr(z))
        stub.stub_fail_in(0)
        # device memory beyond what the context says it holds; then a call that rebuilds
        # the operator of whatever hierarchy there is
        over = stub.stub_bytes() - held() - base
        rc2 = L.tohip_set_densities(c.ptr, _lib.dptr(x))
        rows.append((rc, over, rc2))
        if rc == 0:
            break
        if k % 3 == 0:  # and the call made again
            assert L.tohip_mg_apply(c.ptr, _lib.dptr(r), _lib.dptr(z)) == 0
            c = context()
            assert L.tohip_set_densities(c.ptr, _lib.dptr(x)) == 0
            base = stub.stub_bytes() - held()
    del c
    import gc
    gc.collect()
    print(json.dumps(dict(rows=rows, live=stub.stub_live())), flush=True)
""")

# Calls that make their buffers on first use.  Graph launches fail, which ends the
# solver runs after they have all that they need.
GROUPS = SETUP + textwrap.dedent("""
    stub.stub_fail_graphs(1)

    def held():
        b = C.c_int64()
        assert L.tohip_memory(c.ptr, C.byref(b), None, None) == 0
        return b.value

    def start():
        global c, x
        c = context()
        c.lib.tohip_set_densities(c.ptr, _lib.dptr(x))
        c.lib.tohip_set_load(c.ptr, _lib.dptr(r))
        assert c.lib.tohip_filter_setup(c.ptr, 1.5) == 0

    def csr():
        return L.tohip_csr_matvec(c.ptr, _lib.dptr(r), _lib.dptr(z)), 0

    def solve():
        it, rs = C.c_int64(), C.c_double()
        return L.tohip_solve(c.ptr, _lib.dptr(r), None, 0.0, 1e-8, 10, 1, 0, C.byref(it),
                             C.byref(rs)), -2

    def mma():
        o = _lib.SimpOpts(volfrac=0.5, rmin=1.5, move=0.2, oc_tol=1e-9, rel_tol=1e-8,
                          iterations=1, maxiter=10, inner_rel_tol=0.1)
        m = _lib.MmaOpts(s_init=0.5, s_incr=1.2, s_decr=0.7)
        h = np.empty(4), np.empty(4, np.int64), np.empty(4)
        return L.tohip_simp_run_mma(c.ptr, C.byref(o), C.byref(m), _lib.dptr(x.copy()),
                                    _lib.dptr(h[0]), h[1].ctypes.data_as(C.POINTER(C.c_int64)), _lib.dptr(h[2])), -2

    def beso():
        o = _lib.BesoOpts(maxiter=2, vol_limit=0.5, rmin=1.5, er=0.02, tol=1e-4, sens_tol=1e-6,
                          k=4, penalty_p=3.0, rel_tol=1e-8, pcg_maxiter=10)
        res, out, hist = _lib.BesoResultC(), np.empty(c.ncells), np.empty(4)
        return L.tohip_beso_run(c.ptr, C.byref(o), _lib.dptr(np.ones(c.ncells)), None,
                                _lib.dptr(out), C.byref(res), _lib.dptr(hist)), -2

    def filt():
        return L.tohip_filter_setup(c.ptr, 2.5), 0

    for name, f in dict(csr=csr, solve=solve, mma=mma, beso=beso, filt=filt).items():
        start()
        f()
        whole = held()
        start()
        b0, k = held(), 0
        while True:
            k += 1
            stub.stub_fail_in(k)
            rc, good = f()
            stub.stub_fail_in(0)
            err = L.tohip_last_error(c.ptr).decode()
            if k > 40 or rc == good and (rc == 0 or "out of memory" not in err):
                break
            assert rc == -2 and "out of memory" in err, (name, k, rc, err)
            rc, good = f() if k % 2 == 0 else (good, good)
            assert rc == good, (name, k, rc, L.tohip_last_error(c.ptr).decode())
            if k % 2 == 0:
                assert held() == whole, (name, k, held(), whole)
                start()
        assert k > 2 and k < 40, (name, k)
        print(name, k, whole - b0)
    del c
    import gc
    gc.collect()
    assert stub.stub_live() == 0, stub.stub_live()
""")


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("stub") / "hip_host_stub.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-w",
                    os.path.join(ROOT, "tests", "hip_host_stub.c"), "-o", so], check=True)
    return so


def test_error_ends_with_its_call(T, stub):
    """The runtime keeps an error until it is asked for; the next call must not fail of it."""
    p = subprocess.run([sys.executable, "-c", ERROR, stub, ROOT, "[24, 16, 16]"],
                       stdout=subprocess.PIPE, stderr=subprocess.PIPE, timeout=120)
    assert p.returncode == 0, p.stderr.decode()[-2000:]


# coarsest levels: one workgroup's (3x2x2, 4x2), one of sweeps (13x9x5, 39x29)
@pytest.mark.parametrize("nels", [(24, 16, 16), (32, 16), (26, 18, 10), (78, 58)])
def test_multigrid_setup(T, stub, nels):
    """Each allocation of the set-up fails once: nothing is lost, the densities can be
    set, and the call made again succeeds."""
    p = subprocess.run([sys.executable, "-c", SWEEP, stub, ROOT, json.dumps(nels)],
                       stdout=subprocess.PIPE, stderr=subprocess.PIPE, timeout=120)
    assert p.returncode == 0, p.stderr.decode()[-2000:]
    out = json.loads(p.stdout.decode().splitlines()[-1])
    assert len(out["rows"]) > 8
    for k, (rc, over, rc2) in enumerate(out["rows"]):
        assert rc == (0 if k == len(out["rows"]) - 1 else -2), (k, rc)
        assert over == 0 and rc2 == 0, (k, over, rc2)
    assert out["live"] == 0


def test_groups_of_buffers(T, stub):
    """Buffers made on first use: when one of them cannot be had, the call made again gets
    the rest, and no more."""
    p = subprocess.run([sys.executable, "-c", GROUPS, stub, ROOT, "[6, 4, 4]"],
                       stdout=subprocess.PIPE, stderr=subprocess.PIPE, timeout=120)
    assert p.returncode == 0, p.stdout.decode() + p.stderr.decode()[-2000:]
