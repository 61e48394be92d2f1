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
