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

SCRIPT = textwrap.dedent("""
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


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("stub") / "hip_host_stub.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-w",
                    os.path.join(ROOT, "tests", "hip_host_stub.c"), "-o", so], check=True)
    return so


def test_error_ends_with_its_call(T, stub):
    """The runtime keeps an error until it is asked for; the next call must not fail of it."""
    p = subprocess.run([sys.executable, "-c", SCRIPT, stub, ROOT, "[24, 16, 16]"],
                       stdout=subprocess.PIPE, stderr=subprocess.PIPE, timeout=120)
    assert p.returncode == 0, p.stderr.decode()[-2000:]
