"""CPU: which iteration graphs a one-launch PCG solve launches between two looks at its
state, on residual histories of known length."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HARNESS = """
#include "pcg1_schedule.h"
using namespace tohip;
// Solve of `need` iterations (res[i] after i) with the limit maxiter.
extern "C" void run(long long need, long long maxiter, const double* res, double tol,
                    long long* launched, long long* looks, long long* graphs) {
    Pcg1Schedule s;
    const long long end = need < maxiter ? need : maxiter;
    *launched = *looks = *graphs = 0;
    for (;;) {
        *launched += (long long)s.launches * kPcg1GraphIters[s.graph];
        *graphs += s.launches;
        ++*looks;
        if (*launched > end || *looks > 100000) return;  // a launch past the end sets done
        const long long it = *launched;
        s.next(it, maxiter, res[it] * res[it], res[0] * res[0], tol);
    }
}
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    d = tmp_path_factory.mktemp("schedule")
    (d / "h.cpp").write_text(HARNESS)
    so = str(d / "h.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-I",
                    os.path.join(ROOT, "topopt.jl_amd", "csrc"), str(d / "h.cpp"), "-o", so],
                   check=True)
    f = C.CDLL(so).run

    def call(need, maxiter, res, tol):
        out = [C.c_longlong() for _ in range(3)]
        r = np.ascontiguousarray(res, np.float64)
        f(C.c_longlong(need), C.c_longlong(maxiter), r.ctypes.data_as(C.c_void_p),
          C.c_double(tol), *(C.byref(o) for o in out))
        return [o.value for o in out]
    return call


@pytest.mark.parametrize("need", [0, 1, 5, 30, 31])
def test_near_solves_take_one_short_graph(run, need):
    assert run(need, 10000, np.ones(40), 0.0) == [32, 1, 1]


@pytest.mark.parametrize("need", [32, 40, 63, 64, 100, 537, 1268, 8032])
def test_steady_convergence(run, need):
    res = 10.0 ** (-8 * np.arange(need + 400) / need)
    launched, looks, graphs = run(need, 10**6, res, 1e-8)
    assert need < launched <= need + 64
    assert looks <= 8 + need // 192 and graphs <= 12 + need / 56


@pytest.mark.parametrize("maxiter", [0, 1, 20, 32, 33, 60, 70, 150, 1000])
@pytest.mark.parametrize("history", ["steady", "level", "rising"])
def test_iteration_limit(run, maxiter, history):
    """No graphs for iterations that the limit does not allow, whatever the history."""
    k = np.arange(maxiter + 400)
    res = {"steady": 10.0 ** (-k / 1e4), "level": np.ones(k.size), "rising": 1.001 ** k}[history]
    launched, looks, _ = run(10**9, maxiter, res, 1e-30)
    assert maxiter < launched <= max(32, maxiter + 24)
    assert looks <= 6 + maxiter // 60


def test_energy_rule_has_no_prediction(run):
    launched, looks, graphs = run(200, 700, 0.9 ** np.arange(800), 0.0)
    assert (launched, looks, graphs) == (32 + 3 * 64, 4, 4)
