"""The work that users of this framework have it do, as cases that can be timed.

A case is a dict of plain values; its "kind" says which entry points a pass
goes through:

  simp     the device-resident SIMP loop (``simp_run``): filter, solve,
           sensitivity, pullback and design update per iteration
  eval     one function and gradient evaluation for an external optimizer:
           (projected) density filter, ComplianceFun, pullbacks, VolumeFun
  heat     one ThermalComplianceFun evaluation: the temperature solve, its
           adjoint and the gradient
  csr      one ComplianceFun evaluation on the assembled-matrix CG solver
  predict  one displacement prediction of the warm-start network
  train    Adam steps of the warm-start network on pairs held on the device

Solves are asked for tighter tolerances than the defaults (1e-8), so that two
correct solvers agree to many digits; an iteration costs the same.
"""
from __future__ import annotations

import functools
import math
import os

import numpy as np
import torch

import _pkg

T = _pkg.load_package()
WEIGHTS = os.path.join(_pkg.PKG_DIR, "weights", "warmstart_%s.npz")
DENSE_MAX = 18000  # unknowns up to which exact() solves a dense system


def listed():
    return [
        # the 2D tutorial size: the reference's solver, every launch counts
        dict(name="simp2d_160x40_fp64", kind="simp", nx=160, ny=40, nz=0, precision="fp64",
             optimizer="oc", volfrac=0.5, rmin=2.0, iterations=6, load="reference"),
        # a large 2D design with the tutorials' optimizer on the multigrid path
        dict(name="simp2d_640x320_mma", kind="simp", nx=640, ny=320, nz=0, precision="mixed_mg",
             optimizer="mma", volfrac=0.4, rmin=3.0, iterations=4, load="reference"),
        # the headline grid on the reference's own solver, FP64 Jacobi PCG
        dict(name="simp3d_120_fp64", kind="simp", nx=120, ny=40, nz=40, precision="fp64",
             optimizer="oc", volfrac=0.3, rmin=1.5, iterations=2, load="centre"),
        # the headline grid and solver
        dict(name="simp3d_120_mg", kind="simp", nx=120, ny=40, nz=40, precision="mixed_mg",
             optimizer="oc", volfrac=0.3, rmin=1.5, iterations=5, load="centre"),
        # the largest design, 12.8 million unknowns
        dict(name="simp3d_256_mg", kind="simp", nx=256, ny=128, nz=128, precision="mixed_mg",
             optimizer="oc", volfrac=0.2, rmin=2.0, iterations=2, load="centre"),
        # one evaluation for an optimizer outside, small box cells, odd counts
        dict(name="eval3d_27x14x10_fp64", kind="eval", nx=27, ny=14, nz=10, hx=1.0, hy=1.5,
             hz=0.75, precision="fp64", rmin=2.0, penalty="rational", projected=True),
        # the same at a size where the multigrid path is chosen, one coarse level odd
        dict(name="eval3d_76x36x28_mg", kind="eval", nx=76, ny=36, nz=28, hx=1.0, hy=1.0,
             hz=1.0, precision="mixed_mg", rmin=1.5, penalty="power", projected=False),
        # the heat tree of the tutorials
        dict(name="heat2d_80x60", kind="heat", nx=80, ny=60, nz=0),
        # conduction in 3D, about a million nodes
        dict(name="heat3d_128x96x80", kind="heat", nx=128, ny=96, nz=80),
        # the assembled-matrix solver
        dict(name="csr3d_60x20x20", kind="csr", nx=60, ny=20, nz=20),
        # a prediction at the headline grid, with the trained weights
        dict(name="predict_120x40x40", kind="predict", nx=120, ny=40, nz=40),
        # training as the driver does it: batches of 8
        dict(name="train_64x32x32_b8", kind="train", nx=64, ny=32, nz=32, batch=8, steps=2),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["simp", "simp", "eval", "eval", "heat", "csr", "predict", "train"])
    flat = rng.random() < 0.4
    if kind == "simp":
        prec = rng.choice(["fp64", "mixed", "mixed_mg", "mixed_mg"])
        c = dict(kind=kind, precision=prec, optimizer=rng.choice(["oc", "oc", "mma"]),
                 volfrac=round(rng.uniform(0.2, 0.5), 3), rmin=round(rng.uniform(1.5, 3.0), 2),
                 iterations=rng.randint(2, 4))
        if flat:
            nx = _log_int(rng, 60, 700 if prec == "mixed_mg" else 240)
            c.update(nx=nx, ny=2 * max(8, nx // rng.randint(4, 8)), nz=0, load="reference")
        else:
            nx = _log_int(rng, 24, 130 if prec == "mixed_mg" else 70)
            c.update(nx=nx, ny=2 * max(4, nx // rng.randint(4, 7)),
                     nz=2 * max(4, nx // rng.randint(4, 7)),
                     load=rng.choice(["reference", "centre"]))
        if prec == "mixed_mg":  # even cell counts, at least two levels
            for k in ("nx", "ny", "nz"):
                c[k] -= c[k] % 4
        return c
    if kind == "eval":
        prec = rng.choice(["fp64", "fp64", "mixed_mg"])
        nx = _log_int(rng, 20, 96)
        c = dict(kind=kind, nx=nx, ny=2 * max(4, nx // rng.randint(4, 7)),
                 nz=0 if flat else 2 * max(4, nx // rng.randint(4, 7)), hx=1.0,
                 hy=rng.choice([1.0, 1.5]), hz=rng.choice([1.0, 0.75]), precision=prec,
                 rmin=rng.choice([1.5, 2.0, 2.5]),
                 penalty=rng.choice(["power", "rational", "sinh"]), projected=rng.random() < 0.5)
        if prec == "mixed_mg":
            for k in ("nx", "ny", "nz"):
                c[k] -= c[k] % 4
            c.update(hy=1.0, hz=1.0)
        return c
    if kind == "heat":
        if flat:
            return dict(kind=kind, nx=_log_int(rng, 30, 400), ny=_log_int(rng, 30, 300), nz=0)
        return dict(kind=kind, nx=_log_int(rng, 12, 120), ny=_log_int(rng, 12, 90),
                    nz=_log_int(rng, 8, 80))
    if kind == "csr":
        nx = _log_int(rng, 16, 90 if not flat else 200)
        return dict(kind=kind, nx=nx, ny=2 * max(3, nx // 6), nz=0 if flat else 2 * max(3, nx // 6))
    if kind == "predict":
        return dict(kind=kind, nx=8 * rng.randint(3, 20), ny=8 * rng.randint(2, 6),
                    nz=8 * rng.randint(2, 6))
    return dict(kind=kind, nx=8 * rng.randint(3, 8), ny=8 * rng.randint(2, 4),
                nz=8 * rng.randint(2, 4), batch=rng.choice([1, 2, 4, 8]), steps=rng.randint(1, 2))


# ------------------------------------------------------------------ inputs --

def _nels(c):
    return (c["nx"], c["ny"]) + ((c["nz"],) if c["nz"] else ())


@functools.lru_cache(maxsize=2)
def _cantilever(nels, sizes, load):
    return T.PointLoadCantilever(nels, sizes=sizes, load=load)


@functools.lru_cache(maxsize=2)
def _heat_tree(nels):
    return T.HeatTree(nels)


def _smooth(nels, seed, waves=6):
    """A smooth random field over the cells, in [-1, 1]: a few products of
    cosines, in cell order (x fastest)."""
    g = np.random.default_rng(seed)
    n = tuple(nels) + (1,) * (3 - len(nels))
    s = np.zeros((n[2], n[1], n[0]))
    for _ in range(waves):
        ax = [np.cos(g.uniform(0.5, 6.0) * np.pi * (np.arange(m) + 0.5) / m +
                     g.uniform(0, 2 * np.pi)) for m in n]
        s += g.uniform(0.5, 1.0) * ax[2][:, None, None] * ax[1][None, :, None] * ax[0]
    return (s / np.abs(s).max()).reshape(-1)


def _penalty(c):
    return {"power": T.PowerPenaltyFun, "rational": T.RationalPenaltyFun,
            "sinh": T.SinhPenaltyFun}[c["penalty"]](3.0)


def prepare(c, seed):
    kind, nels = c["kind"], _nels(c)
    if kind == "simp":
        prob = _cantilever(nels, None, c["load"])
        s = T.FEASolver(T.HIPMatrixFreeSolver, prob, xmin=1e-9, penalty=T.PowerPenaltyFun(3.0),
                        precision=c["precision"])
        # the first iterations of a run from a slightly perturbed start
        return dict(case=c, solver=s, x0=c["volfrac"] * (1 + 0.4 * _smooth(nels, seed)))
    if kind == "eval":
        prob = _cantilever(nels, (c["hx"], c["hy"], c["hz"])[:len(nels)], "reference")
        s = T.FEASolver(T.HIPMatrixFreeSolver, prob, penalty=_penalty(c), abstol=0.0,
                        reltol=1e-11, cg_max_iter=50000, precision=c["precision"])
        filt = (T.ProjectedDensityFilterFun(s, rmin=c["rmin"],
                                            projection=T.HeavisideProjectionFun(4.0))
                if c["projected"] else T.DensityFilterFun(s, c["rmin"]))
        # a design in mid-run: solid, void and grey
        x = np.clip(0.5 + 0.8 * _smooth(nels, seed), 0.0, 1.0)
        return dict(case=c, filt=filt, comp=T.ComplianceFun(s), vol=T.VolumeFun(s), x=x)
    if kind == "heat":
        s = T.FEASolver(T.HIPMatrixFreeSolver, _heat_tree(nels), penalty=T.PowerPenaltyFun(3.0),
                        abstol=0.0, reltol=1e-12, cg_max_iter=50000)
        x = np.clip(0.5 + 0.7 * _smooth(nels, seed), 0.05, 1.0)
        return dict(case=c, fun=T.ThermalComplianceFun(s), x=x)
    if kind == "csr":
        prob = _cantilever(nels, None, "reference")
        s = T.FEASolver(T.HIPCGAssemblySolver, prob, penalty=T.PowerPenaltyFun(3.0), abstol=0.0,
                        reltol=1e-11, cg_max_iter=50000, preconditioner="jacobi")
        x = np.clip(0.5 + 0.6 * _smooth(nels, seed), 0.1, 1.0)
        return dict(case=c, comp=T.ComplianceFun(s), x=x)
    from topopt_jl_amd import nn as NN
    g = np.random.default_rng(seed)
    if kind == "predict":
        net = NN.WarmStartNet(nels, max_batch=1)
        net.load(_weights(nels))
        return dict(case=c, net=net, x=np.clip(0.5 + 0.8 * _smooth(nels, seed), 0.0, 1.0),
                    f=_tip_load(nels, g))
    net = NN.WarmStartNet(nels, max_batch=c["batch"], max_samples=c["batch"])
    net.set_params(_initial_weights(seed))
    for x, f, u in _pairs(c, seed):
        net.add_sample(x, f, u)
    return dict(case=c, net=net)


def _weights(nels):
    p = WEIGHTS % "x".join(map(str, nels))
    return p if os.path.exists(p) else WEIGHTS % "64x32x32"


def _tip_load(nels, g):
    """A unit load along -y at a node of the free face (node-major)."""
    from topopt_jl_amd import nn as NN
    return NN.cantilever_load(nels, int(g.integers(0, nels[1] + 1)),
                              int(g.integers(0, nels[2] + 1)))


# (cin, cout) of the network's convolutions; the inputs have 6 channels of 8 in use
_CONVS = [(8, 16), (16, 16), (16, 32), (32, 32), (32, 64), (64, 64), (64, 128), (128, 128),
          (192, 64), (64, 64), (96, 32), (32, 32), (48, 16), (16, 16), (16, 8)]


def _initial_weights(seed):
    """He initialisation, biases zero, a small last layer with 3 of 8 outputs in use."""
    g = np.random.default_rng(seed)
    out = []
    for i, (ci, co) in enumerate(_CONVS):
        t = 8 if i == len(_CONVS) - 1 else 27
        w = g.standard_normal((co, t * ci)) * math.sqrt(2.0 / (t * ci))
        if t == 8:
            w *= 0.1
            w[3:] = 0
        out += [w.reshape(-1), np.zeros(co)]
    return np.concatenate(out).astype(np.float32)


def _pairs(c, seed):
    """Training pairs: densities, a tip load and a bending displacement."""
    nels = _nels(c)
    g = np.random.default_rng(seed)
    X, Y, Z = (np.arange(n + 1) / n for n in nels)
    for b in range(c["batch"]):
        x = np.clip(0.4 + 0.6 * _smooth(nels, 1000 * seed + b), 0.0, 1.0)
        a, w = g.uniform(0.5, 2.0), g.uniform(-0.3, 0.3)
        u = np.zeros((nels[2] + 1, nels[1] + 1, nels[0] + 1, 3))
        u[..., 1] = -a * X**2 * (3 - X)
        u[..., 0] = a * (X * (2 - X)) * (Y[None, :, None] - 0.5) * nels[1] / nels[0]
        u[..., 2] = w * X**2 * (Z[:, None, None] - 0.5)
        yield x, _tip_load(nels, g), u.reshape(-1)


# -------------------------------------------------------------------- pass --

def run(st):
    c = st["case"]
    if c["kind"] == "simp":
        r = T.simp_run(st["solver"], volfrac=c["volfrac"], rmin=c["rmin"],
                       iterations=c["iterations"], x0=st["x0"], rel_tol=1e-11, move=0.2,
                       optimizer=c["optimizer"])
        return dict(x=r.x, obj=r.obj, u=st["solver"].u)
    if c["kind"] == "eval":
        xf = st["filt"](T.PseudoDensities(st["x"]))
        obj = st["comp"](xf)
        grad = st["filt"].pullback(st["comp"].pullback())
        return dict(x=xf.x, obj=obj, cell=st["comp"].cell_comp, grad=grad, vol=st["vol"](xf))
    if c["kind"] == "heat":
        obj = st["fun"](T.PseudoDensities(st["x"]))
        return dict(obj=obj, grad=st["fun"].pullback(), T=st["fun"].solver.u)
    if c["kind"] == "csr":
        obj = st["comp"](T.PseudoDensities(st["x"]))
        return dict(obj=obj, grad=st["comp"].pullback(), u=st["comp"].solver.u)
    if c["kind"] == "predict":
        return st["net"].predict(st["x"], st["f"])
    st["net"].train(c["steps"], c["batch"], 2e-4, seed=1)
    return st["net"].get_params()


def _solve_iterations(c):
    """Iterations of one solve to the tolerance asked for, roughly."""
    n = max(_nels(c))
    if c["kind"] == "heat":
        return 5 * n
    return 45 if c.get("precision") == "mixed_mg" else 10 * n


def work(c):
    nels = _nels(c)
    dim, cells = len(nels), math.prod(nels)
    nodes = math.prod(n + 1 for n in nels)
    if c["kind"] in ("predict", "train"):
        from topopt_jl_amd import nn as NN
        flops = NN.conv_flops(nels, c.get("batch", 1))
        par = 1463624
        if c["kind"] == "predict":  # densities and load in, displacement out, BF16 weights
            return dict(bytes=8 * cells + 24 * nodes + 12 * nodes + 2 * par, flops=flops)
        # features, targets, parameters and both moments; forward, input and weight gradients
        return dict(bytes=c["steps"] * (c["batch"] * (16 * cells + 12 * nodes) + 28 * par),
                    flops=3 * flops * c["steps"])
    nd = nodes * (1 if c["kind"] == "heat" else dim)
    low = c.get("precision") in ("mixed", "mixed_mg")
    s = 4 if low else 8
    solves = c.get("iterations", 1) * (2 if c["kind"] == "heat" else 1)
    its = _solve_iterations(c) * solves
    nc = 1 << dim
    # an iteration reads and writes x, r and p and reads the diagonal and the moduli
    sweep = 7 * s * nd + s * cells
    elem = cells * 2 * (nc if c["kind"] == "heat" else dim * nc) * nc
    return dict(bytes=its * sweep + solves * (6 * 8 * cells + 16 * nd),
                flops=its * (elem + 10 * nd))


# ------------------------------------------------------- the same in 64 bits --
# Plain dense algebra on small grids (in the problem's numbering of the
# unknowns), the network in float64 torch.

_CORNERS = [(0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1)]


def exact(c, seed):
    if c["kind"] == "predict":
        return _exact_predict(c, seed)
    if c["kind"] == "train":
        return _exact_train(c, seed)
    nels = _nels(c)
    unknowns = math.prod(n + 1 for n in nels) * (1 if c["kind"] == "heat" else len(nels))
    if unknowns * math.sqrt(c.get("iterations", 1)) > 2.5 * DENSE_MAX or unknowns > DENSE_MAX:
        return None
    if c["kind"] == "heat":
        return _exact_heat(c, seed)
    if c["kind"] == "csr":
        x = np.clip(0.5 + 0.6 * _smooth(nels, seed), 0.1, 1.0)
        obj, cell, grad, u = _Dense(nels, (1.0,) * len(nels), "reference").compliance(
            x, 1e-3, lambda v: (v**3, 3 * v**2))
        return dict(obj=obj, grad=grad, u=u)
    if c["kind"] == "eval":
        return _exact_eval(c, seed)
    return _exact_simp(c, seed) if c["optimizer"] == "oc" else None


def _gauss(dim):
    a = 1 / math.sqrt(3.0)
    pts = [-a, a]
    return [(p, q, r) for p in pts for q in pts for r in (pts if dim == 3 else [0.0])]


def _shape_grads(dim, h):
    """Gradients of the corner shape functions at the Gauss points, and the weight."""
    out = []
    cs = _CORNERS[:1 << dim]
    for p in _gauss(dim):
        G = np.zeros((len(cs), dim))
        for a, cc in enumerate(cs):
            sg = [2 * v - 1 for v in cc]
            N1 = [(1 + sg[d] * p[d]) / 2 for d in range(dim)]
            for d in range(dim):
                G[a, d] = sg[d] / h[d] * math.prod(N1[e] for e in range(dim) if e != d)
        out.append(G)
    return out, math.prod(h) / 2**dim


class _Dense:
    """A point-load cantilever (E = 1, nu = 0.3) by dense Cholesky."""

    def __init__(self, nels, h, load):
        prob = _cantilever(tuple(nels), tuple(h) if h else None, load)
        dim = self.dim = len(nels)
        lam, mu = 0.3 / (1.3 * 0.4), 1 / 2.6
        C = np.zeros((dim, dim, dim, dim))
        I = np.eye(dim)
        C += lam * np.einsum("ij,kl->ijkl", I, I)
        C += mu * (np.einsum("ik,jl->ijkl", I, I) + np.einsum("il,jk->ijkl", I, I))
        grads, w = _shape_grads(dim, h)
        n = dim << dim
        Ke = sum(w * np.einsum("aj,ijkl,bl->aibk", G, C, G) for G in grads).reshape(n, n)
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.Ke = torch.tensor(Ke, device=dev)
        self.dofs = torch.tensor(prob.cell_dofs.T - 1, device=dev)  # cells x n
        self.free = torch.tensor(np.flatnonzero(prob.fixed == 0), device=dev)
        self.f = torch.tensor(prob.f, device=dev)
        self.nd = prob.ndofs

    def solve(self, E):
        K = _assemble(self.nd, self.dofs, self.Ke, E)
        return _free_solve(K, self.free, self.f)

    def energies(self, u):
        ue = u[self.dofs]
        return ((ue @ self.Ke) * ue).sum(1)

    def compliance(self, x, xmin, pen):
        v, dv = (torch.tensor(a, device=self.Ke.device) for a in pen(np.asarray(x)))
        rho, drho = xmin + (1 - xmin) * v, (1 - xmin) * dv
        u = self.solve(rho)
        ce = self.energies(u)
        return (float((rho * ce).sum()), ce.cpu().numpy(), (-drho * ce).cpu().numpy(),
                u.cpu().numpy())


def _assemble(nd, dofs, Ke, E):
    K = torch.zeros(nd, nd, dtype=torch.float64, device=Ke.device)
    n = dofs.shape[1]
    for a in range(n):
        idx = dofs[:, a:a + 1] * nd + dofs
        K.view(-1).index_put_((idx.reshape(-1),), (E[:, None] * Ke[a][None, :]).reshape(-1),
                              accumulate=True)
    return K


def _free_solve(K, free, f):
    A = K[free][:, free]
    L = torch.linalg.cholesky(A)
    b = f[free][:, None]
    x = torch.cholesky_solve(b, L)
    for _ in range(3):  # iterative refinement
        x = x + torch.cholesky_solve(b - A @ x, L)
    u = torch.zeros_like(f)
    u[free] = x[:, 0]
    return u


class _Filter:
    """The density filter: node weights (rmin - distance) around a cell centre,
    a node's value the sum over the cells that share it."""

    def __init__(self, nels, h, rmin):
        self.nels = tuple(nels) + (1,) * (3 - len(nels))
        self.dim = dim = len(nels)
        H = [int(math.ceil(rmin / h[d] + 1)) for d in range(dim)] + [0] * (3 - dim)
        self.taps = []
        for o in np.ndindex(*(2 * k + 2 for k in H)):
            off = [o[d] - H[d] for d in range(3)]
            r = math.sqrt(sum(((off[d] - 0.5) * h[d])**2 for d in range(dim)))
            if r < rmin and (dim == 3 or off[2] == 0):
                self.taps.append((off, rmin - r))
        one = self._gather(self._nodes(np.ones(self.nels[::-1])))
        self.den = one

    def _nshape(self):
        n = self.nels
        return (n[2] + 1 if self.dim == 3 else 1, n[1] + 1, n[0] + 1)

    def _nodes(self, x):
        S = np.zeros(self._nshape())
        n = self.nels
        for c in _CORNERS[:1 << self.dim]:
            S[c[2]:c[2] + n[2], c[1]:c[1] + n[1], c[0]:c[0] + n[0]] += x
        return S

    def _windows(self, off):
        sl = []
        for d in (2, 1, 0):
            n = self.nels[d]
            N = n + 1 if (d < self.dim) else 1
            lo, hi = max(0, -off[d]), min(n, N - off[d])
            sl.append((slice(lo, max(lo, hi)), slice(lo + off[d], max(lo, hi) + off[d])))
        return tuple(s[0] for s in sl), tuple(s[1] for s in sl)

    def _gather(self, S):
        y = np.zeros(self.nels[::-1])
        for off, w in self.taps:
            a, b = self._windows(off)
            y[a] += w * S[b]
        return y

    def apply(self, x):
        return (self._gather(self._nodes(x.reshape(self.nels[::-1]))) / self.den).reshape(-1)

    def transpose(self, y):
        v = y.reshape(self.nels[::-1]) / self.den
        S = np.zeros(self._nshape())
        for off, w in self.taps:
            a, b = self._windows(off)
            S[b] += w * v[a]
        n = self.nels
        out = np.zeros(n[::-1])
        for c in _CORNERS[:1 << self.dim]:
            out += S[c[2]:c[2] + n[2], c[1]:c[1] + n[1], c[0]:c[0] + n[0]]
        return out.reshape(-1)


def _exact_eval(c, seed):
    nels = _nels(c)
    h = (c["hx"], c["hy"], c["hz"])[:len(nels)]
    x = np.clip(0.5 + 0.8 * _smooth(nels, seed), 0.0, 1.0)
    F = _Filter(nels, h, c["rmin"])
    y = F.apply(x)
    dpost = np.ones_like(y)
    if c["projected"]:
        e, eb = np.exp(-4.0 * y), math.exp(-4.0)
        y, dpost = 1 - e + y * eb, 4.0 * e + eb
    pen = {"power": lambda v: (v**3, 3 * v**2),
           "rational": lambda v: (v / (1 + 3 * (1 - v)), 4 / (1 + 3 * (1 - v))**2),
           "sinh": lambda v: (np.sinh(3 * v) / math.sinh(3), 3 * np.cosh(3 * v) / math.sinh(3))}
    obj, cell, grad, _ = _Dense(nels, h, "reference").compliance(y, 1e-3, pen[c["penalty"]])
    return dict(x=y, obj=obj, cell=cell, grad=F.transpose(grad * dpost), vol=float(y.mean()))


def _exact_simp(c, seed):
    nels = _nels(c)
    h = (1.0,) * len(nels)
    F, K = _Filter(nels, h, c["rmin"]), _Dense(nels, h, c["load"])
    x = c["volfrac"] * (1 + 0.4 * _smooth(nels, seed))
    dv = F.transpose(np.ones_like(x)) / x.size
    objs = []
    for _ in range(c["iterations"]):
        obj, _, grad, u = K.compliance(F.apply(x), 1e-9, lambda v: (v**3, 3 * v**2))
        objs.append(obj)
        dc = F.transpose(grad)
        lo, hi = 1e-30, 1e30
        while hi / lo > 1 + 1e-14:
            lm = math.sqrt(lo * hi)
            new = np.clip(x * np.sqrt(np.maximum(-dc, 0) / (lm * dv)), np.maximum(x - 0.2, 0),
                          np.minimum(x + 0.2, 1))
            lo, hi = (lm, hi) if float(dv @ new) > c["volfrac"] else (lo, lm)
        x = new
    return dict(x=x, obj=np.array(objs), u=u)


def _exact_heat(c, seed):
    nels = _nels(c)
    prob = _heat_tree(nels)
    dim = len(nels)
    grads, w = _shape_grads(dim, (1.0,) * dim)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    Ke = torch.tensor(sum(w * G @ G.T for G in grads), device=dev)
    dofs = torch.tensor(prob.cell_dofs.T - 1, device=dev)
    x = torch.tensor(np.clip(0.5 + 0.7 * _smooth(nels, seed), 0.05, 1.0), device=dev)
    rho, drho = 1e-3 + (1 - 1e-3) * x**3, (1 - 1e-3) * 3 * x**2
    Q = torch.tensor(prob.fixedload, device=dev)
    u = _free_solve(_assemble(prob.ndofs, dofs, Ke, rho),
                    torch.tensor(np.flatnonzero(prob.fixed == 0), device=dev), Q)
    ue = u[dofs]  # the adjoint of Q'T with T = 0 where prescribed is -T
    grad = -drho * ((ue @ Ke) * ue).sum(1)
    return dict(obj=float(Q @ u), grad=grad.cpu().numpy(), T=u.cpu().numpy())


def _layers(p):
    out, at = [], 0
    for i, (ci, co) in enumerate(_CONVS):
        t = 8 if i == 14 else 27
        w = p[at:at + co * t * ci].reshape(co, t, ci)
        at += co * t * ci
        out.append((w, p[at:at + co]))
        at += co
    return out


def _conv(x, wb, k):
    """x [B, D, H, W, ci] zero padded by 1, stride 1, one product per tap."""
    w, b = wb
    x = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
    D, H, W = (n - k + 1 for n in x.shape[1:4])
    y = b.expand(x.shape[0] * D * H * W, -1)
    for t in range(k**3):
        z, r, q = t // (k * k), t // k % k, t % k
        y = y + x[:, z:z + D, r:r + H, q:q + W].reshape(-1, x.shape[4]) @ w[:, t].T
    return y.reshape(x.shape[0], D, H, W, -1)


def _network(p, x):
    L = _layers(p)
    act = lambda i, v: torch.nn.functional.silu(_conv(v, L[i], 3))  # noqa: E731

    def pool(v):
        B, D, H, W, C = v.shape
        return v.reshape(B, D // 2, 2, H // 2, 2, W // 2, 2, C).mean((2, 4, 6))

    def up(v):
        for d in (1, 2, 3):
            v = v.repeat_interleave(2, d)
        return v

    e0 = act(1, act(0, x))
    e1 = act(3, act(2, pool(e0)))
    e2 = act(5, act(4, pool(e1)))
    e3 = act(7, act(6, pool(e2)))
    d2 = act(9, act(8, torch.cat([up(e3), e2], -1)))
    d1 = act(11, act(10, torch.cat([up(d2), e1], -1)))
    d0 = act(13, act(12, torch.cat([up(d1), e0], -1)))
    return _conv(d0, L[14], 2)[..., :3]


def _features(nels, x, f, dev):
    nx, ny, nz = nels
    F = np.zeros((nz, ny, nx, 8))
    F[..., 0] = x.reshape(nz, ny, nx)
    fn = f.reshape(nz + 1, ny + 1, nx + 1, 3)
    for c in _CORNERS:
        F[..., 1:4] += fn[c[2]:c[2] + nz, c[1]:c[1] + ny, c[0]:c[0] + nx]
    F[:, :, 0, 4] = 1  # the clamped face x = 0
    F[..., 5] = 1
    return torch.tensor(F, device=dev)


def _exact_predict(c, seed):
    nels = _nels(c)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    p = torch.tensor(np.load(_weights(nels))["params"].astype(np.float64), device=dev)
    x = np.clip(0.5 + 0.8 * _smooth(nels, seed), 0.0, 1.0)
    f = _tip_load(nels, np.random.default_rng(seed))
    with torch.no_grad():
        return _network(p, _features(nels, x, f, dev)[None]).reshape(-1).cpu().numpy()


def _exact_train(c, seed):
    nels = _nels(c)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    p = torch.tensor(_initial_weights(seed).astype(np.float64), device=dev)
    m, v = torch.zeros_like(p), torch.zeros_like(p)
    data = [(_features(nels, x, f, dev), torch.tensor(u / math.sqrt((u**2).mean()), device=dev))
            for x, f, u in _pairs(c, seed)]
    for step in range(1, c["steps"] + 1):
        p.requires_grad_(True)
        g = torch.zeros_like(p)
        for X, u in data:  # every step's batch is the whole set
            loss = ((_network(p, X[None]).reshape(-1) - u)**2).mean() / len(data)
            g += torch.autograd.grad(loss, p)[0]
        p = p.detach()
        m = 0.9 * m + 0.1 * g
        v = 0.999 * v + 0.001 * g * g
        p = p - 2e-4 * (m / (1 - 0.9**step)) / ((v / (1 - 0.999**step)).sqrt() + 1e-8)
    return p.cpu().numpy()
