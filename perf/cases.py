"""The work a user of the package has it do, as cases to be timed.

``listed()`` holds the cases, ``draw(rng)`` gives more of the same ranges,
``prepare(case, seed)`` makes what a program has in hand before the call,
``run(state)`` is one pass through the public entry points, ``work(case)`` what
a pass cannot do without, and ``exact(case, seed)`` the same results from
plain 64-bit torch: Q is block tridiagonal in time, so its dense blocks
are eliminated slice by slice.

Kinds:
  loglik     logLike(par) of a space-time model, with or without its gradient
  spatial    logLike(par) of the anisotropic Whittle-Matern model of one slice
  separable  logLike(par) of the separable model Qt (x) Qs
  batch      BatchEvaluator.loglik over several lattices of uneven size
  solve      right-hand sides against a factor that is held
  selinv     factorisation, log-determinant and selected inverse (qinv)
  mean       conditional mean by IC(0) PCG with FP64 residual replacement
  probes     FP32 block PCG for 64 probes and their estimate of Q_c^-1
  network    forward and backward pass of the preconditioner network
"""
import math

import numpy as np
import torch

import spdepy_amd as sp
from spdepy_amd import spdes
from spdepy_amd.batch import BatchEvaluator
from spdepy_amd.krylov import IterativeSolver
from spdepy_amd.learned import LearnedPreconditioner
from spdepy_amd.plan import Plan

LEAF = 128      # the package's own leaf size


def _lattice(kind, M, N, T, bc, **more):
    return dict(kind=kind, M=M, N=N, T=T, bc=bc, **more)


def listed():
    return [
        # one evaluation inside an optimiser on a small spatial data set
        dict(name="spatial_100x100", **_lattice("spatial", 100, 100, 1, 3, m=500)),
        # the small stationary fit: a few milliseconds, launches and latency count
        dict(name="loglik_iso_30x30x10", **_lattice("loglik", 30, 30, 10, 1, model="iso", m=200, r=1, grad=True)),
        # an anisotropic fit on a 40 x 40 data grid with a border of 10 cells
        dict(name="loglik_ani_60x60x12", **_lattice("loglik", 60, 60, 12, 3, model="ani", m=2000, r=1, grad=True)),
        # the full-size B-spline model (386 parameters), one step of its fit
        dict(name="loglik_bspline_100x100x20",
             **_lattice("loglik", 100, 100, 20, 1, model="bspline", m=5000, r=1, grad=True)),
        # values only (a line search, a profile likelihood) for three realisations on a periodic lattice
        dict(name="value_iso_73x58x9", **_lattice("loglik", 73, 58, 9, 2, model="iso", m=1500, r=3, grad=False)),
        # separable model, Q with a 75-point pattern
        dict(name="separable_40x36x10", **_lattice("separable", 40, 36, 10, 3, m=1000)),
        # many models of uneven size at once over a pool of streams
        dict(name="batch_8_models", kind="batch", bc=1, m=1000,
             shapes="40x40x5 57x83x7 101x64x6 73x73x10 120x48x9 90x111x5 66x95x8 45x118x7"),
        # 100 right-hand sides (probes, realisations) against one factor
        dict(name="solve_100_81x67x9", **_lattice("solve", 81, 67, 9, 3, k=100)),
        # marginal variances: factor, log-determinant and selected inverse
        dict(name="selinv_64x64x16", **_lattice("selinv", 64, 64, 16, 3, m=1500)),
        # the factor-free route at full size: conditional mean, and the probes of its gradient
        dict(name="mean_100x100x20", **_lattice("mean", 100, 100, 20, 1, m=5000)),
        dict(name="probes_100x100x20", **_lattice("probes", 100, 100, 20, 1, m=5000, tol=1e-3)),
        # one training pass of the preconditioner network at the size it is trained on
        dict(name="network_100x100x20", **_lattice("network", 100, 100, 20, 1)),
    ]


def draw(rng):
    """Sizes spread over their logarithm; lattices up to those listed."""
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def cells(lo, hi, tlo, thi, most):
        while True:
            M, N, T = size(lo, hi), size(lo, hi), size(tlo, thi)
            if M * N * T <= most:
                return M, N, T

    def m_of(M, N, T):
        n = M * N * T
        return max(8, min(int(n * math.exp(rng.uniform(math.log(0.01), math.log(0.2)))), 8000, n))
    kind = rng.choice(["loglik", "loglik", "loglik", "spatial", "separable", "batch", "solve", "selinv", "mean", "probes",
                       "network"])
    if kind == "loglik":
        model = rng.choice(["iso", "ani", "bspline"])
        bc = rng.choice([1, 3] if model == "bspline" else [1, 2, 3])
        M, N, T = cells(8, 110, 3, 20, 40000 if bc == 2 else 160000)
        return _lattice(kind, M, N, T, bc, model=model, m=m_of(M, N, T), r=rng.choice([1, 1, 1, 2, 5]),
                        grad=rng.random() < 0.75)
    if kind == "spatial":
        M, N, T = cells(20, 160, 1, 1, 20000)
        return _lattice(kind, M, N, T, 3, m=m_of(M, N, T))
    if kind == "separable":
        M, N, T = cells(12, 60, 3, 12, 20000)
        return _lattice(kind, M, N, T, 3, m=m_of(M, N, T))
    if kind == "batch":
        shapes = ["%dx%dx%d" % cells(24, 120, 4, 10, 60000) for _ in range(rng.randint(2, 8))]
        return dict(kind=kind, bc=1, m=rng.randint(100, 2000), shapes=" ".join(shapes))
    if kind == "solve":
        M, N, T = cells(16, 100, 3, 16, 80000)
        return _lattice(kind, M, N, T, 3, k=size(1, 128))
    if kind == "selinv":
        M, N, T = cells(16, 100, 3, 16, 80000)
        return _lattice(kind, M, N, T, rng.choice([1, 3]), m=m_of(M, N, T))
    M, N, T = cells(16, 100, 4, 20, 200000)
    if kind == "mean":
        return _lattice(kind, M, N, T, 1, m=m_of(M, N, T))
    if kind == "probes":
        return _lattice(kind, M, N, T, 1, m=m_of(M, N, T), tol=rng.choice([1e-3, 1e-4]))
    return _lattice(kind, M, N, T, 1)


# ---------------------------------------------------------------- inputs
def _axis(n):
    return (np.arange(n) + 0.5) / n


def _nbs(case):
    return 8 if min(case["M"], case["N"]) >= 64 else 3


def _parameters(case, rng):
    """Parameters over the ranges the models are fitted in; tau = 100."""
    tau = [math.log(100.0)]
    if case["kind"] == "spatial":
        return np.array([rng.uniform(math.log(0.3), math.log(5.0)), rng.uniform(math.log(0.1), 0.0)]
                        + list(0.3 * rng.normal(size=2)) + tau)
    if case["kind"] == "separable":
        return np.hstack([0.3 * rng.normal(size=9), math.log(0.5) + 0.3 * rng.normal(size=9),
                          0.3 * rng.normal(size=18), [math.log(rng.uniform(0.3, 0.9))], tau])
    if case.get("model") == "bspline" or case["kind"] in ("mean", "probes"):
        Np = _nbs(case) ** 2
        return np.hstack([0.1 * rng.normal(size=Np), math.log(0.5) + 0.1 * rng.normal(size=Np),
                          0.3 * rng.normal(size=4 * Np), [0.0], tau])
    a, phi = math.sqrt(rng.uniform(0.05, 1.0)), rng.uniform(0.0, 2.0 * math.pi)
    v = [] if case.get("model", "iso") == "iso" else list(0.4 * rng.normal(size=2))
    return np.array([rng.uniform(math.log(0.1), math.log(10.0)), rng.uniform(math.log(0.1), math.log(5.0))] + v
                    + [a * math.cos(phi), a * math.sin(phi), 0.2 * rng.normal()] + tau)


def _data(case, rng, r=1):
    """Observed cells in order, and a smooth field there with noise of 0.1."""
    M, N, T, m = case["M"], case["N"], case["T"], case["m"]
    idx = np.sort(rng.choice(M * N * T, m, replace=False))
    x, y, t = (idx % M + 0.5) / M, (idx // M % N + 0.5) / N, (idx // (M * N)) / max(T - 1, 1)
    cols = []
    for _ in range(r):
        f = np.zeros(m)
        for _ in range(6):
            k = rng.normal(size=3) * np.array([6.0, 6.0, 4.0])
            f += 0.4 * rng.normal() * np.cos(k[0] * x + k[1] * y + k[2] * t + rng.uniform(0, 2 * math.pi))
        cols.append(f + 0.1 * rng.normal(size=m))
    return idx, np.column_stack(cols) if r > 1 else cols[0]


def _inputs(case, seed):
    """(parameters, observed cells, observations) of the seed."""
    rng = np.random.default_rng([seed, case["M"], case["N"], case["T"]])
    par = _parameters(case, rng)
    idx, y = _data(case, rng, case.get("r", 1)) if "m" in case else (None, None)
    return par, idx, y


def _model(case):
    M, N, T, bc = (case[k] for k in ("M", "N", "T", "bc"))
    kind = case["kind"]
    if kind == "spatial":
        return spdes.WhittleMaternAnisotropic2D(grid=sp.grid(x=_axis(M), y=_axis(N)), bc=bc)
    nbs = _nbs(case) if case.get("model") == "bspline" or kind in ("mean", "probes") else 3
    g = sp.grid(x=_axis(M), y=_axis(N), t=np.arange(float(T)), Nbs=nbs)
    if kind == "separable":
        return spdes.SeperableSpatialTemporal2D(grid=g, bc=bc)
    g0 = sp.grid(x=_axis(M), y=_axis(N), Nbs=nbs)
    mod0 = spdes.WhittleMatern2D(grid=g0, bc=bc)
    mod0.setPars(_MOD0)
    cls = {"iso": spdes.AdvectionIDiffusion2D, "ani": spdes.AdvectionDiffusion2D,
           "bspline": spdes.VarAdvectionVarDiffusion2D}
    return cls["bspline" if kind in ("mean", "probes") else case.get("model", "iso")](grid=g, mod0=mod0, bc=bc)


_MOD0 = np.array([0.0, math.log(0.5), 0.0])   # the initial state: kappa 1, gamma 0.5


def _members(case):
    out = []
    for i, s in enumerate(case["shapes"].split()):
        M, N, T = (int(v) for v in s.split("x"))
        out.append(_lattice("loglik", M, N, T, case["bc"], model="iso", m=min(case["m"] * (i + 1), 8000, M * N * T // 2)))
    return out


def _weights(case, idx, tau):
    """tau times the number of observations of each cell (device)."""
    w = np.zeros(case["M"] * case["N"] * case["T"])
    w[idx] = tau
    return torch.as_tensor(w).cuda()


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        models, pars = [], []
        for i, c in enumerate(_members(case)):
            par, idx, y = _inputs(c, seed + 1000 * i)
            mod = _model(c)
            mod.initFit(y, idx=idx, fitQ0=False)
            models.append(mod)
            pars.append(par)
        return dict(kind=kind, evaluator=BatchEvaluator(models, nstreams=8), pars=pars)
    if kind == "network":
        shape = (case["M"], case["N"], case["T"])
        feat, dout, theta = _network_inputs(case, seed)
        feat, dout = torch.as_tensor(feat).cuda(), torch.as_tensor(dout).cuda()
        return dict(kind=kind, net=LearnedPreconditioner(params=theta), feat=feat, dout=dout, shape=shape)
    par, idx, y = _inputs(case, seed)
    mod = _model(case)
    if kind in ("loglik", "spatial", "separable"):
        if kind == "loglik":
            mod.initFit(y, idx=idx, fitQ0=False)
        else:
            mod.initFit(y, idx=idx)
        return dict(kind=kind, mod=mod, par=par, grad=case.get("grad", True))
    eng = mod._engine()
    qval = eng.assemble(mod._coeffs(par))
    if kind == "solve":
        plan = Plan(case["M"], case["N"], case["T"], case["bc"], leaf_max=LEAF)
        plan.factor(0, qval)
        return dict(kind=kind, plan=plan, rhs=torch.as_tensor(_rhs(case, seed)).cuda())
    add = _weights(case, idx, math.exp(par[-1]))
    if kind == "selinv":
        return dict(kind=kind, eng=eng, qval=qval, add=add)
    state = dict(kind=kind, it=IterativeSolver(eng.plan), qval=qval, add=add)
    if kind == "mean":
        state["b"] = torch.as_tensor(_sty(case, idx, y, math.exp(par[-1]))).cuda()
    else:
        state["V"] = torch.as_tensor(_signs(case, seed)).cuda()
        state["tol"] = case["tol"]
    return state


def _rhs(case, seed):
    n = case["M"] * case["N"] * case["T"]
    return np.random.default_rng([seed, 1]).normal(size=(n, case["k"]))


def _sty(case, idx, y, tau):
    b = np.zeros(case["M"] * case["N"] * case["T"])
    b[idx] = tau * y
    return b


def _signs(case, seed):
    n = case["M"] * case["N"] * case["T"]
    return np.random.default_rng([seed, 2]).choice(np.array([-1.0, 1.0], np.float32), size=(n, 64))


def _network_inputs(case, seed):
    """Jacobi-scaled stencil coefficients (most in [-0.5, 0]), the loss
    gradient of the 22 corrections, and weights of the trained ones' size."""
    rng = np.random.default_rng([seed, 3])
    P = case["M"] * case["N"] * case["T"]
    feat = np.zeros((P, 8), np.float32)
    feat[:, 0] = rng.random(P) < 0.025
    feat[:, 1:7] = -0.5 * rng.random((P, 6), dtype=np.float32)
    dout = (rng.standard_normal((P, 22), dtype=np.float32) / P).astype(np.float32)
    theta = []
    for layer, cin in enumerate((8, 32, 32, 32)):
        W = (math.sqrt(2.0 / (9 * cin)) * rng.normal(size=(9 * cin, 32))).astype(np.float32)
        b = (0.02 * rng.normal(size=32)).astype(np.float32)
        if layer == 3:
            W[:, 22:] = b[22:] = 0.0
        theta += [W.ravel(), b]
    return feat, dout, np.concatenate(theta)


# ------------------------------------------------------------------ pass
def run(state):
    kind = state["kind"]
    if kind in ("loglik", "spatial", "separable"):
        out = state["mod"].logLike(state["par"], grad=state["grad"])
        return (np.float64(out[0]), out[1]) if state["grad"] else (np.float64(out),)
    if kind == "batch":
        return [(np.float64(v), g) for v, g in state["evaluator"].loglik(state["pars"])]
    if kind == "solve":
        return state["plan"].solve(0, state["rhs"])
    if kind == "selinv":
        fac = spdes.Factor(state["eng"], 0, state["qval"], state["add"])
        return np.float64(fac.logdet()), fac.selinv()
    if kind == "network":
        net = state["net"]
        acts = net.forward(state["feat"], state["shape"])
        return acts[-1], net.backward(acts, state["dout"], state["shape"])
    it = state["it"]
    logdet = it.factor(state["qval"], state["add"])
    if kind == "mean":
        x, _ = it.replace(state["b"])
        return np.float64(logdet), x
    U, _ = it.solve(state["V"], tol=state["tol"])
    return U, it.hutch_pattern(U, state["V"])


# ------------------------------------------------------------------ work
_INFO = {}


def _info(M, N, T, bc, wide=False):
    key = (M, N, T, bc, wide)
    if key not in _INFO:
        _INFO[key] = Plan(M, N, T, bc, leaf_max=LEAF, host_only=True, wide=wide).info
    return _INFO[key]


def work(case):
    """Sparse Cholesky and selected-inverse operations of the lattice's
    nested dissection; bytes of what comes in and goes out once."""
    kind = case["kind"]
    if kind == "batch":
        parts = [work(dict(c, r=1, grad=True)) for c in _members(case)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    M, N, T, bc = (case[k] for k in ("M", "N", "T", "bc"))
    n = M * N * T
    if kind == "network":
        per = 9 * (8 + 3 * 32) * 32
        return dict(bytes=4.0 * n * (8 + 22 + 32), flops=2.0 * n * (2 * per + 9 * 3 * 32 * 32))
    i = _info(M, N, T, bc, kind == "separable")
    if kind in ("loglik", "separable", "spatial"):
        fl = float(i["flops_factor"])
        if case.get("grad", True):
            fl += i["flops_selinv"]
        one = i if kind == "spatial" else _info(M, N, 1, bc)
        fl += one["flops_factor"] * (1 if kind != "loglik" else 2)
        if case.get("grad", True):
            fl += one["flops_selinv"] * (1 if kind != "loglik" else 2)
        return dict(bytes=8.0 * case["m"] * (1 + case.get("r", 1)), flops=fl)
    if kind == "solve":
        return dict(bytes=8.0 * (i["nnz_L"] + 2 * n * case["k"]), flops=4.0 * i["nnz_L"] * case["k"])
    if kind == "selinv":
        return dict(bytes=8.0 * (2 * i["nnz_struct"] + n), flops=float(i["flops_factor"] + i["flops_selinv"]))
    if kind == "mean":
        return dict(bytes=8.0 * (i["nnz_struct"] + 3 * n), flops=2.0 * i["nnz_struct"])
    return dict(bytes=16.0 * i["nnz_struct"] + 8.0 * n + 2 * 4.0 * 64 * n, flops=2.0 * 64 * i["nnz_struct"])


# ----------------------------------------------------- the same in 64 bits
_F64 = torch.float64


def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _splines(t, lo, hi, nb):
    """Quadratic B-splines on uniform knots, the outermost two summed."""
    kn = np.linspace(lo - 2 * (hi - lo) / nb, hi + 2 * (hi - lo) / nb, nb + 5)

    def bump(i, d):
        if d == 0:
            last = (t <= kn[i + 1]) if i == nb + 3 else (t < kn[i + 1])
            return ((t >= kn[i]) & last).astype(np.float64)
        return ((t - kn[i]) / (kn[i + d] - kn[i]) * bump(i, d - 1)
                + (kn[i + d + 1] - t) / (kn[i + d + 1] - kn[i + 1]) * bump(i + 1, d - 1))
    b = [bump(i, 2) for i in range(nb + 2)]
    return np.stack([b[0] + b[1]] + b[2:-2] + [b[-2] + b[-1]], 1)


class _Cells:
    """One slice: spacing, neighbours under the boundary rule, bases."""

    def __init__(self, M, N, bc, nbs):
        self.M, self.N, self.bc, self.nbs, self.Ns = M, N, bc, nbs, M * N
        x, y = _axis(M), _axis(N)
        self.hx, self.hy = (x[-1] - x[0]) / (M - 1), (y[-1] - y[0]) / (N - 1)
        self.V = self.hx * self.hy
        k = np.arange(M * N)
        self.i, self.j = k % M, k // M
        self.x, self.y = x, y

    def basis(self, dx, dy):
        ex, ey = (self.hx / 2, self.hy / 2) if dx or dy else (0.0, 0.0)
        bx = _splines(self.x[self.i] + dx, self.x[0] - ex, self.x[-1] + ex, self.nbs)
        by = _splines(self.y[self.j] + dy, self.y[0] - ey, self.y[-1] + ey, self.nbs)
        return torch.as_tensor((by[:, :, None] * bx[:, None, :]).reshape(self.Ns, -1), device=_dev())

    def faces(self):
        """Bases on the W, E, S, N faces."""
        hx, hy = self.hx / 2, self.hy / 2
        return [self.basis(-hx, 0), self.basis(hx, 0), self.basis(0, -hy), self.basis(0, hy)]

    def scatter(self, slots):
        """Dense operator from {(dx, dy): value per cell}; a neighbour outside is
        dropped (bc 3), wrapped (bc 2) or the cell's own row or column (bc 1)."""
        A = torch.zeros(self.Ns * self.Ns, dtype=_F64, device=_dev())
        for (dx, dy), v in slots.items():
            a, b = self.i + dx, self.j + dy
            keep = np.ones(self.Ns, bool)
            if self.bc == 1:
                a, b = np.clip(a, 0, self.M - 1), np.clip(b, 0, self.N - 1)
            elif self.bc == 2:
                a, b = a % self.M, b % self.N
            else:
                keep = (a >= 0) & (a < self.M) & (b >= 0) & (b < self.N)
            rows = np.flatnonzero(keep)
            at = torch.as_tensor(rows * self.Ns + (a + b * self.M)[rows], device=_dev())
            A = A.index_add(0, at, v[torch.as_tensor(rows, device=_dev())])
        return A.view(self.Ns, self.Ns)

    def diffusion(self, W, E, S, N, constant):
        """div(H grad): H per face as (h00, h01, h10, h11)."""
        rx, ry = self.hy / self.hx, self.hx / self.hy
        one = torch.ones(self.Ns, dtype=_F64, device=_dev())
        if self.bc == 1:      # no flux: the boundary faces (with fields: of the first cell alone)
            i, j = torch.as_tensor(self.i, device=_dev()), torch.as_tensor(self.j, device=_dev())
            if constant:
                kw, ke, ks, kn = i > 0, i < self.M - 1, j > 0, j < self.N - 1
            else:
                first = torch.arange(self.Ns, device=_dev()) > 0
                kw, ke, ks, kn = first, one > 0, first, one > 0
            W, E, S, N = ([h * k for h in f] for f, k in ((W, kw), (E, ke), (S, ks), (N, kn)))
        if constant:          # the off-diagonal face terms all read h10
            cS, cN = S[2], N[2]
        else:
            cS, cN = S[1], N[1]
        return {(0, 0): -rx * (E[0] + W[0]) - ry * (N[3] + S[3]),
                (1, 0): rx * E[0] + 0.25 * (cN - cS), (-1, 0): rx * W[0] - 0.25 * (cN - cS),
                (0, 1): ry * N[3] + 0.25 * (E[2] - W[2]), (0, -1): ry * S[3] - 0.25 * (E[2] - W[2]),
                (1, 1): 0.25 * (cN + E[2]), (-1, -1): 0.25 * (cS + W[2]),
                (-1, 1): -0.25 * (cN + W[2]), (1, -1): -0.25 * (cS + E[2])}

    def advection(self, E, N, W, S):
        """Upwind flux of fields on the faces; at a closed border the flux is
        zero and the centre's derivative in that direction is taken as zero."""
        hx, hy = self.hx, self.hy
        cx = (E.abs() + E + W.abs() - W) * hy / 2
        cy = (N.abs() + N + S.abs() - S) * hx / 2
        if self.bc == 1:
            i, j = torch.as_tensor(self.i, device=_dev()), torch.as_tensor(self.j, device=_dev())
            e, w, n, s = i == self.M - 1, i == 0, j == self.N - 1, j == 0
            E, W, N, S = (torch.where(b, torch.zeros_like(f), f) for f, b in ((E, e), (W, w), (N, n), (S, s)))
            cx = (E.abs() + E + W.abs() - W) * hy / 2
            cy = (N.abs() + N + S.abs() - S) * hx / 2
            cx = torch.where(e | w, cx.detach(), cx)
            cy = torch.where(n | s, cy.detach(), cy)
        return {(0, 0): cx + cy, (1, 0): -(E.abs() - E) * hy / 2, (-1, 0): -(W.abs() + W) * hy / 2,
                (0, 1): -(N.abs() - N) * hx / 2, (0, -1): -(S.abs() + S) * hx / 2}

    def advection_constant(self, wx, wy):
        hx, hy, one = self.hx, self.hy, torch.ones(self.Ns, dtype=_F64, device=_dev())
        out = {(0, 0): (wx.abs() * hy + wy.abs() * hx) * one, (1, 0): -(wx.abs() - wx) * hy / 2 * one,
               (-1, 0): -(wx.abs() + wx) * hy / 2 * one, (0, 1): -(wy.abs() - wy) * hx / 2 * one,
               (0, -1): -(wy.abs() + wy) * hx / 2 * one}
        if self.bc == 1:
            i, j = torch.as_tensor(self.i, device=_dev()), torch.as_tensor(self.j, device=_dev())
            e, w, n, s = i == self.M - 1, i == 0, j == self.N - 1, j == 0
            off = (wx.abs() * hy / 2).detach() * (e | w) + (wy.abs() * hx / 2).detach() * (n | s)
            # the model's derivative stencils subtract the border term itself
            c = out[(0, 0)]
            out[(0, 0)] = c - off - off * ((wx - wx.detach()) + (wy - wy.detach()))
            for d, b in (((1, 0), e), ((-1, 0), w), ((0, 1), n), ((0, -1), s)):
                out[d] = torch.where(b, torch.zeros_like(out[d]), out[d])
        return out


def _tensor(g, vx, vy):
    """g I + v v^T as (h00, h01, h10, h11)."""
    return [g + vx * vx, vx * vy, vx * vy, g + vy * vy]


def _add(*parts):
    out = {}
    for s, slots in parts:
        for d, v in slots.items():
            out[d] = out[d] + s * v if d in out else s * v
    return out


class _LogDet(torch.autograd.Function):
    """log|det A|; the gradient A^-T from (A^T A)^-1 A^T after two Newton steps."""

    @staticmethod
    def forward(ctx, A):
        ctx.save_for_backward(A)
        return torch.linalg.slogdet(A)[1]

    @staticmethod
    def backward(ctx, g):
        A, = ctx.saved_tensors
        X = torch.cholesky_inverse(torch.linalg.cholesky(A.T @ A)) @ A.T
        for _ in range(2):
            R = A @ X
            R.diagonal().sub_(1.0)
            X = X - X @ R
        return g * X.T


class _Precision:
    """Diagonal blocks first, mid, last and the block above the diagonal (times
    up[t]) of Q as functions of the parameters, with log|Q|."""

    def __init__(self, case, par):
        M, N, self.T, bc = (case[k] for k in ("M", "N", "T", "bc"))
        kind = case["kind"]
        bspline = case.get("model") == "bspline" or kind in ("mean", "probes")
        c = self.cells = _Cells(M, N, bc, _nbs(case) if bspline else 3)
        one = torch.ones(c.Ns, dtype=_F64, device=_dev())
        eye = {(0, 0): one * c.V}
        zero = 0.0 * one
        if kind == "spatial":
            h = [f * one for f in _tensor(par[1].exp(), par[2], par[3])]
            A = c.scatter(_add((par[0].exp(), eye), (-1.0, c.diffusion(h, h, h, h, True))))
            self.logdet = 2 * _LogDet.apply(A) - c.Ns * math.log(c.V)
            self.first = self.mid = self.last = A.T @ A / c.V
            self.weights, self.up = [1.0], []
            return
        if kind == "separable":
            b, fs = c.basis(0, 0), c.faces()
            kap = (b @ par[:9]).exp()
            hs = [_tensor((f @ par[9:18]).exp(), f @ par[18:27], f @ par[27:36]) for f in fs]
            A = c.scatter(_add((1.0, {(0, 0): c.V * kap}), (-1.0, c.diffusion(*hs, False))))
            Qs = A.T @ A / c.V
            rho = par[36].exp()
            den = 1 - rho * rho
            self.first = self.last = Qs / den
            self.mid = Qs * (1 + rho * rho) / den
            self.upper = -rho / den * Qs
            self.logdet = self.T * (2 * _LogDet.apply(A) - c.Ns * math.log(c.V)) \
                - c.Ns * (self.T - 1) * torch.log(den)
            return
        k0, g0 = math.exp(_MOD0[0]), math.exp(_MOD0[1])
        h0 = [g0 * one, zero, zero, g0 * one]
        A0 = c.scatter(_add((k0, eye), (-1.0, c.diffusion(h0, h0, h0, h0, True))))
        if bspline:
            Np = c.nbs ** 2
            b, fs = c.basis(0, 0), c.faces()
            kap = (b @ par[:Np]).exp()
            hs = [_tensor((f @ par[Np:2 * Np]).exp(), f @ par[2 * Np:3 * Np], f @ par[3 * Np:4 * Np]) for f in fs]
            cx, cy = par[4 * Np:5 * Np], par[5 * Np:6 * Np]
            dif, adv = c.diffusion(*hs, False), c.advection(fs[1] @ cx, fs[3] @ cy, fs[0] @ cx, fs[2] @ cy)
            sigma = par[6 * Np].exp()
        else:
            kap = par[0].exp() * one
            iso = case.get("model", "iso") == "iso"
            vx, vy = (0.0, 0.0) if iso else (par[2], par[3])
            h = [f * one for f in _tensor(par[1].exp(), vx, vy)]
            w = 2 if iso else 4
            dif, adv = c.diffusion(h, h, h, h, bc != 2), c.advection_constant(par[w], par[w + 1])
            sigma = par[w + 2].exp()
        # dt = 1; B = A / V, q the diagonal of Qs
        B = c.scatter(_add((1.0, {(0, 0): c.V * (1 + kap)}), (-1.0, dif), (1.0, adv))) / c.V
        q = c.V * kap * kap / sigma
        self.last = B.T @ (q[:, None] * B)
        self.mid = self.last + torch.diag(q)
        self.first = A0.T @ A0 / c.V + torch.diag(q)
        self.upper = -q[:, None] * B
        self.logdet = 2 * _LogDet.apply(A0) - c.Ns * math.log(c.V) \
            + (self.T - 1) * (2 * _LogDet.apply(B) + torch.log(q).sum())

    def block(self, t):
        return self.first if t == 0 else (self.last if t == self.T - 1 else self.mid)


class _Blocks:
    """Block elimination of Q + diag(add) slice by slice."""

    def __init__(self, P, add):
        self.T, Ns = P.T, P.cells.Ns
        self.U = P.upper.detach() if self.T > 1 else None
        self.inv, self.logdet = [], 0.0
        for t in range(self.T):
            S = P.block(t).detach() + torch.diag(add.view(self.T, Ns)[t])
            if t:
                S = S - self.U.T @ (self.inv[-1] @ self.U)
            L = torch.linalg.cholesky(0.5 * (S + S.T))
            self.logdet += 2 * float(torch.log(torch.diagonal(L)).sum())
            self.inv.append(torch.cholesky_inverse(L))

    def solve(self, B):
        T = self.T
        b = list(B.view(T, -1, B.shape[1]))
        for t in range(1, T):
            b[t] = b[t] - self.U.T @ (self.inv[t - 1] @ b[t - 1])
        x = [None] * T
        for t in range(T - 1, -1, -1):
            x[t] = self.inv[t] @ (b[t] if t == T - 1 else b[t] - self.U @ x[t + 1])
        return torch.cat(x)

    def inverse(self):
        """(t, diagonal block, block above the diagonal) from the last slice."""
        T = self.T
        S = self.inv[-1]
        yield T - 1, S, None
        for t in range(T - 2, -1, -1):
            K = self.inv[t] @ self.U
            KS = K @ S
            S = self.inv[t] + KS @ K.T
            yield t, S, -KS


def _loglik(case, seed):
    par, idx, y = _inputs(case, seed)
    grad = case.get("grad", True)
    p = torch.tensor(par, device=_dev(), requires_grad=True)
    m, r = len(idx), case.get("r", 1)
    y = torch.as_tensor(y, device=_dev()).view(m, r)
    tau, at = math.exp(par[-1]), torch.as_tensor(idx, device=_dev())
    n, T = case["M"] * case["N"] * case["T"], case["T"]
    add = torch.zeros(n, dtype=_F64, device=_dev())
    add[at] = tau
    with torch.set_grad_enabled(grad):
        P = _Precision(case, p)
    with torch.no_grad():
        F = _Blocks(P, add)
        b = torch.zeros(n, r, dtype=_F64, device=_dev())
        b[at] = tau * y
        mu = F.solve(b)
        rss = float(((y - mu[at]) ** 2).sum())
        w = list(mu.view(T, -1, r))
        quad = sum(float((w[t] * (P.block(t) @ w[t])).sum()) for t in range(T)) \
            + sum(2 * float((w[t] * (P.upper @ w[t + 1])).sum()) for t in range(T - 1))
    like = 0.5 * r * float(P.logdet) + 0.5 * m * r * math.log(tau) - 0.5 * r * F.logdet - 0.5 * quad - 0.5 * tau * rss
    if not grad:
        return (np.float64(-like / (m * r)),)
    # -1/2 r Q_c^-1 - 1/2 mu mu^T on the blocks, summed over equal ones
    G, up, trace = {}, 0.0, 0.0
    with torch.no_grad():
        for t, S, O in F.inverse():
            key = "first" if t == 0 else ("last" if t == T - 1 else "mid")
            G[key] = G.get(key, 0.0) - 0.5 * r * S - 0.5 * w[t] @ w[t].T
            trace += float((torch.diagonal(S) * add.view(T, -1)[t]).sum())
            if O is not None:
                up = up - r * O - w[t] @ w[t + 1].T
    F.inv.clear()
    s = 0.5 * r * P.logdet + sum((g * getattr(P, k)).sum() for k, g in G.items())
    if T > 1:
        s = s + (up * P.upper).sum()
    s.backward()
    jac = p.grad.detach().clone()
    jac[-1] = 0.5 * m * r - 0.5 * r * trace - 0.5 * tau * rss
    return np.float64(-like / (m * r)), -jac.cpu().numpy() / (m * r)


def _on_pattern(case, F, left=None, right=None):
    """Inverse (or the sum of products of left and right) on the pattern of Q,
    row by row in the order of the columns."""
    M, N, T, bc = (case[k] for k in ("M", "N", "T", "bc"))
    c = _Cells(M, N, bc, 3)
    i, j = torch.as_tensor(c.i, device=_dev()), torch.as_tensor(c.j, device=_dev())

    def window(h):
        """(rows x offsets) neighbours in one slice, -1 outside."""
        out = []
        for dy in range(-h, h + 1):
            for dx in range(-h, h + 1):
                a, b = i + dx, j + dy
                if bc == 2:
                    a, b = a % M, b % N
                ok = (a >= 0) & (a < M) & (b >= 0) & (b < N)
                out.append(torch.where(ok, a + b * M, torch.full_like(a, -1)))
        return torch.sort(torch.stack(out, 1), 1)[0]
    w5, w3 = window(2), window(1)
    rows5 = torch.arange(c.Ns, device=_dev())[:, None]
    vals = [[None] * 3 for _ in range(T)]
    if left is None:
        for t, S, O in F.inverse():
            vals[t][1] = S[rows5, w5]
            if O is not None:
                vals[t][2] = O[rows5, w3]
                vals[t + 1][0] = O.T[rows5, w3]
    else:
        a, b = left.view(T, c.Ns, -1), right.view(T, c.Ns, -1)

        def pair(s, t, w):
            acc = torch.zeros(w.shape, dtype=_F64, device=_dev())
            for q in range(w.shape[1]):
                at = w[:, q].clamp(min=0)
                acc[:, q] = 0.5 * ((a[s] * b[t][at]).sum(1) + (b[s] * a[t][at]).sum(1))
            return acc / a.shape[2]
        for t in range(T):
            vals[t][1] = pair(t, t, w5)
            if t:
                vals[t][0] = pair(t, t - 1, w3)
            if t + 1 < T:
                vals[t][2] = pair(t, t + 1, w3)
    out = []
    for t in range(T):
        v = torch.cat([x for x in vals[t] if x is not None], 1)
        k = torch.cat([w for w, x in zip((w3, w5, w3), vals[t]) if x is not None], 1)
        out.append(v[k >= 0])
    return torch.cat(out).cpu()


def _network(case, seed):
    feat, dout, theta = _network_inputs(case, seed)
    M, N, T = case["M"], case["N"], case["T"]
    x = torch.as_tensor(feat, device=_dev()).double().view(T, N, M, 8)
    th = torch.as_tensor(theta, device=_dev()).double().requires_grad_(True)
    off = 0
    for layer, cin in enumerate((8, 32, 32, 32)):
        W = th[off:off + 9 * cin * 32].view(9, cin, 32)
        b = th[off + 9 * cin * 32:off + 9 * cin * 32 + 32]
        off += 9 * cin * 32 + 32
        z = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
        y = b
        for tap in range(9):
            dy, dx = tap // 3, tap % 3
            y = y + z[:, dy:dy + N, dx:dx + M, :] @ W[tap]
        x = y.clamp(min=0) if layer < 3 else y
    out = x.reshape(M * N * T, 32)
    (out[:, :22] * torch.as_tensor(dout, device=_dev()).double()).sum().backward()
    return out.detach().cpu(), th.grad.cpu()


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        return [_loglik(c, seed + 1000 * i) for i, c in enumerate(_members(case))]
    if kind == "network":
        return _network(case, seed)
    if kind in ("loglik", "spatial", "separable"):
        return _loglik(case, seed)
    par, idx, y = _inputs(case, seed)
    n = case["M"] * case["N"] * case["T"]
    add = torch.zeros(n, dtype=_F64, device=_dev())
    if idx is not None:
        add[torch.as_tensor(idx, device=_dev())] = math.exp(par[-1])
    with torch.no_grad():
        P = _Precision(case, torch.tensor(par, device=_dev()))
        F = _Blocks(P, add)
        if kind == "solve":
            return F.solve(torch.as_tensor(_rhs(case, seed), device=_dev())).cpu()
        if kind == "selinv":
            return np.float64(F.logdet), _on_pattern(case, F)
        if kind == "mean":      # the log-determinant there is the incomplete factor's own
            b = torch.as_tensor(_sty(case, idx, y, math.exp(par[-1])), device=_dev())
            return None, F.solve(b[:, None])[:, 0].cpu()
        V = torch.as_tensor(_signs(case, seed), device=_dev()).double()
        U = F.solve(V)
        return U.cpu(), _on_pattern(case, F, U, V)
