"""Drop-in SPDE model classes of the GMRF hot path.

Same names, parameter layouts, method signatures and return conventions as
berild/spdepy ``src/spdepy/spdes``:
  * WhittleMatern2D / WhittleMaternAnisotropic2D / WhittleMaternHa2D
    (``whittle_matern{,_anisotropic,_ha}2D.py``) -- the initial-state model;
  * AdvectionIDiffusion2D / AdvectionDiffusion2D / AdvectionHaDiffusion2D
    (``advection_{i,,ha_}diffusion2D.py``) -- stationary space-time models;
  * VarAdvectionVarDiffusion2D (``var_advection_var_diffusion2D.py``) --
    B-spline advection and anisotropic diffusion fields.
``makeQ`` returns (Q, Q_fac, dQ) with Q a scipy CSC matrix carrying the
reference's sparsity pattern; ``logLike(par, nh1=100, grad=True)`` returns
-loglik/(m r) and its gradient.  All numerics run on the GPU through the
native library (no CPU fallback).  ``logLike`` takes one extra keyword,
``trace``: "exact" (default) contracts with the selected inverse;
"hutchinson" reproduces the reference's stochastic estimator with nh1
Rademacher probes drawn from numpy's global legacy RNG exactly as
``advection_idiffusion2D.py:182`` does.
"""
import ctypes

import numpy as np
from scipy import sparse

from . import _native as nat
from .engine import (Coefficients, Engine, KronEngine, OUT_DGX, OUT_DGY, OUT_H, OUT_H0, OUT_HC, OUT_KAPPA, OUT_KAPPA0,
                     OUT_WIDTH, OUT_WX, OUT_WY, OUT_ADVDIR)
from .plan import _ptr, _stream


# ------------------------------------------------------------- H tensors
def h_tensor(kind, gamma, vx=0.0, vy=0.0):
    """Diffusion tensor and its derivatives w.r.t. (log gamma, vx, vy):
    iso gamma I; ani gamma I + v v^T; ha gamma(cosh|v| I + sinh|v|/|v| [[vx,vy],[vy,-vx]])
    (advection_idiffusion2D.py:97, advection_diffusion2D.py:100,
    advection_ha_diffusion2D.py:109-115 and their gradient blocks)."""
    eye = np.eye(2)
    if kind == "iso":
        return gamma * eye, [gamma * eye]
    if kind == "ani":
        v = np.array([vx, vy])
        ex, ey = np.array([1.0, 0.0]), np.array([0.0, 1.0])
        return (gamma * eye + np.outer(v, v),
                [gamma * eye, np.outer(ex, v) + np.outer(v, ex), np.outer(ey, v) + np.outer(v, ey)])
    a = np.sqrt(vx * vx + vy * vy)
    mv = np.array([[vx, vy], [vy, -vx]])
    ch, sh = (np.exp(a) + np.exp(-a)) / 2, (np.exp(a) - np.exp(-a)) / 2
    H = gamma * (ch * eye + sh / a * mv)
    dvx = gamma / a * (vx * sh * eye + vx / a * (ch - sh / a) * mv + sh * np.array([[1.0, 0.0], [0.0, -1.0]]))
    dvy = gamma / a * (vy * sh * eye + vy / a * (ch - sh / a) * mv + sh * np.array([[0.0, 1.0], [1.0, 0.0]]))
    return H, [H, dvx, dvy]


# ------------------------------------------------------- native stencils
def _torch():
    import torch
    return torch


def stencil_diffusion(shape2, H, hx, hy, bc, variable):
    """Reference slot triplets of the diffusion stencil computed on the GPU
    (replaces AH_new/AH_Row/AH_Col/AH_Val/AH_delete)."""
    torch = _torch()
    M, N = int(shape2[0]), int(shape2[1])
    Ht = torch.as_tensor(np.ascontiguousarray(H, dtype=np.float64).reshape(-1)).cuda()
    row = torch.empty(M * N * 9, dtype=torch.int32, device="cuda")
    col = torch.empty_like(row)
    val = torch.empty(M * N * 9, dtype=torch.float64, device="cuda")
    nat.check(nat.lib().spde_stencil_diffusion(M, N, _ptr(Ht), int(variable), hx, hy, bc, _ptr(row), _ptr(col),
                                               _ptr(val), _stream(torch)))
    return row.cpu().numpy(), col.cpu().numpy(), val.cpu().numpy()


def stencil_advection(shape2, G, hx, hy, diff, bc, variable, dG=None):
    """Reference slot triplets of the upwind stencil computed on the GPU
    (replaces Aw_new/Aw_Row/Aw_Col/Aw_Val/Aw_delete)."""
    torch = _torch()
    M, N = int(shape2[0]), int(shape2[1])
    Gt = torch.as_tensor(np.ascontiguousarray(G, dtype=np.float64).reshape(-1)).cuda()
    dGt = None if dG is None else torch.as_tensor(np.ascontiguousarray(dG, dtype=np.float64).reshape(-1)).cuda()
    row = torch.empty(M * N * 5, dtype=torch.int32, device="cuda")
    col = torch.empty_like(row)
    val = torch.empty(M * N * 5, dtype=torch.float64, device="cuda")
    nat.check(nat.lib().spde_stencil_advection(M, N, _ptr(Gt), _ptr(dGt), int(variable), hx, hy, diff, bc,
                                               _ptr(row), _ptr(col), _ptr(val), _stream(torch)))
    return row.cpu().numpy(), col.cpu().numpy(), val.cpu().numpy()


def _triplets_csc(row, col, val, n, nan_to_zero=False):
    keep = row != n
    v = val[keep].copy()
    if nan_to_zero:
        v[np.isnan(v)] = 0.0
    return sparse.csc_matrix((v, (row[keep], col[keep])), shape=(n, n))


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


class _StencilMixin:
    def _obs_cols(self):
        """The observed cell of each row of S (one entry per row), kept while
        S is the same object."""
        cached = getattr(self, "_obs_cache", None)
        if cached is not None and cached[0] is self.S:
            return cached[1]
        S = self.S.tocsr()
        if np.any(np.diff(S.indptr) != 1):
            raise ValueError("observation matrix must have one entry per row")
        cols = S.indices.astype(np.int64)
        self._obs_cache = (self.S, cols)
        return cols

    def Ah(self, Hs):
        shp = self.grid.shape
        n = int(shp[0] * shp[1])
        Hs = np.asarray(Hs, dtype=np.float64)
        variable = Hs.size != 4
        return _triplets_csc(*stencil_diffusion(shp, Hs, self.grid.hx, self.grid.hy, self.bc, variable), n)

    def Aw(self, ws, dws=None, diff=3):
        shp = self.grid.shape
        n = int(shp[0] * shp[1])
        ws = np.asarray(ws, dtype=np.float64)
        variable = ws.size != 2
        return _triplets_csc(*stencil_advection(shp, ws, self.grid.hx, self.grid.hy, diff, self.bc, variable,
                                                dws), n, nan_to_zero=variable)


# -------------------------------------------------------- factor object
class Factor:
    """Device-resident Cholesky factor with the CHOLMOD Factor calls the
    reference uses (``logdet``, ``solve_A``, ``solve_Lt``, ``apply_Pt``).
    P is this library's nested-dissection permutation.  If the plan's slot
    was reused by a later factorisation the factor is recomputed from the
    stored values first."""

    def __init__(self, engine, slot, qval, diag_add=None):
        self.engine, self.slot, self.qval, self.diag_add = engine, slot, qval, diag_add
        self._logdet = None

    def _ensure(self):
        plan = self.engine.plan
        if plan.slot_owner.get(self.slot) is not self:
            self._logdet = plan.factor(self.slot, self.qval, self.diag_add, owner=self)

    def logdet(self):
        self._ensure()
        return self._logdet

    def selinv(self):
        """Q^-1 on the structural pattern (device tensor, structural order)."""
        self._ensure()
        return self.engine.plan.selinv(self.slot)

    def _solve(self, b, mode):
        torch = _torch()
        self._ensure()
        arr = np.asarray(b, dtype=np.float64)
        one = arr.ndim == 1
        x = self.engine.plan.solve(self.slot, torch.as_tensor(arr.reshape(arr.shape[0], -1)).cuda(), mode,
                                   overwrite=True)
        out = x.cpu().numpy()
        return out.reshape(-1) if one else out

    def solve_A(self, b):
        return self._solve(b, nat.SOLVE_A)

    def solve_L(self, b, use_LDLt_decomposition=False):
        """L^-1 b with b in elimination order (CHOLMOD's solve_L)."""
        return self._solve(b, nat.SOLVE_L_NOPERM)

    def solve_Lt(self, b, use_LDLt_decomposition=False):
        """L^-T b, the result in elimination order (CHOLMOD's solve_Lt)."""
        return self._solve(b, nat.SOLVE_LT_NOPERM)

    def apply_P(self, b):
        """P b: natural order -> elimination order."""
        return self._solve(b, nat.SOLVE_P)

    def apply_Pt(self, b):
        """P^T b: elimination order -> natural order."""
        return self._solve(b, nat.SOLVE_PT)

    def pt_solve_Lt(self, b):
        """P^T L^-T b in one call (apply_Pt(solve_Lt(b)) without the round trip)."""
        return self._solve(b, nat.SOLVE_LT)

    def solve_L_p(self, b):
        """L^-1 P b in one call (solve_L(apply_P(b)))."""
        return self._solve(b, nat.SOLVE_L)


class _SpatialGeom:
    """Geometry of a spatial grid as the coefficient block expects it (a
    unit time step; only the initial-state block A0 is used)."""

    def __init__(self, g):
        self.hx, self.hy, self.V, self.dt = g.hx, g.hy, g.V, 1.0


# --------------------------------------------------------- spatial model
class _WhittleMaternBase(_StencilMixin):
    kind = "iso"

    def __init__(self, grid, par=None, bc=3):
        self.grid, self.bc = grid, bc
        self.Q = None
        self.Q_fac = None
        self.data = None
        self.r = None
        self.S = None
        if par is None:
            self.setPars(self._default())
        else:
            self.setQ(par=par)

    def _default(self):
        return np.array([-1, -1, np.log(100)] if self.kind == "iso" else [-1, -1, 0.1, 0.1, np.log(100)],
                        dtype=np.float64)

    def getPars(self, *args, **kwargs):
        return np.array(self.par, dtype=np.float64)

    def setPars(self, par):
        self.par = np.array(par, dtype=np.float64)
        self.kappa, self.gamma = self.par[0], self.par[1]
        if self.kind != "iso":
            self.vx, self.vy = self.par[2], self.par[3]
        self.tau = self.par[-1]
        self.sigma = np.log(np.sqrt(1 / np.exp(self.tau)))

    def nself(self):
        return 3 if self.kind == "iso" else 5

    def h0(self, par):
        """(kappa0, H0, [dH0/dlog gamma, dH0/dvx, dH0/dvy])."""
        vx, vy = (par[2], par[3]) if self.kind != "iso" else (0.0, 0.0)
        H, dH = h_tensor(self.kind, np.exp(par[1]), vx, vy)
        return np.exp(par[0]), H, dH

    def initFit(self, data, **kwargs):
        assert data.shape[0] <= self.grid.Ns
        self.data = data
        self.r = data.shape[1] if data.ndim == 2 else 1
        self.S = self.grid.getS(idxs=kwargs.get("idx"))
        return self._default()

    def setQ(self, par=None, S=None):
        if par is None:
            par = self.getPars()
        else:
            self.setPars(par)
        self.Q, self.Q_fac, _ = self.makeQ(par=par, grad=False)
        self.S = self.grid.getS()

    def makeQ(self, par, grad=True):
        """Q0 = A0^T iDv A0, A0 = Dv kappa - A_H(H) (whittle_matern2D.py:59-85),
        assembled on the GPU, with its device Cholesky factor (the reference
        returns cholesky(Q), :72); dQ as explicit matrices when grad."""
        par = np.asarray(par, dtype=np.float64)
        eng = self._engine()
        qval = eng.assemble(self._coeffs(par))
        Q = eng.to_scipy(qval)
        self._last_qval = qval
        fac = Factor(eng, 0, qval)
        if not grad:
            return Q, fac, None
        g = self.grid
        kappa, H, dH = self.h0(par)
        Dk = kappa * sparse.eye(g.Ns)
        A = g.Dv @ Dk - self.Ah(H)
        dQ = []
        dA = (g.Dv @ Dk).tocsc()
        dQ.append(dA.T @ g.iDv @ A + A.T @ g.iDv @ dA)
        for d in dH:
            dA = -self.Ah(d)
            dQ.append(dA.T @ g.iDv @ A + A.T @ g.iDv @ dA)
        return Q, fac, dQ

    # ---------------------------------------------------- log-likelihood
    def _engine(self):
        if getattr(self, "_eng", None) is None:
            self._eng = Engine(self.grid, self.bc)
        return self._eng

    def _coeffs(self, par):
        kappa, H, _ = self.h0(par)
        g = self.grid
        c = Coefficients(_SpatialGeom(g), variable=False, kappa=1.0, H=np.eye(2), G=(0.0, 0.0), sigma=1.0,
                         kappa0=kappa, H0=H)
        return c


    def logLike(self, par, nh1=100, grad=True, trace="exact"):
        """whittle_matern2D.py:90-126: -loglik/(m r) and its gradient for
        par = [log kappa, log gamma, (vx, vy,) log tau].  trace="exact" uses
        the selected inverses of Q and Q_c; "hutchinson" the reference's
        estimator with the same numpy probe stream (:103)."""
        par = np.asarray(par, dtype=np.float64)
        eng = self._engine()
        coeffs = self._coeffs(par)
        probes = None
        if grad and trace == "hutchinson":
            probes = (2 * np.random.randint(1, 3, self.grid.n * nh1) - 3).reshape(self.grid.n, nh1)
        like, parts = eng.loglik(coeffs, self._obs_cols(), self.data, par[-1], grad=grad, trace=trace,
                                 probes=probes, logdet="factor")
        if not grad:
            return like
        colsum = parts["colsum"]
        kappa, _, dH = self.h0(par)
        g = [kappa * colsum[OUT_KAPPA0]]
        g += [float(np.dot(colsum[OUT_H0:OUT_H0 + 4], d.reshape(4))) for d in dH]
        g += [parts["g_tau"]]
        m, r = parts["m"], parts["r"]
        return like, -np.array(g) / (m * r)

    def print(self, par):
        s = "| κ = %2.2f, γ = %2.2f" % (np.exp(par[0]), np.exp(par[1]))
        if self.kind != "iso":
            s += ", vx = %2.2f, vy = %2.2f" % (par[2], par[3])
        return s + ",τ = %2.2f" % np.exp(par[-1])


class WhittleMatern2D(_WhittleMaternBase):
    kind = "iso"


class WhittleMaternAnisotropic2D(_WhittleMaternBase):
    kind = "ani"


class WhittleMaternHa2D(_WhittleMaternBase):
    kind = "ha"


# ------------------------------------------- variable Whittle-Matern models
class _VarWhittleMaternBase(_StencilMixin):
    """Spatial Matern models with B-spline fields (var_whittle_matern2D.py,
    var_whittle_matern_anisotropic2D.py, var_whittle_matern_ha2D.py):
    Q = A^T iDv A, A = Dv Dk - A_H(H) with the variable diffusion stencil,
    kappa = exp(bs c_kappa), gamma = exp(bsH c_gamma) on the faces and per face
    H = gamma I (iso), gamma I + v v^T (ani), gamma expm([[vx, vy], [vy, -vx]])
    (ha).  par = [c_kappa, c_gamma, (c_vx, c_vy,) log tau] (Np = Nbs^2 each;
    the reference's ha class fixes Nbs = 3).  On the GPU, A0 of the one-slice
    plan is assembled from the fields (spde_coeffs.a0_variable)."""
    kind = "iso"
    label = "isotropic"

    def __init__(self, grid, par=None, bc=3):
        self.grid, self.bc = grid, bc
        self.type = "var-whittle-matern-%s-2D-bc%d" % (self.label, bc)
        self.Np = grid.Nbs2
        self.Q = self.Q_fac = self.data = self.r = self.S = None
        self._eng = None
        if par is None:
            self.setPars(self._default())
        else:
            self.setQ(par=par)

    def _nfield(self):
        return 2 if self.kind == "iso" else 4

    def _default(self):
        Np = self.Np
        v = [[-1.0] * Np, [-1.0] * Np] + ([[0.1] * Np, [0.1] * Np] if self.kind != "iso" else [])
        return np.hstack(v + [[np.log(100)]]).astype(np.float64)

    def getPars(self, *args, **kwargs):
        return np.hstack([self.coef, [self.tau]]).astype(np.float64)

    def setPars(self, par):
        par = np.asarray(par, dtype=np.float64)
        self.coef = par[:-1].copy()
        self.kappa, self.gamma = par[:self.Np], par[self.Np:2 * self.Np]
        self.tau = par[-1]
        self.sigma = np.log(np.sqrt(1 / np.exp(self.tau)))

    def initFit(self, data, **kwargs):
        assert data.shape[0] <= self.grid.Ns
        self.data = data
        self.r = data.shape[1] if data.ndim == 2 else 1
        self.S = self.grid.getS(idxs=kwargs.get("idx"))
        return self._default()


    def _engine(self):
        if self._eng is None:
            self._eng = Engine(self.grid, self.bc)
        return self._eng

    # fields --------------------------------------------------------------
    def _host_fields(self, par):
        """kappa[Ns], H[Ns,4,2,2] and dH/d(log gamma, vx, vy) per face."""
        g, Np = self.grid, self.Np
        kappa = np.exp(g.bs @ par[:Np])
        gam = np.exp(g.bsH @ par[Np:2 * Np])
        I = np.eye(2)
        if self.kind != "ha":
            H = gam[:, :, None, None] * I
            d = [H.copy()]
            if self.kind == "ani":
                v = np.stack([g.bsH @ par[2 * Np:3 * Np], g.bsH @ par[3 * Np:4 * Np]], axis=2)
                H = H + v[:, :, :, None] * v[:, :, None, :]
                for a in range(2):
                    e = np.zeros_like(v)
                    e[:, :, a] = 1.0
                    d.append(v[:, :, :, None] * e[:, :, None, :] + e[:, :, :, None] * v[:, :, None, :])
            return kappa, H, d
        vx, vy = g.bsH @ par[2 * Np:3 * Np], g.bsH @ par[3 * Np:4 * Np]
        a = np.sqrt(vx ** 2 + vy ** 2)
        mV = np.zeros(vx.shape + (2, 2))
        mV[..., 0, 0], mV[..., 0, 1], mV[..., 1, 0], mV[..., 1, 1] = vx, vy, vy, -vx
        ch, sh = np.cosh(a), np.sinh(a)
        H = (gam * ch)[..., None, None] * I + (gam * sh / a)[..., None, None] * mV
        Dx = np.zeros_like(mV)
        Dx[..., 0, 0], Dx[..., 1, 1] = 1.0, -1.0
        Dy = np.zeros_like(mV)
        Dy[..., 0, 1], Dy[..., 1, 0] = 1.0, 1.0
        d = [H.copy()]
        for u, D in ((vx, Dx), (vy, Dy)):
            d.append((gam * sh * u / a)[..., None, None] * I + (gam * (ch * u - sh * u / a) / a ** 2)[..., None, None] * mV
                     + (gam * sh / a)[..., None, None] * D)
        return kappa, H, d

    def _dev_bases(self):
        if self.kind == "ha" or self.grid.Ne:
            return None
        if getattr(self, "_bases", None) is None:
            import torch
            g = self.grid
            bs = torch.as_tensor(np.ascontiguousarray(g.bs, dtype=np.float64)).cuda()
            bsH = torch.as_tensor(np.ascontiguousarray(g.bsH, dtype=np.float64)).cuda()
            wd = ctypes.c_int64()
            nat.check(nat.lib().spde_fields_contract_workspace(g.Ns, self.Np, ctypes.byref(wd)))
            work = torch.empty(int(wd.value), dtype=torch.float64, device="cuda")
            self._bases = ((bs, bsH, bsH), work)   # no advection faces: zero coefficients
        return self._bases

    def _coeffs(self, par):
        geom = _SpatialGeom(self.grid)
        bases = self._dev_bases()
        if bases is None:
            kappa, H, d = self._host_fields(par)
            self._hfields = (kappa, H, d)
            return Coefficients(geom, variable=True, kappa=kappa, H=H, G=np.zeros((self.grid.Ns, 4)), sigma=1.0,
                                kappa0=1.0, H0=np.eye(2), a0_variable=True)
        import torch
        (bs, bsH, bsA), _ = bases
        Ns, nb = self.grid.Ns, self.Np
        c6 = np.zeros(6 * nb)
        c6[:self._nfield() * nb] = par[:self._nfield() * nb]
        coef = torch.as_tensor(c6).cuda()
        kappa = torch.empty(Ns, dtype=torch.float64, device="cuda")
        H = torch.empty(Ns * 16, dtype=torch.float64, device="cuda")
        G = torch.empty(Ns * 4, dtype=torch.float64, device="cuda")
        fgv = torch.empty(Ns * 12, dtype=torch.float64, device="cuda")
        st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        nat.check(nat.lib().spde_fields_eval(Ns, nb, _p(bs), _p(bsH), _p(bsA), _p(coef), _p(kappa), _p(H), _p(G),
                                             _p(fgv), st))
        self._fields_dev = (kappa, fgv)
        return Coefficients(geom, variable=True, kappa=kappa, H=H, G=G, sigma=1.0, kappa0=1.0, H0=np.eye(2),
                            a0_variable=True)

    def _device_contract(self):
        bases = self._dev_bases()
        if bases is None:
            return None

        def contract(cells):
            import torch
            (bs, bsH, bsA), work = bases
            kappa, fgv = self._fields_dev
            Ns, nb = self.grid.Ns, self.Np
            res = torch.empty(6 * nb + OUT_WIDTH, dtype=torch.float64, device="cuda")
            st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
            nat.check(nat.lib().spde_fields_contract(Ns, nb, _p(bs), _p(bsH), _p(bsA), _p(cells), _p(kappa), _p(fgv),
                                                     _p(work), _p(res), st))
            h = res.cpu().numpy()
            return h[:6 * nb], h[6 * nb:]
        return contract

    # precision and likelihood ------------------------------------------
    def makeQ(self, par, grad=True):
        """Q on the GPU with the reference's scipy pattern; dQ is not
        materialised (logLike contracts it)."""
        par = np.asarray(par, dtype=np.float64)
        eng = self._engine()
        qval = eng.assemble(self._coeffs(par))
        Q = eng.to_scipy(qval)
        self._last_qval = qval
        return Q, Factor(eng, 0, qval), (_LazyDQ(self, par) if grad else None)

    def setQ(self, par=None, S=None, simple=False):
        if par is None:
            par = self.getPars()
        else:
            self.setPars(par)
        if S is not None:
            self.S = S
        self.Q, self.Q_fac, _ = self.makeQ(par=par, grad=False)
        self.S = self.grid.getS()

    def logLike(self, par, nh1=100, grad=True, trace="exact"):
        """var_whittle_matern2D.py:83-130 (and the anisotropic / ha files):
        -loglik/(m r) and its gradient; trace="exact" uses the selected
        inverses of Q and Q_c, "hutchinson" the reference's estimator."""
        par = np.asarray(par, dtype=np.float64)
        eng = self._engine()
        coeffs = self._coeffs(par)
        probes = None
        if grad and trace == "hutchinson":
            probes = (2 * np.random.randint(1, 3, self.grid.n * nh1) - 3).reshape(self.grid.n, nh1)
        like, parts = eng.loglik(coeffs, self._obs_cols(), self.data, par[-1], grad=grad, trace=trace,
                                 probes=probes, logdet="factor", contract=self._device_contract())
        if not grad:
            return like
        g = self._field_grad(parts)
        g.append(parts["g_tau"])
        m, r = parts["m"], parts["r"]
        return like, -np.array(g) / (m * r)

    def _field_grad(self, parts):
        """Contraction of the per-cell A0 adjoints onto the field coefficients."""
        nf, Np = self._nfield(), self.Np
        if "coef_grad" in parts:
            return list(parts["coef_grad"][:nf * Np])
        gr = self.grid
        cells = parts["cells"]
        kappa, H, d = self._hfields
        Hb = cells[:, OUT_H:OUT_H + 16].reshape(-1, 4, 2, 2)
        g = list(gr.bs.T @ (cells[:, OUT_KAPPA] * kappa))
        for dH in d:
            g += list(np.einsum("kfi,kf->i", gr.bsH, (Hb * dH).sum(axis=(2, 3))))
        return g

    def print(self, par):
        Np = self.Np
        s = "| κ = %2.2f, γ = %2.2f" % (np.exp(par[:Np]).mean(), np.exp(par[Np:2 * Np]).mean())
        if self.kind != "iso":
            s += ", vx = %2.2f, vy = %2.2f" % (par[2 * Np:3 * Np].mean(), par[3 * Np:4 * Np].mean())
        return s + ",τ = %2.2f" % np.exp(par[-1])


class VarWhittleMatern2D(_VarWhittleMaternBase):
    kind, label = "iso", "isotropic"


class VarWhittleMaternAnisotropic2D(_VarWhittleMaternBase):
    kind, label = "ani", "anisotropic"


class VarWhittleMaternHa2D(_VarWhittleMaternBase):
    kind, label = "ha", "ha"


# ---------------------------------------------------- space-time models
class _SpaceTimeBase(_StencilMixin):
    """Shared logLike / makeQ plumbing of the space-time models."""

    def _engine(self):
        if getattr(self, "_eng", None) is None:
            self._eng = Engine(self.grid, self.bc)
        return self._eng

    def _mod0_split(self, par):
        """Initial-state parameters carried in par (fitQ0) or the model's own."""
        p0 = self._par_mod0(par)
        src = p0 if p0 is not None else self.mod0.getPars()
        kappa0, H0, dH0 = self.mod0.h0(src)
        return p0, kappa0, H0, dH0

    def initFit(self, data, **kwargs):
        assert data.shape[0] <= self.grid.n
        if kwargs.get("fitQ0") is not None:
            assert type(kwargs.get("fitQ0")) is bool
            self.fitQ0 = kwargs.get("fitQ0")
        x0 = self.mod0.getPars()[:-1] if self.fitQ0 else np.zeros(0)
        par = np.hstack([self._init_self(), x0, [np.log(100)]]).astype(np.float64)
        self.data = data
        self.r = data.shape[1] if data.ndim == 2 else 1
        self.S = self.grid.getS(idxs=kwargs.get("idx"))
        self._obs_idx = kwargs.get("idx")
        return par

    def setQ(self, par=None, S=None):
        if par is None:
            par = self.getPars()
        else:
            self.setPars(par)
        if S is not None:
            self.S = S
        self.Q, self.Q_fac, _ = self.makeQ(par=par, grad=False)
        self.S = self.grid.getS()

    def makeQ(self, par, grad=True):
        par = np.asarray(par, dtype=np.float64)
        eng = self._engine()
        coeffs = self._coeffs(par)
        qval = eng.assemble(coeffs)
        Q = eng.to_scipy(qval)
        fac = Factor(eng, 0, qval)
        self._last_qval = qval
        if not grad:
            return Q, fac, None
        dirs = self._directions(par) if hasattr(self, "_directions") else None
        if dirs is None:
            return Q, fac, _LazyDQ(self, par)
        return Q, fac, _TangentDQ(self, par, coeffs, dirs)

    def _mod0_directions(self, par):
        """dQ of the initial-state parameters carried in par (fitQ0): the
        Whittle-Matern derivatives placed in block (0, 0)
        (advection_idiffusion2D.py:157-162)."""
        p0, kappa0, H0, dH0 = self._mod0_split(par)
        if p0 is None:
            return []
        out = [lambda: _direction(kind=2, dkappa0=kappa0, dH0=np.zeros(4))]
        out += [(lambda d=d: _direction(kind=2, dkappa0=0.0, dH0=d)) for d in dH0]
        return out


    def logLike(self, par, nh1=100, grad=True, trace="exact", logdet="closed", method="exact", **pcg):
        """The reference's logLike (advection_idiffusion2D.py:167-207,
        var_advection_var_diffusion2D.py:201-237).  trace="exact" uses the
        selected inverse of Q_c; logdet="closed" takes log|Q| and its
        gradient from the spatial matrices of Q = F^T D F, logdet="factor"
        factorises Q as the reference does (same values to rounding).
        method="pcg": Q_c is not factorised -- PCG with an IC(0)
        preconditioner, stochastic Lanczos for log|Q_c| and the Hutchinson
        trace (``spdepy_amd.krylov.loglik_pcg``; keyword options pass through);
        method="learned": the same with the learned correction of the
        preconditioner (``spdepy_amd.learned``), falling back to the exact
        Cholesky path when the relative standard error of the value exceeds
        tol_like (default 1e-6; None or inf: no fallback) -- decided right
        after the stochastic log-determinant when a bound on |loglik| already
        shows the tolerance out of reach.  The parts of the last evaluation
        are kept in self.last_parts."""
        par = np.asarray(par, dtype=np.float64)
        if not np.all(np.isfinite(par)):
            raise ValueError("logLike: parameters must be finite (got %s)" % par[~np.isfinite(par)][:4])
        eng = self._engine()
        coeffs = self._coeffs(par)
        if method in ("pcg", "learned"):
            from .krylov import loglik_pcg
            tol_like = pcg.pop("tol_like", 1e-6 if method == "learned" else None)
            if tol_like is not None and not np.isfinite(tol_like):
                tol_like = None
            if method == "learned":
                from .learned import default_preconditioner
                net = pcg.pop("preconditioner", None) or default_preconditioner()
                pcg["correction"] = net.corrector()
            like, parts = loglik_pcg(eng, coeffs, self._obs_cols(), self.data, par[-1], grad=grad,
                                     contract=self._device_contract(), adv_dir=self._adv_dir(), tol_like=tol_like,
                                     **pcg)
            if parts.get("infeasible"):
                parts["like_rel_se"] = 0.5 * parts["r"] * parts["logdet_qc_se"] / parts["like_bound"]
            else:
                # relative standard error of the stochastic log|Q_c| in the value
                parts["like_rel_se"] = 0.5 * parts["r"] * parts["logdet_qc_se"] / abs(parts["like_raw"])
            parts["fallback"] = tol_like is not None and parts["like_rel_se"] > tol_like
            self.last_parts = parts
            if parts["fallback"]:
                # the stated error is missed: the exact Cholesky path decides
                out = self.logLike(par, nh1=nh1, grad=grad, trace="exact", logdet=logdet)
                self.last_parts = dict(parts, fallback=True)
                return out
            if not grad:
                return like
            g = self._contract(par, coeffs, parts)
            return like, -g / (parts["m"] * parts["r"])
        if method != "exact":
            raise ValueError("method must be 'exact', 'pcg' or 'learned'")
        probes = None
        if grad and trace == "hutchinson":
            probes = (2 * np.random.randint(1, 3, self.grid.n * nh1) - 3).reshape(self.grid.n, nh1)
        adv_dir = self._adv_dir()
        if grad and trace == "exact" and logdet == "closed" and adv_dir is None:
            # the whole evaluation behind one library call (spde_loglik_grad)
            from .engine import loglik_fused
            like, parts = loglik_fused(eng, coeffs, self._obs_cols(), self.data, par[-1],
                                       contract=self._device_contract())
        else:
            like, parts = eng.loglik(coeffs, self._obs_cols(), self.data, par[-1], grad=grad, trace=trace,
                                     probes=probes, logdet=logdet, contract=self._device_contract(),
                                     adv_dir=adv_dir)
        self.last_parts = parts
        if not grad:
            return like
        g = self._contract(par, coeffs, parts)
        m, r = parts["m"], parts["r"]
        return like, -g / (m * r)

    def _device_contract(self):
        """Contraction of the per-cell adjoints on the device, or None (the
        host contracts them)."""
        return None

    def _adv_dir(self):
        """Advection direction whose scaling is a parameter (cov-advection
        models), or None."""
        return None

    def _mod0_grad(self, par, parts, dH0, kappa0):
        colsum = parts["colsum"]
        if self._par_mod0(par) is None:
            return []
        hbar = colsum[OUT_H0:OUT_H0 + 4]
        out = [kappa0 * colsum[OUT_KAPPA0]]
        out += [float(np.dot(hbar, d.reshape(4))) for d in dH0]
        return out


class _StationaryAdvDiff(_SpaceTimeBase):
    kind = "iso"

    def __init__(self, grid, mod0, par=None, bc=3):
        self.grid, self.mod0, self.bc = grid, mod0, bc
        self.type = {"iso": "advection-idiffusion-2D-bc%d", "ani": "advection-diffusion-2D-bc%d",
                     "ha": "advection-ha-diffusion-2D-bc%d"}[self.kind] % bc
        self.Q = self.Q_fac = self.data = self.r = self.S = None
        self.fitQ0 = True
        self._eng = None
        if par is None:
            self.setPars(np.hstack([self._init_self(), [np.log(100)]]))
        else:
            self.setQ(par=par)

    def _nself(self):
        return 5 if self.kind == "iso" else 7

    def _init_self(self):
        return [-1, -1, 0.1, 0.1, 0] if self.kind == "iso" else [-1, -1, 0.1, 0.1, 0.1, 0.1, 0]

    def _par_mod0(self, par):
        k = self._nself()
        return par[k:] if par.size > k + 1 else None

    def getPars(self, onlySelf=True):
        own = [self.kappa, self.gamma] + ([] if self.kind == "iso" else [self.vx, self.vy]) + \
              [self.wx, self.wy, self.sigma]
        if onlySelf:
            return np.hstack(own + [self.tau]).astype(np.float64)
        return np.hstack(own + [self.mod0.getPars()[:-1], self.tau]).astype(np.float64)

    def setPars(self, par):
        par = np.array(par, dtype=np.float64)
        self.kappa, self.gamma = par[0], par[1]
        if self.kind == "iso":
            self.wx, self.wy, self.sigma = par[2], par[3], par[4]
        else:
            self.vx, self.vy, self.wx, self.wy, self.sigma = par[2], par[3], par[4], par[5], par[6]
        if par.size > self._nself() + 1:
            self.mod0.setPars(par[self._nself():])
        self.tau = par[-1]

    def _split(self, par):
        if self.kind == "iso":
            return par[0], par[1], 0.0, 0.0, par[2:4], par[4]
        return par[0], par[1], par[2], par[3], par[4:6], par[6]

    def _coeffs(self, par):
        kap, gam, vx, vy, ws, sig = self._split(par)
        H, _ = h_tensor(self.kind, np.exp(gam), vx, vy)
        _, kappa0, H0, _ = self._mod0_split(par)
        return Coefficients(self.grid, variable=False, kappa=np.exp(kap), H=H, G=ws, sigma=np.exp(sig),
                            kappa0=kappa0, H0=H0)

    def _directions(self, par):
        """Directions of [log kappa, log gamma, (vx, vy), wx, wy, log sigma,
        (mod0...)]: dA = dt V kappa I and dQs = 2 V kappa^2 for log kappa;
        -dt A_H(dH) for the diffusion parameters; the constant advection
        derivative stencils Aw(., diff = 1, 2) (Acw_2D_b*.cpp) for wx, wy."""
        kap, gam, vx, vy, ws, sig = self._split(np.asarray(par, dtype=np.float64))
        _, dH = h_tensor(self.kind, np.exp(gam), vx, vy)
        out = [lambda: _direction(dkappa_c=np.exp(kap))]
        out += [(lambda d=d: _direction(dH_c=d)) for d in dH]
        out += [lambda: _direction(adv_diff=1), lambda: _direction(adv_diff=2), lambda: _direction(kind=1)]
        return out + self._mod0_directions(par)

    def _contract(self, par, coeffs, parts):
        kap, gam, vx, vy, ws, sig = self._split(par)
        _, dH = h_tensor(self.kind, np.exp(gam), vx, vy)
        _, kappa0, H0, dH0 = self._mod0_split(par)
        colsum = parts["colsum"]
        hbar = colsum[OUT_HC:OUT_HC + 4]
        g = [np.exp(kap) * colsum[OUT_KAPPA]]
        g += [float(np.dot(hbar, d.reshape(4))) for d in dH]
        g += [colsum[OUT_WX], colsum[OUT_WY], parts["g_sigma"]]
        g += self._mod0_grad(par, parts, dH0, kappa0)
        g += [parts["g_tau"]]
        return np.array(g, dtype=np.float64)

    def print(self, par):
        kap, gam, vx, vy, ws, sig = self._split(np.asarray(par))
        s = "| κ = %2.2f, γ = %2.2f" % (np.exp(kap), np.exp(gam))
        if self.kind != "iso":
            s += ", vx = %2.2f, vy = %2.2f" % (vx, vy)
        return s + ", wx = %2.2f, wy = %2.2f, σ = %2.2f, τ = %2.2f" % (ws[0], ws[1], np.exp(sig),
                                                                          np.exp(par[-1]))


class AdvectionIDiffusion2D(_StationaryAdvDiff):
    """Params [log kappa, log gamma, wx, wy, log sigma, (mod0...), log tau]."""
    kind = "iso"


class AdvectionDiffusion2D(_StationaryAdvDiff):
    """Params [log kappa, log gamma, vx, vy, wx, wy, log sigma, (mod0...), log tau]."""
    kind = "ani"


class AdvectionHaDiffusion2D(_StationaryAdvDiff):
    kind = "ha"


class VarAdvectionVarDiffusion2D(_SpaceTimeBase):
    """B-spline fields: par = [c_kappa, c_gamma, c_vx, c_vy, c_wx, c_wy (Np each),
    log sigma, (mod0...), log tau] (var_advection_var_diffusion2D.py:28-45)."""

    def __init__(self, grid, mod0, par=None, bc=3):
        self.grid, self.mod0, self.bc = grid, mod0, bc
        self.type = "var-advection-var-diffusion-2D-bc%d" % bc
        self.Np = grid.Nbs2
        self.Q = self.Q_fac = self.data = self.r = self.S = None
        self.fitQ0 = True
        self._eng = None
        if par is None:
            self.setPars(np.hstack([self._init_self(), [np.log(100)]]))
        else:
            self.setQ(par=par)

    def _init_self(self):
        Np = self.Np
        return np.hstack([[-1] * Np, [-1] * Np, [0.1] * Np * 2, [0.1] * Np * 2, [0]])

    def _par_mod0(self, par):
        k = self.Np * 6 + 1
        return par[k:] if par.size > k + 1 else None

    def getPars(self, onlySelf=True):
        own = [self.kappa, self.gamma, self.vx, self.vy, self.wx, self.wy, self.sigma]
        if onlySelf:
            return np.hstack(own + [self.tau]).astype(np.float64)
        return np.hstack(own + [self.mod0.getPars()[:-1], self.tau]).astype(np.float64)

    def setPars(self, par):
        par = np.array(par, dtype=np.float64)
        Np = self.Np
        self.kappa, self.gamma = par[0:Np], par[Np:2 * Np]
        self.vx, self.vy = par[2 * Np:3 * Np], par[3 * Np:4 * Np]
        self.wx, self.wy = par[4 * Np:5 * Np], par[5 * Np:6 * Np]
        self.sigma = par[6 * Np]
        if par.size > 6 * Np + 2:
            self.mod0.setPars(par[6 * Np + 1:])
        self.tau = par[-1]

    def fields(self, par):
        g, Np = self.grid, self.Np
        kappa = np.exp(g.bs @ par[:Np])
        gamma = np.exp(g.bsH @ par[Np:2 * Np])
        vx = g.bsH @ par[2 * Np:3 * Np]
        vy = g.bsH @ par[3 * Np:4 * Np]
        ws = g.evalAdv(par[4 * Np:6 * Np])
        return kappa, gamma, vx, vy, ws

    def _dev_bases(self):
        """Bases on the device (None on extended grids, whose advection
        faces pass through the host border extrapolation)."""
        g = self.grid
        if g.isExtended:
            return None
        if getattr(self, "_bases", None) is None:
            import torch
            from . import _native as nat
            dev = [torch.as_tensor(np.ascontiguousarray(b, dtype=np.float64)).cuda() for b in (g.bs, g.bsH, g.bsA)]
            wd = ctypes.c_int64()
            nat.check(nat.lib().spde_fields_contract_workspace(g.Ns, self.Np, ctypes.byref(wd)))
            work = torch.empty(int(wd.value), dtype=torch.float64, device="cuda")
            self._bases = (dev, work)
        return self._bases

    def _coeffs(self, par):
        _, kappa0, H0, _ = self._mod0_split(par)
        bases = self._dev_bases()
        if bases is not None:
            import torch
            from . import _native as nat
            (bs, bsH, bsA), _ = bases
            Ns, nb = self.grid.Ns, self.Np
            coef = torch.as_tensor(np.ascontiguousarray(par[:6 * nb], dtype=np.float64)).cuda()
            kappa = torch.empty(Ns, dtype=torch.float64, device="cuda")
            H = torch.empty(Ns * 16, dtype=torch.float64, device="cuda")
            G = torch.empty(Ns * 4, dtype=torch.float64, device="cuda")
            fgv = torch.empty(Ns * 12, dtype=torch.float64, device="cuda")
            st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
            nat.check(nat.lib().spde_fields_eval(Ns, nb, _p(bs), _p(bsH), _p(bsA), _p(coef), _p(kappa), _p(H),
                                                 _p(G), _p(fgv), st))
            self._fields_dev = (kappa, fgv, coef)
            return Coefficients(self.grid, variable=True, kappa=kappa, H=H, G=G, sigma=np.exp(par[6 * self.Np]),
                                kappa0=kappa0, H0=H0)
        kappa, gamma, vx, vy, ws = self.fields(par)
        H = np.empty((self.grid.Ns, 4, 2, 2))
        H[:, :, 0, 0] = gamma + vx * vx
        H[:, :, 0, 1] = vx * vy
        H[:, :, 1, 0] = vy * vx
        H[:, :, 1, 1] = gamma + vy * vy
        self._fields = (kappa, gamma, vx, vy)
        return Coefficients(self.grid, variable=True, kappa=kappa, H=H, G=ws, sigma=np.exp(par[6 * self.Np]),
                            kappa0=kappa0, H0=H0)

    def _device_contract(self):
        bases = self._dev_bases()
        if bases is None:
            return None

        def contract(cells):
            import torch
            from . import _native as nat
            (bs, bsH, bsA), work = bases
            kappa, fgv, _ = self._fields_dev
            Ns, nb = self.grid.Ns, self.Np
            res = torch.empty(6 * nb + OUT_WIDTH, dtype=torch.float64, device="cuda")
            st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
            nat.check(nat.lib().spde_fields_contract(Ns, nb, _p(bs), _p(bsH), _p(bsA), _p(cells), _p(kappa), _p(fgv),
                                                     _p(work), _p(res), st))
            h = res.cpu().numpy()
            return h[:6 * nb], h[6 * nb:]
        return contract

    def _directions(self, par):
        """Directions of the reference's dQ loop (var_advection_var_diffusion2D.py:
        131-183): for coefficient i of kappa, dkappa = bs_i kappa; of gamma,
        dH = I bsH_i gamma per face; of vx / vy, dH = v dv^T + dv v^T with dv
        the face basis on one component; of wx / wy, the variable advection
        derivative stencil with the face direction evalAdv(e_i); then log sigma
        and the initial-state parameters."""
        g, Np = self.grid, self.Np
        par = np.asarray(par, dtype=np.float64)
        kappa, gamma, vx, vy, ws = self.fields(par)
        vv = np.stack([vx, vy], axis=2)
        out = [(lambda i=i: _direction(dkappa=g.bs[:, i] * kappa)) for i in range(Np)]

        def dh_gamma(i):
            d = np.zeros((g.Ns, 4, 2, 2))
            d[:, :, 0, 0] = d[:, :, 1, 1] = g.bsH[:, :, i] * gamma
            return _direction(dH=d)

        def dh_v(comp, i):
            b = g.bsH[:, :, i]
            z = np.zeros_like(b)
            dv = np.stack([b, z] if comp == 0 else [z, b], axis=2)
            d = vv[:, :, :, None] * dv[:, :, None, :] + dv[:, :, :, None] * vv[:, :, None, :]
            return _direction(dH=d)

        def dw(i):
            e = np.zeros(2 * Np)
            e[i] = 1.0
            return _direction(dG=g.evalAdv(e), adv_diff=1 if i < Np else 2)
        out += [(lambda i=i: dh_gamma(i)) for i in range(Np)]
        out += [(lambda c=c, i=i: dh_v(c, i)) for c in (0, 1) for i in range(Np)]
        out += [(lambda i=i: dw(i)) for i in range(2 * Np)]
        out.append(lambda: _direction(kind=1))
        return out + self._mod0_directions(par)

    def _contract(self, par, coeffs, parts):
        g, Np = self.grid, self.Np
        _, kappa0, H0, dH0 = self._mod0_split(par)
        if "coef_grad" in parts:
            out = [parts["coef_grad"], [parts["g_sigma"]], self._mod0_grad(par, parts, dH0, kappa0), [parts["g_tau"]]]
            return np.hstack(out).astype(np.float64)
        kappa, gamma, vx, vy = self._fields
        cells = parts["cells"]
        Hb = cells[:, OUT_H:OUT_H + 16].reshape(-1, 4, 2, 2)
        out = [g.bs.T @ (cells[:, OUT_KAPPA] * kappa)]
        out.append(np.einsum("kfi,kf->i", g.bsH, (Hb[:, :, 0, 0] + Hb[:, :, 1, 1]) * gamma))
        cross = Hb[:, :, 0, 1] + Hb[:, :, 1, 0]
        out.append(np.einsum("kfi,kf->i", g.bsH, 2 * vx * Hb[:, :, 0, 0] + vy * cross))
        out.append(np.einsum("kfi,kf->i", g.bsH, 2 * vy * Hb[:, :, 1, 1] + vx * cross))
        wx_bar = cells[:, OUT_DGX:OUT_DGX + 4]
        wy_bar = cells[:, OUT_DGY:OUT_DGY + 4]
        if g.isExtended:
            Ae = g.ext_map()
            wx_bar, wy_bar = Ae.T @ wx_bar, Ae.T @ wy_bar
        out.append(g.bsA[:, 0, :].T @ wx_bar[:, 0] + g.bsA[:, 2, :].T @ wx_bar[:, 2])
        out.append(g.bsA[:, 1, :].T @ wy_bar[:, 1] + g.bsA[:, 3, :].T @ wy_bar[:, 3])
        out.append([parts["g_sigma"]])
        out.append(self._mod0_grad(par, parts, dH0, kappa0))
        out.append([parts["g_tau"]])
        return np.hstack(out).astype(np.float64)

    def print(self, par):
        Np = self.Np
        return ("| κ = %2.2f, γ = %2.2f, vx = %2.2f, vy = %2.2f, wx = %2.2f, wy = %2.2f, "
                "σ = %2.2f, τ = %2.2f" % (np.exp(par[:Np]).mean(), np.exp(par[Np:2 * Np]).mean(),
                                                     par[2 * Np:3 * Np].mean(), par[3 * Np:4 * Np].mean(),
                                                     par[4 * Np:5 * Np].mean(), par[5 * Np:6 * Np].mean(),
                                                     np.exp(par[6 * Np]), np.exp(par[-1])))


class _FieldAdvDiff(_SpaceTimeBase):
    """Space-time families with some coefficients as B-spline fields and the
    rest constant (advection_var_{i,,ha_}diffusion2D.py: B-spline kappa and
    diffusion, constant advection; var_advection_{i,,ha_}diffusion2D.py:
    constant kappa and diffusion, B-spline advection;
    var_advection_var_{i,ha_}diffusion2D.py: all B-spline).  par = [kappa
    block, gamma block, (vx, vy blocks,) w block, log sigma, (mod0...),
    log tau], a block being Np = Nbs^2 coefficients for a field (2 Np for w)
    or one log-scalar (two scalars for w) for a constant; the reference's
    files fix Nbs = 3.  The per-cell adjoints are contracted on the host."""
    kind, dvar, gvar, name = "iso", True, False, ""
    w0 = 0.1    # initial advection coefficients

    def __init__(self, grid, mod0, par=None, bc=3):
        self.grid, self.mod0, self.bc = grid, mod0, bc
        self.type = "%s-bc%d" % (self.name, bc)
        self.Np = grid.Nbs2
        self.Q = self.Q_fac = self.data = self.r = self.S = None
        self.fitQ0 = True
        self._eng = None
        if par is None:
            self.setPars(np.hstack([self._init_self(), [np.log(100)]]))
        else:
            self.setQ(par=par)

    def _sizes(self):
        nd = self.Np if self.dvar else 1
        return nd, (1 if self.kind == "iso" else 3), (2 * self.Np if self.gvar else 2)

    def _nself(self):
        nd, nh, nw = self._sizes()
        return nd * (1 + nh) + nw + 1

    def _init_self(self):
        nd, nh, nw = self._sizes()
        v = [[-1.0] * nd, [-1.0] * nd] + [[0.1] * nd] * (nh - 1) + [[self.w0] * nw, [0.0]]
        return np.hstack(v)

    def _split(self, par):
        nd, nh, nw = self._sizes()
        blocks, k = [], 0
        for size in [nd] * (1 + nh) + [nw]:
            blocks.append(np.asarray(par[k:k + size], dtype=np.float64))
            k += size
        return blocks, par[k]

    def _par_mod0(self, par):
        k = self._nself()
        return par[k:] if par.size > k + 1 else None

    def getPars(self, onlySelf=True):
        own = np.asarray(self.own, dtype=np.float64)
        if onlySelf:
            return np.hstack([own, [self.tau]])
        return np.hstack([own, self.mod0.getPars()[:-1], [self.tau]])

    def setPars(self, par):
        par = np.asarray(par, dtype=np.float64)
        k = self._nself()
        self.own = par[:k].copy()
        self.sigma = par[k - 1]
        if par.size > k + 1:
            self.mod0.setPars(par[k:])
        self.tau = par[-1]

    def _face_fields(self, blocks):
        """Per-face H[Ns,4,2,2] and its derivatives in (log gamma, vx, vy)."""
        g = self.grid
        gam = np.exp(g.bsH @ blocks[1])
        I = np.eye(2)
        H = gam[:, :, None, None] * I
        if self.kind == "iso":
            return H, [H.copy()]
        vx, vy = g.bsH @ blocks[2], g.bsH @ blocks[3]
        if self.kind == "ani":
            v = np.stack([vx, vy], axis=2)
            d = [H.copy()]
            for a in range(2):
                e = np.zeros_like(v)
                e[:, :, a] = 1.0
                d.append(v[:, :, :, None] * e[:, :, None, :] + e[:, :, :, None] * v[:, :, None, :])
            return H + v[:, :, :, None] * v[:, :, None, :], d
        a = np.sqrt(vx ** 2 + vy ** 2)
        mV = np.zeros(vx.shape + (2, 2))
        mV[..., 0, 0], mV[..., 0, 1], mV[..., 1, 0], mV[..., 1, 1] = vx, vy, vy, -vx
        ch, sh = np.cosh(a), np.sinh(a)
        H = (gam * ch)[..., None, None] * I + (gam * sh / a)[..., None, None] * mV
        Dx = np.zeros_like(mV)
        Dx[..., 0, 0], Dx[..., 1, 1] = 1.0, -1.0
        Dy = np.zeros_like(mV)
        Dy[..., 0, 1], Dy[..., 1, 0] = 1.0, 1.0
        d = [H.copy()]
        for u, D in ((vx, Dx), (vy, Dy)):
            d.append((gam * sh * u / a)[..., None, None] * I + (gam * (ch * u - sh * u / a) / a ** 2)[..., None, None] * mV
                     + (gam * sh / a)[..., None, None] * D)
        return H, d

    def _coeffs(self, par):
        g = self.grid
        blocks, lsig = self._split(par)
        _, kappa0, H0, _ = self._mod0_split(par)
        kw = dict(variable=True, sigma=np.exp(lsig), kappa0=kappa0, H0=H0, kappa=None, H=None, G=None)
        if self.dvar:
            kw["kappa"] = np.exp(g.bs @ blocks[0])
            H, dH = self._face_fields(blocks)
            kw["H"] = H
        else:
            vx, vy = (blocks[2][0], blocks[3][0]) if self.kind != "iso" else (0.0, 0.0)
            Hc, dH = h_tensor(self.kind, np.exp(blocks[1][0]), vx, vy)
            kw["kappa_c"], kw["H_c"] = np.exp(blocks[0][0]), Hc
        if self.gvar:
            kw["G"] = g.evalAdv(blocks[-1])
        else:
            kw["G_c"] = blocks[-1]
        kw["mix"] = 0 if (self.dvar and self.gvar) else (1 if self.dvar else 2)
        self._fields = (kw.get("kappa"), kw.get("kappa_c"), dH)
        return Coefficients(g, **kw)

    def _contract(self, par, coeffs, parts):
        g = self.grid
        _, kappa0, H0, dH0 = self._mod0_split(par)
        kappa, kappa_c, dH = self._fields
        colsum = parts["colsum"]
        out = []
        if self.dvar:
            cells = parts["cells"]
            out.append(g.bs.T @ (cells[:, OUT_KAPPA] * kappa))
            Hb = cells[:, OUT_H:OUT_H + 16].reshape(-1, 4, 2, 2)
            for d in dH:
                out.append(np.einsum("kfi,kf->i", g.bsH, (Hb * d).sum(axis=(2, 3))))
        else:
            out.append([kappa_c * colsum[OUT_KAPPA]])
            hbar = colsum[OUT_HC:OUT_HC + 4]
            out.append([float(np.dot(hbar, d.reshape(4))) for d in dH])
        if self.gvar:
            cells = parts["cells"]
            wx_bar = cells[:, OUT_DGX:OUT_DGX + 4]
            wy_bar = cells[:, OUT_DGY:OUT_DGY + 4]
            if g.isExtended:
                Ae = g.ext_map()
                wx_bar, wy_bar = Ae.T @ wx_bar, Ae.T @ wy_bar
            out.append(g.bsA[:, 0, :].T @ wx_bar[:, 0] + g.bsA[:, 2, :].T @ wx_bar[:, 2])
            out.append(g.bsA[:, 1, :].T @ wy_bar[:, 1] + g.bsA[:, 3, :].T @ wy_bar[:, 3])
        else:
            out.append([colsum[OUT_WX], colsum[OUT_WY]])
        out.append([parts["g_sigma"]])
        out.append(self._mod0_grad(par, parts, dH0, kappa0))
        out.append([parts["g_tau"]])
        return np.hstack(out).astype(np.float64)

    def print(self, par):
        blocks, lsig = self._split(np.asarray(par))
        return "| κ = %2.2f, γ = %2.2f, σ = %2.2f, τ = %2.2f" % (np.exp(blocks[0]).mean(), np.exp(blocks[1]).mean(),
                                                             np.exp(lsig), np.exp(par[-1]))


class AdvectionVarIDiffusion2D(_FieldAdvDiff):
    kind, dvar, gvar, name = "iso", True, False, "advection-var-diffusion-isotropic-2D"


class AdvectionVarDiffusion2D(_FieldAdvDiff):
    kind, dvar, gvar, name = "ani", True, False, "advection-var-diffusion-anisotropic-2D"


class AdvectionVarHaDiffusion2D(_FieldAdvDiff):
    kind, dvar, gvar, name = "ha", True, False, "advection-var-diffusion-ha-2D"


class VarAdvectionIDiffusion2D(_FieldAdvDiff):
    kind, dvar, gvar, name = "iso", False, True, "var-advection-diffusion-isotropic-2D"
    w0 = 0.01   # var_advection_idiffusion2D.py:22


class VarAdvectionDiffusion2D(_FieldAdvDiff):
    kind, dvar, gvar, name = "ani", False, True, "var-advection-diffusion-anisotropic-2D"


class VarAdvectionHaDiffusion2D(_FieldAdvDiff):
    kind, dvar, gvar, name = "ha", False, True, "var-advection-diffusion-ha-2D"


class VarAdvectionVarIDiffusion2D(_FieldAdvDiff):
    kind, dvar, gvar, name = "iso", True, True, "var-advection-var-diffusion-isotropic-2D"


class VarAdvectionVarHaDiffusion2D(_FieldAdvDiff):
    kind, dvar, gvar, name = "ha", True, True, "var-advection-var-diffusion-ha-2D"


class _SeparableBase(_StencilMixin):
    """Separable space-time models Q = Qt (x) Qs (seperable_spatial_temporal2D.py,
    seperable_spatial_temporal_ha2D.py, seperable_spatial_temporal_idiffusion2D.py):
    Qs is the variable Whittle-Matern precision of the same kind (B-spline
    kappa, gamma (, v) fields; A = Dv Dk - A_H(H), Qs = A^T iDv A) and Qt the
    tridiagonal temporal precision:
      anisotropic: par = [c_k, c_g, c_vx, c_vy, log rho, log tau],
                   Qt = tridiag(-rho; 1, 1+rho^2, .., 1+rho^2, 1) / (1 - rho^2);
      isotropic:   par = [c_k, c_g, a, log sigma, log tau];
      ha:          par = [c_k, c_g, c_vx, c_vy, a, log sigma, log tau],
                   Qt = sigma tridiag(-a; 1, 1+a^2, .., 1+a^2, 1).
    (The reference's isotropic and ha makeQt loop over range(10), i.e. are
    written for T = 10; the form here holds for every T and equals theirs at
    T = 10.)  Only Q_c is factorised at full size (log|Q| = Ns log|Qt| +
    T log|Qs|)."""
    kind = "ani"
    label = "ani-"

    def __init__(self, grid, par=None, bc=3):
        from .grids import grid as make_grid
        self.grid, self.bc = grid, bc
        self.type = "seperable-spatial-temporal-%s2D-bc%d" % (self.label, bc)
        self.Np = grid.Nbs2
        self.Q = self.Q_fac = self.data = self.r = self.S = None
        self._eng = None
        g0 = make_grid(x=grid.x, y=grid.y, extend=grid.Ne if grid.Ne else None, Nbs=grid.Nbs)
        wcls = {"iso": VarWhittleMatern2D, "ani": VarWhittleMaternAnisotropic2D, "ha": VarWhittleMaternHa2D}[self.kind]
        self._wm = wcls(grid=g0, bc=bc)
        if par is None:
            self.setPars(self._default())
        else:
            self.setQ(par=par)

    def _ns(self):
        return self.Np * (2 if self.kind == "iso" else 4)

    def _default(self):
        Np = self.Np
        v = [[-1.0] * Np, [-1.0] * Np] + ([[0.1] * Np, [0.1] * Np] if self.kind != "iso" else [])
        v += [[-1.0]] if self.kind == "ani" else [[0.1, 1.0]]
        return np.hstack(v + [[np.log(100)]]).astype(np.float64)

    def getPars(self, *args, **kwargs):
        return np.hstack([self.coef, [self.tau]]).astype(np.float64)

    def setPars(self, par):
        par = np.asarray(par, dtype=np.float64)
        self.coef = par[:-1].copy()
        Np = self.Np
        self.kappa, self.gamma = par[:Np], par[Np:2 * Np]
        if self.kind != "iso":
            self.vx, self.vy = par[2 * Np:3 * Np], par[3 * Np:4 * Np]
        tp = par[self._ns():-1]
        if self.kind == "ani":
            self.rho = tp[0]
        else:
            self.a, self.sigma = tp[0], tp[1]
        self.tau = par[-1]

    def initFit(self, data, **kwargs):
        assert data.shape[0] <= self.grid.n
        self.data = data
        self.r = data.shape[1] if data.ndim == 2 else 1
        self.S = self.grid.getS(idxs=kwargs.get("idx"))
        return self._default()

    _obs_cols = _SpaceTimeBase._obs_cols

    def _engine(self):
        if self._eng is None:
            self._eng = KronEngine(self.grid, self.bc)
        return self._eng

    def qt(self, tp, diff=False):
        """Diagonal | off-diagonal of Qt (makeQt), or of its derivative in
        log rho (ani) / a (iso, ha)."""
        T = self.grid.T
        d, o = np.zeros(T), np.zeros(T - 1)
        if self.kind == "ani":
            rho = np.exp(tp[0])
            den = 1.0 - rho ** 2
            if diff:
                d[:], o[:] = 4 * rho ** 2 / den ** 2, -rho * (1 + rho ** 2) / den ** 2
                d[0] = d[-1] = 2 * rho ** 2 / den ** 2
            else:
                d[:], o[:] = (1 + rho ** 2) / den, -rho / den
                d[0] = d[-1] = 1.0 / den
        else:
            a, sig = tp[0], np.exp(tp[1])
            if diff:
                d[:], o[:] = 2 * a * sig, -sig
                d[0] = d[-1] = 0.0
            else:
                d[:], o[:] = (1 + a ** 2) * sig, -a * sig
                d[0] = d[-1] = sig
        return np.hstack([d, o])

    def _spatial(self, par):
        """Spatial coefficients and Qs (one-slice values) of par."""
        coeffs = self._wm._coeffs(np.hstack([par[:self._ns()], [0.0]]))
        qs = self._wm._engine().assemble(coeffs)
        return coeffs, qs

    def makeQ(self, par, grad=True):
        par = np.asarray(par, dtype=np.float64)
        eng = self._engine()
        _, qs = self._spatial(par)
        qval = eng.assemble(qs, self.qt(par[self._ns():-1]))
        Q = eng.to_scipy(qval)
        self._last_qval = qval
        return Q, Factor(eng, 0, qval), (_LazyDQ(self, par) if grad else None)

    def setQ(self, par=None, S=None):
        if par is None:
            par = self.getPars()
        else:
            self.setPars(par)
        if S is not None:
            self.S = S
        self.Q, self.Q_fac, _ = self.makeQ(par=par, grad=False)
        self.S = self.grid.getS()

    def logLike(self, par, nh1=100, grad=True, trace="exact"):
        """seperable_spatial_temporal2D.py:127-164: -loglik/(m r) and its
        gradient with the exact trace (selected inverses of Q_c and Qs)."""
        if trace != "exact":
            raise NotImplementedError("separable models: the exact trace only")
        par = np.asarray(par, dtype=np.float64)
        eng = self._engine()
        coeffs, qs = self._spatial(par)
        tp = par[self._ns():-1]
        dqts = [self.qt(tp, diff=True)]
        if self.kind != "ani":
            dqts.append(self.qt(tp))          # d/d log sigma: Qt itself
        like, parts = eng.loglik(qs, self.qt(tp), dqts, coeffs, self._obs_cols(), self.data, par[-1], grad=grad,
                                 contract=self._wm._device_contract())
        if not grad:
            return like
        g = self._wm._field_grad(parts) + list(parts["g_temporal"]) + [parts["g_tau"]]
        m, r = parts["m"], parts["r"]
        return like, -np.array(g) / (m * r)

    def print(self, par):
        Np = self.Np
        s = "| κ = %2.2f, γ = %2.2f" % (np.exp(par[:Np]).mean(), np.exp(par[Np:2 * Np]).mean())
        if self.kind != "iso":
            s += ", vx = %2.2f, vy = %2.2f" % (par[2 * Np:3 * Np].mean(), par[3 * Np:4 * Np].mean())
        tp = par[self._ns():-1]
        s += (", ρ = %2.2f" % np.exp(tp[0])) if self.kind == "ani" else (", a = %2.2f, σ = %2.2f" % (tp[0], np.exp(tp[1])))
        return s + ", τ = %2.2f" % np.exp(par[-1])


class SeperableSpatialTemporal2D(_SeparableBase):
    kind, label = "ani", "ani-"


class SeperableSpatialTemporalHa2D(_SeparableBase):
    kind, label = "ha", "ha-"


class SeperableSpatialTemporalIDiffusion2D(_SeparableBase):
    kind, label = "iso", ""


class _CovAdvDiff(_FieldAdvDiff):
    """Cov-advection families: the advection is lambda * ww, a given face
    field (``grid.assimilate_adv`` of ocean currents), with constant
    (cov_advection_{i,,ha_}diffusion2D.py) or B-spline
    (cov_advection_var_{i,,ha_}diffusion2D.py) kappa and diffusion.
    par = [kappa block, gamma block, (vx, vy blocks,) lambda, log sigma,
    (mod0...), log tau].  As in the reference, the lambda derivative of the
    advection operator is the stencil of ww itself (dA = Aw(ww) dt,
    cov_advection_idiffusion2D.py:59,153-159), which is the derivative for
    lambda > 0.  ww comes with the constructor or initFit(ww=...)."""
    gvar = False
    v0, w0 = 0.1, 0.1   # initial v and lambda

    def __init__(self, grid, mod0, par=None, bc=3, ww=None):
        self.grid, self.mod0, self.bc = grid, mod0, bc
        self.type = "%s-bc%d" % (self.name, bc)
        self.Np = grid.Nbs2
        self.Q = self.Q_fac = self.data = self.r = self.S = None
        self.fitQ0 = True
        self._eng = None
        self.ww = None if ww is None else np.asarray(ww, dtype=np.float64)
        self.setPars(np.hstack([self._init_self(), [np.log(100)]]) if par is None else par)

    def _sizes(self):
        nd = self.Np if self.dvar else 1
        return nd, (1 if self.kind == "iso" else 3), 1

    def _init_self(self):
        nd, nh, _ = self._sizes()
        return np.hstack([[-1.0] * nd, [-1.0] * nd] + [[self.v0] * nd] * (nh - 1) + [[self.w0], [0.0]])

    def initFit(self, data, **kwargs):
        if kwargs.get("ww") is not None:
            self.ww = np.asarray(kwargs["ww"], dtype=np.float64)
        assert self.ww is not None, "the advection field ww is needed (initFit(ww=...))"
        return super().initFit(data, **kwargs)

    def _coeffs(self, par):
        assert self.ww is not None, "the advection field ww is needed (initFit(ww=...))"
        g = self.grid
        blocks, lsig = self._split(par)
        _, kappa0, H0, _ = self._mod0_split(par)
        kw = dict(variable=True, sigma=np.exp(lsig), kappa0=kappa0, H0=H0, G=blocks[-1][0] * self.ww)
        if self.dvar:
            kw["kappa"] = np.exp(g.bs @ blocks[0])
            kw["H"], dH = self._face_fields(blocks)
            kw["mix"] = 0
        else:
            vx, vy = (blocks[2][0], blocks[3][0]) if self.kind != "iso" else (0.0, 0.0)
            Hc, dH = h_tensor(self.kind, np.exp(blocks[1][0]), vx, vy)
            kw.update(kappa=None, H=None, kappa_c=np.exp(blocks[0][0]), H_c=Hc, mix=2)
        self._fields = (kw.get("kappa"), kw.get("kappa_c"), dH)
        return Coefficients(g, **kw)

    def _adv_dir(self):
        return self.ww

    def _contract(self, par, coeffs, parts):
        g = self.grid
        _, kappa0, H0, dH0 = self._mod0_split(par)
        kappa, kappa_c, dH = self._fields
        colsum = parts["colsum"]
        out = []
        if self.dvar:
            cells = parts["cells"]
            out.append(g.bs.T @ (cells[:, OUT_KAPPA] * kappa))
            Hb = cells[:, OUT_H:OUT_H + 16].reshape(-1, 4, 2, 2)
            for d in dH:
                out.append(np.einsum("kfi,kf->i", g.bsH, (Hb * d).sum(axis=(2, 3))))
        else:
            out.append([kappa_c * colsum[OUT_KAPPA]])
            hbar = colsum[OUT_HC:OUT_HC + 4]
            out.append([float(np.dot(hbar, d.reshape(4))) for d in dH])
        out.append([colsum[OUT_ADVDIR]])
        out.append([parts["g_sigma"]])
        out.append(self._mod0_grad(par, parts, dH0, kappa0))
        out.append([parts["g_tau"]])
        return np.hstack(out).astype(np.float64)


class CovAdvectionIDiffusion2D(_CovAdvDiff):
    kind, dvar, name = "iso", False, "cov-advection-idiffusion-2D"


class CovAdvectionDiffusion2D(_CovAdvDiff):
    kind, dvar, name = "ani", False, "cov-advection-diffusion-2D"


class CovAdvectionHaDiffusion2D(_CovAdvDiff):
    kind, dvar, name = "ha", False, "cov-advection-ha-diffusion-2D"
    v0, w0 = 0.01, 0.01   # cov_advection_ha_diffusion2D.py:27


class CovAdvectionVarIDiffusion2D(_CovAdvDiff):
    kind, dvar, name = "iso", True, "cov-advection-var-idiffusion-2D"


class CovAdvectionVarDiffusion2D(_CovAdvDiff):
    kind, dvar, name = "ani", True, "cov-advection-var-diffusion-2D"


class CovAdvectionVarHaDiffusion2D(_CovAdvDiff):
    kind, dvar, name = "ha", True, "cov-advection-var-ha-diffusion-2D"


class _TangentDQ:
    """The reference's list of dQ_i (one sparse matrix per parameter except
    tau, in the parameter order; var_advection_var_diffusion2D.py:118-197,
    advection_idiffusion2D.py:118-163), each assembled on demand on the GPU
    as the directional derivative of the block formula along the
    parameter's coefficient direction (``spde_assemble_tangent``), with the
    reference's derivative stencils.  Returned with the scipy pattern (exact
    zeros dropped), like Q."""

    def __init__(self, model, par, coeffs, directions):
        self.model, self.par, self.coeffs, self.dirs = model, par, coeffs, directions

    def __len__(self):
        return len(self.dirs)

    def __iter__(self):
        return (self[i] for i in range(len(self)))

    def __getitem__(self, i):
        if isinstance(i, slice):
            return [self[k] for k in range(*i.indices(len(self)))]
        import torch
        from . import _native as nat
        if i < 0:
            i += len(self)
        if not 0 <= i < len(self):
            raise IndexError(i)
        eng = self.model._engine()
        plan = eng.plan
        base = torch.empty(plan.nnz, dtype=torch.float64, device="cuda")
        plan.assemble(self.coeffs.c, base)       # the base point of the derivative
        d, keep = self.dirs[i]()
        dq = torch.empty(plan.nnz, dtype=torch.float64, device="cuda")
        nat.check(nat.lib().spde_assemble_tangent(plan._h, ctypes.byref(self.coeffs.c), ctypes.byref(d), _p(dq),
                                                  ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
        del keep
        return eng.to_scipy(dq)


def _direction(kind=0, dkappa=None, dkappa_c=0.0, dH=None, dH_c=None, dG=None, adv_diff=0, dkappa0=0.0, dH0=None):
    """A spde_direction and the device arrays it points to."""
    import torch
    from . import _native as nat
    d = nat.Direction()
    d.kind = kind
    keep = []

    def dev(a):
        t = torch.as_tensor(np.ascontiguousarray(a, dtype=np.float64).reshape(-1)).cuda()
        keep.append(t)
        return t.data_ptr()
    if dkappa is not None:
        d.dkappa = dev(dkappa)
    d.dkappa_c = float(dkappa_c)
    if dH is not None:
        d.dH = dev(dH)
        d.has_dH = 1
    if dH_c is not None:
        for q, v in enumerate(np.asarray(dH_c, dtype=np.float64).reshape(4)):
            d.dH_c[q] = v
        d.has_dH = 1
    if dG is not None:
        d.dG = dev(dG)
    d.adv_diff = int(adv_diff)
    d.dkappa0 = float(dkappa0)
    if dH0 is not None:
        for q, v in enumerate(np.asarray(dH0, dtype=np.float64).reshape(4)):
            d.dH0[q] = v
    return d, keep


class _LazyDQ:
    """The reference's list of dQ_i, produced on demand (one matrix per
    parameter except tau).  Not needed by logLike, whose gradient contracts all
    of them at once through the adjoint of the assembly."""

    def __init__(self, model, par):
        self.model, self.par = model, par

    def __len__(self):
        return self.par.size - 1

    def __getitem__(self, i):
        raise NotImplementedError("explicit dQ matrices are not materialised; logLike contracts them on the GPU")


def spde_init(model, grid, parameters=None, ani=True, ha=True, bc=3, mod0=None):
    """Dispatcher (spdes/__init__.py:1-103) for the classes of the hot path."""
    if grid.sdim != 2:
        raise NotImplementedError("only 2-D spatial and space-time grids")
    if model in ("whittle-matern", 1):
        cls = WhittleMaternHa2D if ha else (WhittleMaternAnisotropic2D if ani else WhittleMatern2D)
        return cls(grid=grid, par=parameters, bc=bc)
    if model in ("var-whittle-matern", -1):
        cls = VarWhittleMaternHa2D if ha else (VarWhittleMaternAnisotropic2D if ani else VarWhittleMatern2D)
        return cls(grid=grid, par=parameters, bc=bc)
    if model in ("advection-diffusion", 2):
        cls = AdvectionHaDiffusion2D if ha else (AdvectionDiffusion2D if ani else AdvectionIDiffusion2D)
        return cls(grid=grid, mod0=mod0, par=parameters, bc=bc)
    if model in ("advection-var-diffusion", 3):
        cls = AdvectionVarHaDiffusion2D if ha else (AdvectionVarDiffusion2D if ani else AdvectionVarIDiffusion2D)
        return cls(grid=grid, mod0=mod0, par=parameters, bc=bc)
    if model in ("cov-advection-diffusion", 4):
        cls = CovAdvectionHaDiffusion2D if ha else (CovAdvectionDiffusion2D if ani else CovAdvectionIDiffusion2D)
        return cls(grid=grid, mod0=mod0, par=parameters, bc=bc)
    if model in ("cov-advection-var-diffusion", 5):
        cls = (CovAdvectionVarHaDiffusion2D if ha else
               (CovAdvectionVarDiffusion2D if ani else CovAdvectionVarIDiffusion2D))
        return cls(grid=grid, mod0=mod0, par=parameters, bc=bc)
    if model in ("var-advection-diffusion", 6):
        cls = VarAdvectionHaDiffusion2D if ha else (VarAdvectionDiffusion2D if ani else VarAdvectionIDiffusion2D)
        return cls(grid=grid, mod0=mod0, par=parameters, bc=bc)
    if model in ("var-advection-var-diffusion", 7):
        cls = (VarAdvectionVarHaDiffusion2D if ha else
               (VarAdvectionVarDiffusion2D if ani else VarAdvectionVarIDiffusion2D))
        return cls(grid=grid, mod0=mod0, par=parameters, bc=bc)
    if model in ("seperable-spatial-temporal", 8):
        cls = (SeperableSpatialTemporalHa2D if ha else
               (SeperableSpatialTemporal2D if ani else SeperableSpatialTemporalIDiffusion2D))
        return cls(grid=grid, par=parameters, bc=bc)
    raise NotImplementedError("model %r is outside the GMRF hot path built here" % (model,))
