"""Pins for the oracle's model layer: closed forms, brute force, finite
differences (each chosen so a dropped term, a sign or an index error fails)."""
import numpy as np
import pytest
from scipy import sparse

from oracle import fixtures as F, models as Mo


def _spatial(c):
    m = c["model"]
    if isinstance(m, Mo.VarAdvVarDiff):
        A, q, s = m.spatial_operator(c["par"])
    else:
        A, q, s = Mo.stationary_spatial_operator(m, c["par"])
    A0 = c["mod0"].A0(c["mod0"].par)[0]
    return A, q, s, A0


def _fform(c):
    """F (block lower-bidiagonal) and diag(D) of Q = F^T D F."""
    g = c["grid"]
    A, q, s, A0 = _spatial(c)
    T, Ns = g.T, g.Ns
    blocks = [[None] * T for _ in range(T)]
    blocks[0][0] = A0 / np.sqrt(g.V)
    for t in range(1, T):
        blocks[t][t] = A / g.V
        blocks[t][t - 1] = -sparse.eye(Ns)
    Fm = sparse.bmat(blocks).tocsr()
    d = np.hstack([np.ones(Ns)] + [q / (g.dt * s)] * (T - 1))
    return Fm, d


CASES = {
    "iso_b1": lambda: F.stationary(9, 8, 4, bc=1, m=30),
    "ani_b3": lambda: F.stationary(8, 9, 3, bc=3, kind="ani", m=30),
    "ha_b1": lambda: F.stationary(7, 8, 3, bc=1, kind="ha", m=30),
    "var_b1": lambda: F.small(8, 7, 4, bc=1),
    "var_b3": lambda: F.small(7, 8, 3, bc=3),
    "var_b1_ext": lambda: F.small(6, 6, 3, bc=1, ne=2),
}


@pytest.mark.parametrize("case", sorted(CASES))
def test_q_equals_fform(case):
    c = CASES[case]()
    Q, _ = c["model"].makeQ(c["par"], grad=False)
    Fm, d = _fform(c)
    Qf = (Fm.T @ sparse.diags(d) @ Fm).toarray()
    Qd = Q.toarray()
    assert np.abs(Qd - Qd.T).max() <= 1e-12 * np.abs(Qd).max()
    assert np.allclose(Qd, Qf, rtol=1e-12, atol=1e-12 * np.abs(Qd).max())


@pytest.mark.parametrize("case", sorted(CASES))
def test_logdet_closed_form(case):
    c = CASES[case]()
    g = c["grid"]
    Q, _ = c["model"].makeQ(c["par"], grad=False)
    A, q, s, A0 = _spatial(c)
    cf = Mo.logdet_closed_form(A, q, A0, g.V, g.T, s, g.dt)
    dense = np.linalg.slogdet(Q.toarray())
    assert dense[0] > 0
    assert abs(cf - dense[1]) <= 1e-11 * abs(dense[1])


@pytest.mark.parametrize("case", ["iso_b1", "var_b3", "ha_b1"])
def test_loglike_is_gaussian_marginal(case):
    """-like*m = log N(y; 0, S Q^-1 S^T + I/tau) + m/2 log 2pi  (brute force)."""
    c = CASES[case]()
    g = c["grid"]
    Q, _ = c["model"].makeQ(c["par"], grad=False)
    S = g.getS(c["idx"])
    like, _, _ = Mo.loglike(Q, [], S, c["y"], c["par"][-1])
    tau = np.exp(c["par"][-1])
    m = S.shape[0]
    C = S.toarray() @ np.linalg.solve(Q.toarray(), S.toarray().T) + np.eye(m) / tau
    sgn, ld = np.linalg.slogdet(C)
    y = c["y"]
    logp = -0.5 * ld - 0.5 * y @ np.linalg.solve(C, y)
    assert abs(-like * m - logp) <= 1e-9 * abs(logp)


@pytest.mark.parametrize("case", ["iso_b1", "var_b3"])
def test_loglike_several_realisations_is_sum_of_marginals(case):
    """r independent realisations at the same locations: -like*m*r is the sum
    of the r Gaussian log-densities (brute force), so the r-column terms
    (r log|Q|, r log|Q_c|, the summed quadratic forms) are pinned."""
    c = CASES[case]()
    g = c["grid"]
    Q, _ = c["model"].makeQ(c["par"], grad=False)
    S = g.getS(c["idx"])
    rng = np.random.default_rng(5)
    m = S.shape[0]
    Y = np.column_stack([c["y"], 0.5 * c["y"][::-1], 0.2 * rng.normal(size=m)])
    like, _, _ = Mo.loglike(Q, [], S, Y, c["par"][-1])
    tau = np.exp(c["par"][-1])
    C = S.toarray() @ np.linalg.solve(Q.toarray(), S.toarray().T) + np.eye(m) / tau
    sgn, ld = np.linalg.slogdet(C)
    logp = sum(-0.5 * ld - 0.5 * y @ np.linalg.solve(C, y) for y in Y.T)
    assert abs(-like * m * Y.shape[1] - logp) <= 1e-9 * abs(logp)


def _fd_check(c, which, h=1e-5, rtol=2e-5):
    g = c["grid"]
    S = g.getS(c["idx"])
    par = c["par"]
    Q, dQ = c["model"].makeQ(par, grad=True)
    like, jac, _ = Mo.loglike(Q, dQ, S, c["y"], par[-1], trace="exact")
    for i in which:
        pp, pm = par.copy(), par.copy()
        pp[i] += h
        pm[i] -= h
        lp = Mo.loglike(c["model"].makeQ(pp, grad=False)[0], [], S, c["y"], pp[-1])[0]
        lm = Mo.loglike(c["model"].makeQ(pm, grad=False)[0], [], S, c["y"], pm[-1])[0]
        fd = (lp - lm) / (2 * h)
        assert abs(fd - jac[i]) <= rtol * max(abs(fd), 1e-3), (i, fd, jac[i])


def test_gradient_fd_var_dirichlet():
    c = CASES["var_b3"]()
    Np = c["grid"].Nbs2
    _fd_check(c, list(range(0, 6 * Np, 2)) + [6 * Np, 6 * Np + 1])


def test_gradient_fd_stationary_dirichlet():
    c = CASES["ani_b3"]()
    _fd_check(c, range(8))


def test_gradient_fd_stationary_neumann_non_advection():
    """bc=1 advection derivative stencils are not the operator's derivative
    (Acw_2D_b1.cpp:63-80), so only the other parameters are FD-checked here."""
    c = CASES["iso_b1"]()
    _fd_check(c, [0, 1, 4, 5])


def test_pattern_iso_corners_vanish():
    """Isotropic H gives exact-zero diffusion corners; scipy's sums drop them
    so an interior row of Q has 13 + 5 + 5 entries (5-point A), not 25 + 9 + 9."""
    c = F.stationary(9, 9, 3, bc=1, m=10)
    Q, _ = c["model"].makeQ(c["par"], grad=False)
    g = c["grid"]
    k = 4 + 4 * 9 + 1 * 81
    assert Q.tocsr()[k].nnz == 23
    c = F.small(9, 9, 3, bc=1)
    Q, _ = c["model"].makeQ(c["par"], grad=False)
    assert Q.tocsr()[k].nnz == 43


def test_fform_sampler_solves_factor():
    c = CASES["var_b1"]()
    g = c["grid"]
    A, q, s, A0 = _spatial(c)
    z = np.random.default_rng(0).normal(size=(g.n, 3))
    x = Mo.sample_fform(A, q, A0, g.V, g.T, s, g.dt, z)
    Fm, d = _fform(c)
    assert np.allclose(Fm @ x, z / np.sqrt(d)[:, None], rtol=1e-10, atol=1e-10)


def test_hutchinson_probes_stream():
    """Legacy global RandomState stream (NEP 19): the reference's probe matrix."""
    V1 = Mo.reference_probes(10, 4, seed=5)
    np.random.seed(5)
    raw = np.random.randint(1, 3, 40)
    assert np.array_equal(V1.ravel(), 2 * raw - 3)
    assert set(np.unique(V1)) == {-1.0, 1.0}


@pytest.mark.parametrize("kind", ["iso", "ani", "ha"])
def test_var_whittle_matern_derivatives_and_h_map(kind):
    """Variable Whittle-Matern oracle: every dQ_i against central differences
    of Q, and the ha face tensor against gamma * expm([[vx, vy], [vy, -vx]])."""
    from scipy.linalg import expm
    from oracle import grid as OG
    g = OG.SpatialGrid(F.axis(9), F.axis(8), Nbs=3)
    m = Mo.VarWhittleMatern(g, kind, bc=1)
    rng = np.random.default_rng(1)
    par = 0.3 * rng.normal(size=m.Np * (2 if kind == "iso" else 4) + 1)
    Q, dQ = m.makeQ(par)
    for i in range(0, par.size - 1, 4):
        h = 1e-6
        pp, pm = par.copy(), par.copy()
        pp[i] += h
        pm[i] -= h
        fd = (m.makeQ(pp, False)[0] - m.makeQ(pm, False)[0]) / (2 * h)
        assert abs(fd - dQ[i]).max() <= 1e-6 * abs(dQ[i]).max(), i
    if kind == "ha":
        _, H, *_ = m.fields(par)
        _, cg, cvx, cvy = m.split(par)
        vx, vy, gam = g.evalBH(cvx), g.evalBH(cvy), np.exp(g.evalBH(cg))
        for k, f in [(0, 0), (17, 2), (40, 3)]:
            ref = gam[k, f] * expm(np.array([[vx[k, f], vy[k, f]], [vy[k, f], -vx[k, f]]]))
            assert np.allclose(H[k, f], ref, rtol=1e-13, atol=1e-15)


FIELD_COMBOS = [(k, dv, gv) for k in ("iso", "ani", "ha") for dv, gv in ((True, False), (False, True), (True, True))]


@pytest.mark.parametrize("kind,dvar,gvar", FIELD_COMBOS)
def test_field_families_reduce_to_stationary(kind, dvar, gvar):
    """With every B-spline field constant (the bases sum to one) and bc=3 the
    field families are the stationary model of the same kind: Q agrees to
    rounding.  (At bc=1 the variable stencils' border rows differ from the
    constant ones in the reference as well, so this pin is a bc=3 one.)"""
    from oracle import grid as OG
    g = OG.STGrid(F.axis(8), F.axis(7), np.arange(4.0), Nbs=3)
    mod0 = F.mod0_iso(8, 7, bc=3)
    Np = g.Nbs2
    nh = 1 if kind == "iso" else 3
    ps = (np.array([0.2, np.log(0.5), 0.3, -0.2, 0.1, np.log(100.0)]) if kind == "iso" else
          np.array([0.2, np.log(0.5), 0.4, -0.3, 0.3, -0.2, 0.1, np.log(100.0)]))
    Qs, _ = Mo.StationaryAdvDiff(g, mod0, kind=kind, bc=3).makeQ(ps, grad=False)
    fm = Mo.FieldAdvDiff(g, mod0, kind, dvar, gvar, bc=3)
    nd = Np if dvar else 1
    blocks = [np.full(nd, ps[i]) for i in range(1 + nh)]
    w = ps[1 + nh:3 + nh]
    blocks.append(np.repeat(w, Np) if gvar else w)
    Qf, _ = fm.makeQ(np.hstack(blocks + [ps[-2:]]), grad=False)
    assert abs(Qf - Qs).max() <= 1e-13 * abs(Qs).max()


def test_field_family_ani_all_fields_is_var_model():
    """All-field anisotropic case = the 100x100x20 B-spline model (pinned separately)."""
    c = F.small(8, 7, 4, bc=1)
    fm = Mo.FieldAdvDiff(c["grid"], c["mod0"], "ani", True, True, bc=1)
    Qv, _ = c["model"].makeQ(c["par"], grad=False)
    Qf, _ = fm.makeQ(c["par"], grad=False)
    assert abs(Qf - Qv).max() == 0.0


@pytest.mark.parametrize("kind,dvar,gvar", FIELD_COMBOS)
def test_field_family_derivatives(kind, dvar, gvar):
    """Every 3rd dQ_i against central differences of Q (bc=3, where the
    advection stencils' derivatives are the operator's)."""
    c = F.field_model(kind=kind, dvar=dvar, gvar=gvar, bc=3)
    m, par = c["model"], c["par"]
    Q, dQ = m.makeQ(par, grad=True)
    assert len(dQ) == par.size - 1
    for i in list(range(0, par.size - 1, 3)) + [par.size - 2]:
        h = 1e-6
        pp, pm = par.copy(), par.copy()
        pp[i] += h
        pm[i] -= h
        fd = (m.makeQ(pp, False)[0] - m.makeQ(pm, False)[0]) / (2 * h)
        assert abs(fd - dQ[i]).max() <= 1e-6 * max(abs(dQ[i]).max(), 1e-3 * abs(Q).max()), i


@pytest.mark.parametrize("kind", ["iso", "ani", "ha"])
def test_separable_temporal_precision_and_derivatives(kind):
    """Separable oracle: Qt^-1 is the AR(1) covariance (rho^|t-t'| for ani;
    a^|t-t'| / (sigma (1 - a^2)) for iso/ha), Q = Qt (x) Qs with Qs the
    variable Whittle-Matern precision, and every 3rd dQ_i (plus the temporal
    ones) against central differences of Q."""
    from oracle import grid as OG
    g = OG.STGrid(F.axis(7), F.axis(6), np.arange(10.0), Nbs=3)
    m = Mo.Separable(g, kind, bc=3)
    rng = np.random.default_rng(3)
    tp = [np.log(0.6)] if kind == "ani" else [0.7, np.log(2.0)]
    par = np.hstack([0.3 * rng.normal(size=m.ns), tp, [np.log(100.0)]])
    Qt = m.qt(np.array(tp), 10).toarray()
    lag = np.abs(np.subtract.outer(np.arange(10), np.arange(10)))
    cov = 0.6 ** lag if kind == "ani" else 0.7 ** lag / (2.0 * (1 - 0.49))
    assert np.allclose(np.linalg.inv(Qt), cov, rtol=1e-12, atol=1e-12)
    Q, dQ = m.makeQ(par)
    Qs, _ = m.wm.makeQ(np.hstack([par[:m.ns], [0.0]]), grad=False)
    assert abs(Q[:g.Ns, :g.Ns] - Qt[0, 0] * Qs).max() <= 1e-12 * abs(Qs).max()
    assert abs(Q[g.Ns:2 * g.Ns, :g.Ns] - Qt[1, 0] * Qs).max() <= 1e-12 * abs(Qs).max()
    assert len(dQ) == par.size - 1
    for i in list(range(0, m.ns, 3)) + list(range(m.ns, par.size - 1)):
        h = 1e-6
        pp, pm = par.copy(), par.copy()
        pp[i] += h
        pm[i] -= h
        fd = (m.makeQ(pp, False)[0] - m.makeQ(pm, False)[0]) / (2 * h)
        assert abs(fd - dQ[i]).max() <= 1e-6 * abs(dQ[i]).max(), i


def test_assimilate_adv_faces():
    """Face velocities from currents: a constant field stays constant on
    every face (border faces use the cell alone), a linear one gives the face
    mid-points inside and the cell value at the border; extended grids
    extrapolate with the advection border map."""
    from oracle import grid as OG
    import spdepy_amd as sp
    M, N = 6, 5
    for ne in (None, 2):
        og = OG.STGrid(F.axis(M), F.axis(N), np.arange(3.0), extend=ne, Nbs=3)
        pg = sp.grid(x=F.axis(M), y=F.axis(N), t=np.arange(3.0), extend=ne, Nbs=3)
        X, Y = np.meshgrid(F.axis(M), F.axis(N))
        we, wn = X.ravel(), 2 * Y.ravel()
        wo, wp = og.assimilate_adv(we, wn), pg.assimilate_adv(we, wn)
        assert np.allclose(wo, wp, rtol=0, atol=1e-15)
        if ne is None:
            h = 1.0 / M
            i = np.arange(M * N) % M
            assert np.allclose(wo[:, 0], np.where(i + 1 < M, we + h / 2, we))
            assert np.allclose(wo[:, 2], np.where(i > 0, we - h / 2, we))
            c = og.assimilate_adv(np.full(M * N, 0.7), np.full(M * N, -0.3))
            assert np.allclose(c[:, [0, 2]], 0.7) and np.allclose(c[:, [1, 3]], -0.3)
        else:
            assert wo.shape == (og.Ns, 4)
            assert np.allclose(wo, og._ext_map() @ OG.STGrid(F.axis(M), F.axis(N), np.arange(3.0)).assimilate_adv(we, wn))


@pytest.mark.parametrize("kind,dvar", [("iso", False), ("ani", True), ("ha", False)])
def test_cov_family_derivatives(kind, dvar):
    """Cov-advection oracle (advection lambda * ww): with lambda > 0 at bc=3
    the reference's dA = Aw(ww) dt is the derivative, so every 3rd dQ_i and
    the lambda one match central differences of Q."""
    c = F.field_model(kind=kind, dvar=dvar, gvar=False, bc=3, cov=0.8)
    m, par = c["model"], c["par"]
    Q, dQ = m.makeQ(par, grad=True)
    assert len(dQ) == par.size - 1
    for i in list(range(0, par.size - 3, 3)) + [par.size - 3, par.size - 2]:
        h = 1e-6
        pp, pm = par.copy(), par.copy()
        pp[i] += h
        pm[i] -= h
        fd = (m.makeQ(pp, False)[0] - m.makeQ(pm, False)[0]) / (2 * h)
        assert abs(fd - dQ[i]).max() <= 1e-6 * max(abs(dQ[i]).max(), 1e-3 * abs(Q).max()), i


def test_golden_30x30x10_is_the_oracle():
    """tests/golden/stationary_30x30x10.npz (the GPU parity target at 30 x 30 x 10) is what
    the oracle computes now (dense inverses at n = 9,000: ~15 s)."""
    import os
    gold = np.load(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "stationary_30x30x10.npz"))
    c = F.stationary()
    # y holds sparse solves, whose last bits depend on the host's BLAS kernels: equal to
    # the rounding that the value below is held to
    assert np.array_equal(c["idx"], gold["idx"])
    assert np.abs(c["y"] - gold["y"]).max() <= 1e-12 * np.abs(gold["y"]).max()
    Q, dQ = c["model"].makeQ(c["par"], grad=True)
    S = c["grid"].getS(c["idx"])
    like, jac, _ = Mo.loglike(Q.tocsc(), dQ, S, c["y"], c["par"][-1], trace="exact")
    assert abs(like - float(gold["like"])) <= 1e-12 * abs(like)
    assert np.allclose(jac, gold["jac"], rtol=1e-10, atol=1e-12 * np.abs(jac).max())


def test_sparse_lu_logdet_branch_matches_closed_form_at_30x30x10():
    """The oracle's n > 4,000 branch (sparse LU with symmetric pivoting, the
    CHOLMOD stand-in for log|Q| and log|Q_c|) against the closed form and the
    determinant lemma at 30 x 30 x 10 (n = 9,000)."""
    c = F.stationary()
    g = c["grid"]
    Q, _ = c["model"].makeQ(c["par"], grad=False)
    A, q, s = Mo.stationary_spatial_operator(c["model"], c["par"])
    A0 = c["mod0"].A0(c["mod0"].par)[0]
    cf = Mo.logdet_closed_form(A, q, A0, g.V, g.T, s, g.dt)
    assert abs(Mo.logdet_spd(Q) - cf) <= 1e-11 * abs(cf)
    tau = np.exp(c["par"][-1])
    cols = g.n2e(c["idx"])
    S = g.getS(c["idx"])
    Qc = (Q + tau * (S.T @ S)).tocsc()
    W = Mo.qinv_columns(A, q, A0, g.V, g.T, s, g.dt, cols)
    K = W[cols] + np.eye(len(cols)) / tau
    lemma = cf + len(cols) * np.log(tau) + np.linalg.slogdet(0.5 * (K + K.T))[1]
    assert abs(Mo.logdet_spd(Qc) - lemma) <= 1e-11 * abs(lemma)


def test_woodbury_route_reproduces_golden_30x30x10():
    """The Woodbury form that writes the 100 x 100 x 20 fixture reproduces the
    dense-inverse values of tests/golden/stationary_30x30x10.npz at n = 9,000."""
    import os
    gold = np.load(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "stationary_30x30x10.npz"))
    c = F.stationary()
    g, model, par = c["grid"], c["model"], c["par"]
    M, N, T = g.shape
    Q, dQ = model.makeQ(par, grad=True)
    A, q, s = Mo.stationary_spatial_operator(model, par)
    A0 = c["mod0"].A0(c["mod0"].par)[0]
    like, jac, _ = Mo.loglike_woodbury(Q, dQ, A, q, A0, g.V, T, s, g.dt, M, N, g.n2e(c["idx"]), c["y"], par[-1])
    assert abs(like - float(gold["like"])) <= 1e-11 * abs(like)
    # the golden gradient subtracts the traces of two dense inverses (Q and
    # Q_c, condition ~1e8 at n = 9,000), which carries ~1e-9 of the
    # gradient's scale in round-off; the Woodbury form takes the difference
    # directly
    assert np.allclose(jac, gold["jac"], rtol=0, atol=5e-9 * np.abs(jac).max())
