"""Full-size (100 x 100 x 20, n = 200,000) checks of the GPU path through
size-independent properties: the closed-form log-determinant, central finite
differences of the gradient, bitwise determinism, and agreement of the
sampler with the selected inverse."""
import numpy as np
import pytest

from oracle import models as Mo
from tests.gpu_util import step

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def workload():
    import bench
    step("build 100x100x20 workload")
    mod, par = bench.build_workload()
    return mod, par


def test_logdet_matches_closed_form(workload):
    from oracle import fixtures as F
    mod, par = workload
    step("factor Q at 100x100x20")
    Q, fac, _ = mod.makeQ(par, grad=False)
    ld = fac.logdet()
    c = F.bspline_100x100x20()
    assert np.allclose(c["par"], par)
    A, q, s = c["model"].spatial_operator(c["par"])
    A0 = c["mod0"].A0(c["mod0"].par)[0]
    cf = Mo.logdet_closed_form(A, q, A0, c["grid"].V, 20, s, c["grid"].dt)
    assert abs(ld - cf) <= 1e-11 * abs(cf), (ld, cf)


def test_gradient_central_differences(workload):
    """bc=1: the advection derivative stencils of the reference are not the
    operator's derivative at boundary cells, so w-coefficients are skipped."""
    mod, par = workload
    step("logLike + grad at 100x100x20")
    like, jac = mod.logLike(par)
    Np = mod.Np

    def central(i, h):
        pp, pm = par.copy(), par.copy()
        pp[i] += h
        pm[i] -= h
        return (mod.logLike(pp, grad=False) - mod.logLike(pm, grad=False)) / (2 * h)

    # The analytic gradient subtracts two traces of size ~n (Q^-1 and Q_c^-1
    # against dQ) and the differences subtract log-likelihoods of size ~n, so
    # both carry round-off of a few 1e-9 of the gradient's scale; a wrong
    # adjoint term shows up as an O(1) relative error.
    scale = np.abs(jac).max()
    bad = []
    for i in [0, 27, Np + 5, 2 * Np + 9, 3 * Np + 40, 6 * Np, 6 * Np + 1]:
        step("finite difference %d" % i)
        fd = (4 * central(i, 1e-4) - central(i, 2e-4)) / 3   # Richardson: O(h^4)
        err = abs(fd - jac[i])
        print("  param %4d  grad %+.10e  fd %+.10e  err/scale %.2e" % (i, jac[i], fd, err / scale))
        if err > 2e-6 * abs(jac[i]) + 2e-6 * scale:
            bad.append((i, fd, jac[i]))
    assert not bad, bad


def test_closed_form_route_matches_full_factorisation(workload):
    """log|Q| and its gradient from the spatial matrices of Q = F^T D F agree
    with the full factorisation and selected inverse of Q at 100x100x20."""
    mod, par = workload
    step("logLike closed vs factor at 100x100x20")
    l1, j1 = mod.logLike(par, logdet="closed")
    l2, j2 = mod.logLike(par, logdet="factor")
    print("  like closed %.15e factor %.15e; max grad diff / scale %.2e"
          % (l1, l2, np.abs(j1 - j2).max() / np.abs(j2).max()))
    assert abs(l1 - l2) <= 1e-11 * abs(l2)
    # the factorised route's gradient subtracts two full-size traces whose
    # selected inverses carry ~1e-9 round-off (see the identity test below)
    assert np.allclose(j1, j2, rtol=1e-8, atol=1e-8 * np.abs(j2).max())


def test_evaluation_is_deterministic(workload):
    mod, par = workload
    step("two identical evaluations")
    l1, j1 = mod.logLike(par)
    l2, j2 = mod.logLike(par)
    assert l1 == l2 and np.array_equal(j1, j2)


def test_sampler_and_selected_inverse_identities(workload):
    """Exact identities at full size: x = P^T L^-T z satisfies x^T Q x = z^T z;
    the selected inverse satisfies sum_j Q_ij Sigma_ij = (Q Q^-1)_ii = 1 for
    every row i (Q's pattern holds every j the sum needs)."""
    import torch
    mod, par = workload
    eng = mod._engine()
    qval = eng.assemble(mod._coeffs(par))
    step("factor + sample + selinv")
    eng.plan.factor(0, qval)
    # 16 right-hand sides, as the configuration's 16 conditional samples (the
    # tile-GEMM solve path; one right-hand side takes the bandwidth-bound one)
    z = torch.as_tensor(np.random.default_rng(0).normal(size=(eng.n, 16))).cuda()
    x = eng.plan.solve(0, z, 2)
    qx = eng.plan.spmv(qval, x)
    lhs = (x * qx).sum(0).cpu().numpy()
    rhs = (z * z).sum(0).cpu().numpy()
    assert np.allclose(lhs, rhs, rtol=1e-10)
    sig = eng.plan.selinv(0)
    indptr, _ = eng.plan.structure()
    rows = torch.as_tensor(np.repeat(np.arange(eng.n), np.diff(indptr))).cuda()
    diag = torch.zeros(eng.n, dtype=torch.float64, device="cuda").index_add_(0, rows, qval * sig)
    scale = torch.zeros(eng.n, dtype=torch.float64, device="cuda").index_add_(0, rows, (qval * sig).abs())
    err = float((diag - 1.0).abs().max())
    print("  max |sum_j Q_ij Sigma_ij - 1| = %.3e (row scale sum_j |Q_ij Sigma_ij| up to %.3e)"
          % (err, float(scale.max())))
    # FP64 round-off of the factor and of the recursion grows with the
    # condition number of Q (a few 1e-9 here); a wrong term is an O(1) error
    assert err < 1e-8


def test_fused_entry_point_at_full_size(workload):
    """spde_loglik_grad at 100x100x20 gives the engine path's value and
    per-cell adjoints."""
    from spdepy_amd import engine as E
    mod, par = workload
    eng = mod._engine()
    coeffs = mod._coeffs(par)
    step("engine path at 100x100x20")
    like_e, parts_e = eng.loglik(coeffs, mod._obs_cols(), mod.data, par[-1], grad=True)
    step("fused entry point at 100x100x20")
    like_f, parts_f = E.loglik_fused(eng, coeffs, mod._obs_cols(), mod.data, par[-1])
    assert abs(like_f - like_e) <= 1e-12 * abs(like_e)
    scale = np.abs(parts_e["cells"]).max()
    assert np.allclose(parts_f["cells"], parts_e["cells"], rtol=1e-11, atol=1e-12 * scale)
