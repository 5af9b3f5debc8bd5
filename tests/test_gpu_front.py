"""Dense partial factorisation of the fronts (one launch per level, tiles handed
over by flags) at the edges of its 64-wide tiles, against dense numpy."""
import numpy as np
import pytest

from tests.gpu_util import step

pytestmark = pytest.mark.gpu


def _spd(plan, seed):
    """Values of a well-conditioned matrix on the plan's pattern, and its dense form."""
    indptr, indices = plan.structure()
    n = plan.n
    rows = np.repeat(np.arange(n), np.diff(indptr))
    A = np.zeros((n, n))
    A[rows, indices] = np.random.default_rng(seed).normal(size=len(indices))
    A = 0.5 * (A + A.T)
    A[np.arange(n), np.arange(n)] = 1.0 + np.abs(A).sum(1)
    return A[rows, indices], A


# own columns of the single front (or of the root): one tile less, more or
# equal, two and three tiles, more than 32 column tiles, boundary rows
@pytest.mark.parametrize("M,N,T,leaf", [(7, 9, 1, 5000), (8, 8, 1, 5000), (5, 13, 1, 5000), (8, 16, 1, 5000),
                                        (3, 43, 1, 5000), (10, 19, 1, 5000), (22, 100, 1, 5000), (9, 8, 5, 64),
                                        (12, 11, 6, 65), (17, 16, 4, 8)])
def test_front_factorisation_matches_dense(M, N, T, leaf):
    import torch
    from spdepy_amd.plan import Plan
    plan = Plan(M, N, T, 3, leaf_max=leaf)
    B = np.random.default_rng(1).normal(size=(plan.n, 2))
    logdets = []
    for seed in (0, 1, 0):          # the counters start over each time
        q, A = _spd(plan, seed)
        step("front %dx%dx%d leaf %d seed %d" % (M, N, T, leaf, seed))
        ld = plan.factor(0, torch.as_tensor(q).cuda())
        ref = np.linalg.slogdet(A)[1]
        assert abs(ld - ref) <= 1e-12 * abs(ref)
        X = plan.solve(0, torch.as_tensor(B).cuda()).cpu().numpy()
        assert np.abs(A @ X - B).max() <= 1e-11 * np.abs(B).max()
        logdets.append(ld)
    assert logdets[0] == logdets[2]


@pytest.mark.parametrize("M,N,at", [(8, 8, 0), (8, 8, 63), (10, 19, 70), (22, 100, 2199)])
def test_front_factorisation_reports_the_pivot(M, N, at):
    import torch
    from spdepy_amd import _native as nat
    from spdepy_amd.plan import Plan
    plan = Plan(M, N, 1, 3, leaf_max=5000)
    q, A = _spd(plan, 2)
    indptr, indices = plan.structure()
    k = int(plan.export()["perm"][at])
    q = q.copy()
    q[indptr[k] + int(np.flatnonzero(indices[indptr[k]:indptr[k + 1]] == k)[0])] = -1.0
    step("front %dx%d negative pivot %d" % (M, N, at))
    with pytest.raises(nat.NotPositiveDefinite, match="lattice index %d\\)" % k):
        plan.factor(0, torch.as_tensor(q).cuda())


# one column needs no change of layout: the right-hand side must still be the caller's
@pytest.mark.parametrize("shape", [(), (1,), (2,)])
def test_solve_leaves_its_right_hand_side(shape):
    import torch
    from spdepy_amd.plan import Plan
    plan = Plan(7, 9, 2, 3)
    q, A = _spd(plan, 4)
    plan.factor(0, torch.as_tensor(q).cuda())
    b = np.random.default_rng(5).normal(size=(plan.n,) + shape)
    B = torch.as_tensor(b).cuda()
    step("solve of shape %s" % (b.shape,))
    X = plan.solve(0, B)
    assert np.array_equal(B.cpu().numpy(), b)
    assert np.abs(A @ X.cpu().numpy() - b).max() <= 1e-11 * np.abs(b).max()
