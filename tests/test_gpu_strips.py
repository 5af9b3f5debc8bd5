"""The one-column preconditioner in strips of lines against the colour-by-colour
sweeps that two equal columns take: the same few PCG iterations."""
import ctypes

import numpy as np
import pytest

from tests.gpu_util import step

pytestmark = pytest.mark.gpu


def _strips(it):
    """(lines per strip, whether the strips hold the current factor, LDS of a probe block)."""
    from spdepy_amd import _native as nat
    out = [ctypes.c_int32() for _ in range(3)]
    nat.check(nat.lib().spde_debug_ic_strips(it._h, *[ctypes.byref(x) for x in out]))
    return [x.value for x in out]


def _solver(M, N, T, bc):
    """A solver of a stationary model on the lattice, and its values of Q."""
    import spdepy_amd as sp
    from spdepy_amd import spdes
    from spdepy_amd.krylov import IterativeSolver
    ax = lambda n: (np.arange(n) + 0.5) / n
    g = sp.grid(x=ax(M), y=ax(N), t=np.arange(float(T)))
    mod0 = spdes.WhittleMatern2D(grid=sp.grid(x=ax(M), y=ax(N)), bc=bc)
    mod = spdes.AdvectionIDiffusion2D(grid=g, mod0=mod0, bc=bc)
    eng = mod._engine()
    q = eng.assemble(mod._coeffs(np.array([0.5, -0.5, 0.4, -0.3, 0.0, 4.0])))
    return IterativeSolver(eng.plan), q


# fewer lines than a strip, one and several strips, lines beside the border, long
# lines, and lines too long for the strips (colours)
@pytest.mark.parametrize("M,N,T,bc", [(5, 4, 2, 1), (7, 9, 3, 3), (16, 30, 2, 1), (33, 5, 4, 3), (4, 61, 5, 1),
                                      (100, 23, 3, 3), (12, 10, 16, 1), (3, 2, 7, 3), (230, 19, 2, 1)])
def test_strips_match_colours(M, N, T, bc):
    it, q = _solver(M, N, T, bc)
    _one_column_matches_two(it, q, M, N, T, bc)


# one slice: no odd ones, the two even sweeps alone
@pytest.mark.parametrize("M,N,bc", [(5, 4, 1), (16, 30, 3), (100, 23, 1)])
def test_strips_match_colours_on_one_slice(M, N, bc):
    import torch
    from spdepy_amd.krylov import IterativeSolver
    from spdepy_amd.plan import Plan
    plan = Plan(M, N, 1, bc)
    indptr, indices = plan.structure()
    rows = np.repeat(np.arange(plan.n), np.diff(indptr))
    # symmetric, diagonally dominant, entries that differ along a row and between rows
    q = np.where(rows == indices, 30.0, -1.0 / (1.0 + 0.01 * (rows + indices)))
    _one_column_matches_two(IterativeSolver(plan), torch.as_tensor(q).cuda(), M, N, 1, bc)


def _one_column_matches_two(it, q, M, N, T, bc):
    import torch
    step("strips %dx%dx%d bc %d" % (M, N, T, bc))
    # the route that one column takes: strips, but for the lines too long for them
    assert (_strips(it)[0] > 0) == (M != 230)
    it.factor(q, torch.full((it.n,), 50.0, dtype=torch.float64, device="cuda"))
    b = torch.as_tensor(np.random.default_rng(3).normal(size=(it.n, 1)).astype(np.float32)).cuda()
    for its in (1, 4):
        one, _ = it.solve(b, tol=1e-30, maxit=its)
        two, _ = it.solve(b.repeat(1, 2).contiguous(), tol=1e-30, maxit=its)
        a, c = one[:, 0].double(), two[:, 0].double()
        # FP32 recurrences with other orders of summation: 1e-7 an operation
        assert float((a - c).norm() / c.norm()) <= 1e-5


# The strips are filled when one column needs them, from the factor of that
# moment: not by the factorisation or for many columns, after a correction again,
# and once for a handle and its view
def test_strips_hold_the_current_factor():
    import torch
    it, q = _solver(16, 30, 4, 1)
    rng = np.random.default_rng(5)
    add = torch.full((it.n,), 50.0, dtype=torch.float64, device="cuda")
    b = torch.as_tensor(rng.normal(size=(it.n, 1)).astype(np.float32)).cuda()
    corr = torch.as_tensor(0.05 * rng.normal(size=(it.n, 22)).astype(np.float32)).cuda()
    view, other = it.view(), torch.cuda.Stream()

    def matches(solver, stream):
        with torch.cuda.stream(stream):
            one, _ = solver.solve(b, tol=1e-30, maxit=3)
            assert _strips(it)[1] == 1
            two, _ = solver.solve(b.repeat(1, 2).contiguous(), tol=1e-30, maxit=3)
            return float((one[:, 0] - two[:, 0]).norm() / two[:, 0].norm()) <= 1e-5
    step("strips filled on use")
    assert _strips(it)[1] == 0
    it.factor(q, add)
    it.solve(b.repeat(1, 64).contiguous(), tol=1e-30, maxit=1)
    assert _strips(it)[1] == 0
    assert matches(it, torch.cuda.current_stream()) and matches(view, other)
    it.correct(corr)
    assert _strips(it)[1] == 0
    assert matches(view, other) and matches(it, torch.cuda.current_stream())
    it.factor(q, 3.0 * add)
    assert _strips(it)[1] == 0
    x, info = it.replace(b[:, 0].double().contiguous(), tol=1e-8)
    assert _strips(it)[1] == 1 and info["relres"] <= 1e-8


# The reservation of the probes' blocks is for a mean that needs no LDS itself:
# strips, the line in cells, just under it, and a lattice without strips
@pytest.mark.parametrize("M,N,T,bc,lds", [(64, 64, 32, 1, 0), (64, 64, 31, 1, 32768), (16, 16, 4, 3, 32768),
                                          (66, 66, 32, 2, 32768)])
def test_probes_leave_room_for_the_strips(M, N, T, bc, lds):
    from spdepy_amd.krylov import IterativeSolver
    from spdepy_amd.plan import Plan
    it = IterativeSolver(Plan(M, N, T, bc))
    step("probe blocks %dx%dx%d bc %d" % (M, N, T, bc))
    lines, _, reserved = _strips(it)
    assert (lines > 0) == (bc != 2) and reserved == lds
