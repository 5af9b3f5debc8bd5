"""Solutions of more than 4 GiB (first of the GPU tests by name: the plans that later
ones keep leave no room for it)."""
import pytest

from tests.gpu_util import step

pytestmark = pytest.mark.gpu


def test_many_columns_on_a_long_lattice():
    """64 right-hand sides at n = 8.6 million, where the last columns of a tile of
    the solution lie more than 4 GiB behind its first: each is solved like the others."""
    import torch
    from spdepy_amd.plan import Plan
    if torch.cuda.mem_get_info()[0] < 80e9:
        pytest.skip("needs 80 GB of device memory: other tests' plans hold it")
    plan = Plan(2, 4300000, 1, 3, nslots=1)
    indptr, indices = plan.structure()
    step("values at n = %d" % plan.n)
    ip, ix = torch.as_tensor(indptr).cuda(), torch.as_tensor(indices).cuda()
    rows = torch.repeat_interleave(torch.arange(plan.n, device="cuda", dtype=torch.int32), ip[1:] - ip[:-1])
    q = torch.where(rows == ix, 30.0, -1.0).double()      # diagonally dominant: at most 24 neighbours
    del ip, ix, rows
    plan.factor(0, q)
    B = torch.randn((plan.n, 64), dtype=torch.float64, device="cuda",
                    generator=torch.Generator(device="cuda").manual_seed(0))
    step("64 columns at n = %d" % plan.n)
    X = plan.solve(0, B)
    for c in (0, 31, 60, 61, 62, 63):
        r = plan.spmv(q, X[:, c].contiguous()) - B[:, c]
        # condition below 10, a few dozen operations an entry: some 1e-15 of the column
        assert float(r.norm() / B[:, c].norm()) <= 1e-13, c
    del plan, q, B, X, r
    torch.cuda.empty_cache()
