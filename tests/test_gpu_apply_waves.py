"""Blocks beyond the register kernels, a wave per pair (k_apply_waves) and, above 256 values,
a workgroup per pair, against the oracle: FP64 1e-13, FP32 5e-6 relative (2-norm)."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


@pytest.mark.parametrize("nd,lev,deg,T,conn", [
    (2, 3, 6, 2, True), (2, 2, 7, 1, False), (2, 3, 8, 3, False), (3, 2, 5, 2, True), (3, 1, 6, 1, False),
    (4, 2, 3, 16, True), (4, 3, 3, 2, False), (4, 1, 4, 2, True), (5, 1, 3, 2, False), (5, 1, 3, 1, True),
    (3, 1, 7, 1, False), (6, 1, 3, 1, True),  # 343 and 729 values
])
def test_matches_oracle(kmx_gpu, nd, lev, deg, T, conn):
    import torch

    rng = np.random.default_rng(nd * 10 + deg)
    h = O.hash_table_nd(nd, lev, "SG") if conn else O.hash_table_sparse_nd([lev] * nd, max(lev, 1), "SG")
    rp, cols = O.connect_nd(nd, lev, "SG", lev, lev) if conn else (None, None)
    n = deg * 2 ** lev
    mats = [[rng.standard_normal((n, n)) for _ in range(nd)] for _ in range(T)]
    plan = kmx_gpu.Plan(mats, h["idx1d"], deg, rp, cols, adjoint=True)
    x = rng.standard_normal(plan.dof)
    xd = torch.from_numpy(x).cuda()
    ref = O.apply_A(O.ApplyInputs(mats, h["idx1d"], deg, rp, cols), x)
    assert rel(plan.apply(xd).cpu().numpy(), ref) <= 1e-13
    assert rel(plan.apply(xd, prec="fp32").cpu().numpy(), ref) <= 5e-6
    # <A x, z> = <x, A' z>
    z = torch.from_numpy(rng.standard_normal(plan.dof)).cuda()
    for prec, tol in (("fp64", 1e-12), ("fp32", 5e-5)):
        a, b = plan.apply(xd, prec=prec), plan.apply_transpose(z, prec=prec)
        scale = float(a.norm() * z.norm() + xd.norm() * b.norm())
        assert abs(float(a @ z) - float(xd @ b)) <= tol * scale
    again = plan.apply(xd)
    assert torch.equal(again, plan.apply(xd))


def test_rows_of_no_and_few_pairs(kmx_gpu):
    """Fewer pairs than waves, none at all, and unordered lists with a pair listed twice."""
    import torch

    rng = np.random.default_rng(2)
    idx = O.hash_table_sparse_nd([2] * 4, 2, "SG")["idx1d"]
    n = len(idx)
    rows = [list(rng.integers(0, n, size=i % 20)) for i in range(n)]
    rp = np.concatenate([[0], np.cumsum([len(r) for r in rows])])
    cols = np.concatenate([np.asarray(r, dtype=np.int64) for r in rows]) + 1
    mats = [[rng.standard_normal((12, 12)) for _ in range(4)] for _ in range(2)]
    plan = kmx_gpu.Plan(mats, idx, 3, rp, cols)
    x = rng.standard_normal(plan.dof)
    y = plan.apply(torch.from_numpy(x).cuda()).cpu().numpy()
    assert rel(y, O.apply_A(O.ApplyInputs(mats, idx, 3, rp, cols), x)) <= 1e-13
    assert not y[:81].any()
