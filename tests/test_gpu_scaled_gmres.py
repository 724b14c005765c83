"""The operator's diagonal and the scaled Arnoldi step behind backward Euler's GMRES
(time_advance.m:328-349's system), against the assembled operator and the plain step."""
import numpy as np
import pytest

import oracle as O
from kmx import coeffs as K
from kmx import grid as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nd,lev,deg,T,conn", [(1, 4, 3, 2, False), (2, 3, 5, 2, True), (3, 2, 3, 3, True),
                                               (4, 2, 2, 1, False), (6, 1, 2, 2, True), (2, 1, 1, 1, False)])
def test_diagonal_equals_the_assembled_one(kmx_gpu, nd, lev, deg, T, conn):
    rng = np.random.default_rng(nd + deg)
    h = O.hash_table_nd(nd, lev, "SG") if conn else O.hash_table_sparse_nd([lev] * nd, lev, "SG")
    rp, cols = O.connect_nd(nd, lev, "SG", lev, lev) if conn else (None, None)
    n = deg * 2 ** lev
    mats = [[rng.standard_normal((n, n)) for _ in range(nd)] for _ in range(T)]
    plan = kmx_gpu.Plan(mats, h["idx1d"], deg, rp, cols)
    scales = [0.5 + t for t in range(T)]
    for t, s in enumerate(scales):
        plan.set_term_scale(t, s)
    scaled = [[m * (scales[t] if d == 0 else 1.0) for d, m in enumerate(row)] for t, row in enumerate(mats)]
    A = O.build_A(O.ApplyInputs(scaled, h["idx1d"], deg, rp, cols))
    size = sum(np.prod([np.abs(m).max() for m in row]) for row in scaled)
    # T sums of nd products and a scale: a few roundings of the largest product
    assert np.abs(plan.diagonal().cpu().numpy() - np.diag(A)).max() <= (nd + T + 2) * 2.3e-16 * size


def test_diagonal_where_the_list_leaves_elements_out_of_their_own_row(kmx_gpu):
    rng = np.random.default_rng(0)
    mats = [[rng.standard_normal((16, 16)) for _ in range(2)]]
    idx = O.hash_table_sparse_nd([3, 3], 3, "SG")["idx1d"]
    n = len(idx)
    rows = [[j for j in range(n) if (i + j) % 3 or i % 2] for i in range(n)]
    rp = np.concatenate([[0], np.cumsum([len(r) for r in rows])])
    plan = kmx_gpu.Plan(mats, idx, 2, rp, np.concatenate(rows) + 1)
    full = kmx_gpu.Plan(mats, idx, 2).diagonal().cpu().numpy().reshape(n, -1)
    own = np.array([i in r for i, r in enumerate(rows)])
    assert own.any() and not own.all()
    assert np.array_equal(plan.diagonal().cpu().numpy().reshape(n, -1), full * own[:, None])


@pytest.mark.parametrize("n,k", [(1, 0), (300, 0), (300, 5), (32768, 30), (32769, 30), (40000, 3), (2000, 126),
                                 (2000, 127), (256, 61)])
def test_scaled_step_is_the_plain_step_on_the_scaled_vector(kmx_gpu, n, k):
    """w = s0 z + s1 u is the plain step with s0 = 0 and u' = s0 z + s1 u, bit for bit (both
    sums are one rounding of each product and of the sum), and z = S v_{k+1}."""
    import torch
    from kmx import _lib
    from kmx.plan import arnoldi_step

    gen = torch.Generator().manual_seed(n + k)
    V = torch.linalg.qr(torch.randn(n, min(n, k + 1), dtype=torch.float64, generator=gen))[0].t().contiguous()
    V = torch.cat([V, torch.zeros(k + 2 - V.shape[0], n, dtype=torch.float64)]).cuda()
    u = torch.randn(n, dtype=torch.float64, generator=gen).cuda()
    S = torch.rand(n, dtype=torch.float64, generator=gen).cuda() + 0.1
    z = S * V[k]
    outs = []
    for scaled in (True, False):
        Vd, h = V.clone(), torch.zeros(k + 2, dtype=torch.float64, device="cuda")
        work = torch.zeros(_lib.arnoldi_work(n), dtype=torch.float64, device="cuda")
        zd = z.clone()
        if scaled:
            arnoldi_step(n, k, Vd, u, 0.0, 0.25, h, work, scale=S, z=zd)
            assert torch.equal(zd, S * Vd[k + 1])
        else:
            arnoldi_step(n, k, Vd, u, 0.0, 0.25, h, work)
        outs.append((Vd, h))
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
    # with s0: against the same step in numpy
    zd, h = z.clone(), torch.zeros(k + 2, dtype=torch.float64, device="cuda")
    Vd, work = V.clone(), torch.zeros(_lib.arnoldi_work(n), dtype=torch.float64, device="cuda")
    arnoldi_step(n, k, Vd, u, 1.5, -0.25, h, work, scale=S, z=zd)
    w = (1.5 * z - 0.25 * u).cpu().numpy()
    Q = V[:k + 1].cpu().numpy()
    h1 = Q @ w
    assert np.abs(h.cpu().numpy()[:k + 1] - h1).max() <= 1e-12 * max(1.0, np.linalg.norm(w))


@pytest.mark.parametrize("pde,nd,lev,deg,factor", [(K.continuity2, 2, 4, 3, 50.0), (K.diffusion_nd, 3, 3, 2, 200.0),
                                                   (K.advection_diffusion_varcoeff, 2, 4, 3, 0.5)])
def test_backward_euler_against_a_dense_solve(kmx_gpu, pde, nd, lev, deg, factor):
    """Stiff and mild steps, with term scales changed between two steps of one solver."""
    import torch
    from kmx import timestep as TS

    spec = pde(lev) if pde is K.continuity2 else pde(nd, lev)
    mats = K.get_coeff_mats(spec, deg)
    tab = G.hash_table_sparse_nd([lev] * nd, lev, "SG")
    plan = kmx_gpu.Plan(mats, tab.idx1d, deg, None, None, index_base=1, fp32=True)
    f0 = np.random.default_rng(2).standard_normal(plan.dof)
    dt = factor * spec.set_dt(spec, 0.01)
    for s in (1.0, 0.5):
        for t in range(len(mats)):
            plan.set_term_scale(t, s)
        f1, hist, _ = TS.backward_euler(plan, torch.from_numpy(f0).cuda(), dt, tol=1e-12, inner_prec="fp64")
        assert hist[-1] <= 1e-12
        M = np.eye(plan.dof) - dt * s * O.build_A(O.ApplyInputs(mats, tab.idx1d, deg))
        ref = np.linalg.solve(M, f0)
        # |f1 - ref| <= |M^-1| |r|
        bound = 2e-12 * np.linalg.norm(f0) / np.linalg.svd(M, compute_uv=False)[-1]
        assert np.linalg.norm(f1.cpu().numpy() - ref) <= bound
        TS._SOLVERS.pop(plan)  # (a captured product keeps the scales it was captured with)
