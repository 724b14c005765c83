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


@pytest.mark.parametrize("prec", ["fp64", "fp32", "bf16"])
@pytest.mark.parametrize("nd,lev,deg,adapted", [(2, 4, 3, False), (6, 2, 2, False), (3, 3, 3, True), (4, 3, 2, False)])
def test_box_steps_are_the_steps_in_another_order(kmx_gpu, prec, nd, lev, deg, adapted):
    """Steps on vectors in the sweep's order against the apply and the scaled step in element
    order: the same sums in another order.  A chunk run twice gives the same bits."""
    import torch
    from kmx import _lib
    from kmx.plan import arnoldi_step

    pde = K.diffusion_nd(nd, lev + 2 if adapted else lev)
    tab = G.hash_table_sparse_nd([lev] * nd, lev, "SG")
    if adapted:
        tab = G.refine_random(tab, lev + 2, 0.5, np.random.default_rng(1))
    mats = K.get_coeff_mats(pde, deg)
    plan = kmx_gpu.Plan(mats, tab.idx1d, deg, None, None, index_base=1, fp32=True, level_blocks=True,
                        identity=[[d != t for d in range(nd)] for t in range(nd)])
    assert plan.box_values("fp64") == 0  # not switched on
    for p in ("fp64", "fp32"):
        plan.set_sweep(p, True)
    nb, n, steps = plan.box_values(prec), plan.dof, 5
    assert nb >= n and (nb > n) == adapted
    gen = torch.Generator().manual_seed(nd)
    v = torch.randn(n, dtype=torch.float64, generator=gen).cuda()
    v /= torch.linalg.vector_norm(v)
    S = torch.rand(n, dtype=torch.float64, generator=gen).cuda() + 0.5
    back = torch.empty_like(v)
    vb = plan.to_box(v, torch.full((nb,), 7.0, dtype=torch.float64, device="cuda"), prec)
    assert torch.equal(plan.from_box(vb, back, prec), v) and int((vb == 0).sum()) == nb - n
    dt = 20 * pde.set_dt(pde, 0.01)
    V = torch.zeros((steps + 1, n), dtype=torch.float64, device="cuda")
    V[0] = v
    h, u, z = torch.zeros((steps, steps + 2), dtype=torch.float64, device="cuda"), torch.empty_like(v), S * v
    work = torch.empty(_lib.arnoldi_work(n), dtype=torch.float64, device="cuda")
    for k in range(steps):
        plan.apply(z, u, prec=prec)
        arnoldi_step(n, k, V, u, 1.0, -dt, h[k], work, scale=S, z=z)
    Vb = torch.zeros((steps + 1, nb), dtype=torch.float64, device="cuda")
    Vb[0] = vb
    Sb, zb, hb = plan.to_box(S, torch.empty_like(vb), prec), torch.empty_like(vb), torch.zeros_like(h)
    workb = torch.empty(_lib.arnoldi_work(nb), dtype=torch.float64, device="cuda")
    runs = []
    for _ in range(2):
        plan.arnoldi_box_start(Vb[0], Sb, zb, prec)
        for k in range(steps):
            plan.arnoldi_box_step(k, Vb, 1.0, -dt, Sb, zb, hb[k], workb, prec)
        runs.append((Vb.clone(), hb.clone()))
        plan.apply(v, u, prec=prec)  # the boxes hold another vector now
    assert torch.equal(runs[0][0], runs[1][0]) and torch.equal(runs[0][1], runs[1][1])
    # dots in another order, n eps, through 5 steps; a last bit of z may round the other way
    # in the product's precision, whose unit the later steps carry on
    tol = {"fp64": 1e-11, "fp32": 1e-5, "bf16": 5e-2}[prec]
    assert float((hb - h).abs().max()) <= tol * float(h.abs().max())
    for k in range(steps + 1):
        d = plan.from_box(Vb[k], back, prec) - V[k]
        assert float(d.abs().max()) <= tol * max(1.0, float(h.abs().max()))
        assert int((Vb[k] == 0).sum()) >= nb - n
    plan.set_sweep("fp32", False)
    if prec == "fp32":
        with pytest.raises(ValueError):
            plan.to_box(v, vb, prec)


def test_backward_euler_follows_the_sweep_switch(kmx_gpu):
    """The solver kept for a plan is one of its present path: switched on, off and on again."""
    import torch
    from kmx import timestep as TS

    pde = K.diffusion_nd(3, 4)
    tab = G.hash_table_sparse_nd([4] * 3, 4, "SG")
    mats = K.get_coeff_mats(pde, 2)
    plan = kmx_gpu.Plan(mats, tab.idx1d, 2, None, None, index_base=1, fp32=True, level_blocks=True,
                        identity=[[d != t for d in range(3)] for t in range(3)])
    f0 = np.random.default_rng(3).standard_normal(plan.dof)
    dt = 100 * pde.set_dt(pde, 0.01)
    M = np.eye(plan.dof) - dt * O.build_A(O.ApplyInputs(mats, tab.idx1d, 2))
    ref = np.linalg.solve(M, f0)
    bound = 2e-12 * np.linalg.norm(f0) / np.linalg.svd(M, compute_uv=False)[-1]
    for on in (True, False, True):
        for p in ("fp64", "fp32"):
            plan.set_sweep(p, on)
        for _ in range(2):
            f1, hist, _ = TS.backward_euler(plan, torch.from_numpy(f0).cuda(), dt, tol=1e-12)
            assert hist[-1] <= 1e-12
            assert np.linalg.norm(f1.cpu().numpy() - ref) <= bound


@pytest.mark.parametrize("sweep", [False, True])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_backward_euler_follows_its_operator(kmx_gpu, sweep, prec):
    """One kept solver through changes of the operator between its steps: term scales (launch
    arguments of the pair kernels), a matrix of the same zero blocks and one of others (new
    storage of a separable sweep).  Each step takes the inner steps that a plan made for that
    operator takes, and solves its system."""
    import torch
    from kmx import timestep as TS

    pde = K.diffusion_nd(3, 3)
    tab = G.hash_table_sparse_nd([3] * 3, 3, "SG")
    mats = [list(m) for m in K.get_coeff_mats(pde, 2)]
    scales = [1.0] * 3
    n = mats[0][0].shape[0]

    def make():
        p = kmx_gpu.Plan(mats, tab.idx1d, 2, None, None, index_base=1, fp32=True, level_blocks=sweep,
                         identity=[[d != t for d in range(3)] for t in range(3)] if sweep else None)
        if sweep:
            for q in ("fp64", "fp32"):
                p.set_sweep(q, True)
        for t, s in enumerate(scales):
            p.set_term_scale(t, s)
        return p

    def step(p):
        f1, hist, inner = TS.backward_euler(p, torch.from_numpy(f0).cuda(), dt, tol=1e-12, inner_prec=prec)
        assert hist[-1] <= 1e-12
        A = O.build_A(O.ApplyInputs([[s * m[0]] + m[1:] for s, m in zip(scales, mats)], tab.idx1d, 2))
        M = np.eye(p.dof) - dt * A
        bound = 2e-12 * np.linalg.norm(f0) / np.linalg.svd(M, compute_uv=False)[-1]
        assert np.linalg.norm(f1.cpu().numpy() - np.linalg.solve(M, f0)) <= bound
        return inner

    plan = make()
    f0 = np.random.default_rng(5).standard_normal(plan.dof)
    dt = 100 * pde.set_dt(pde, 0.01)
    state = plan.replay_state(prec)
    seen = [step(plan)]
    assert plan.replay_state(prec) == state
    for change in ("scales", "values", "blocks", "scales back"):
        if change == "scales":
            scales[:] = [0.25, 1.0, 0.5]
        elif change == "scales back":
            scales[:] = [1.0] * 3
        else:
            mats[1][1] = 0.5 * mats[1][1] if change == "values" else -40.0 * np.eye(n)
            plan.update_term(1, 1, mats[1][1])
        for t, s in enumerate(scales):
            plan.set_term_scale(t, s)
        assert step(plan) == step(make())
    assert len(TS._SOLVERS[plan]) == 1


@pytest.mark.parametrize("nd,lev,deg", [(1, 9, 2), (1, 9, 3), (1, 7, 4), (2, 7, 3), (2, 6, 4), (3, 6, 2), (3, 5, 3),
                                        (3, 4, 4), (4, 4, 2), (5, 4, 2), (6, 3, 2)])
def test_scaling_costs_no_inner_steps(kmx_gpu, monkeypatch, nd, lev, deg):
    """Diffusion, which the scaling helps least: against the unscaled solver's inner steps over
    steps of 3, 30 and 100 explicit limits, no more of them (a chance step or two of one solve
    aside: 3 of a hundred)."""
    import torch
    from kmx import timestep as TS

    pde = K.diffusion_nd(nd, lev)
    tab = G.hash_table_sparse_nd([lev] * nd, lev, "SG")
    plan = kmx_gpu.Plan(K.get_coeff_mats(pde, deg), tab.idx1d, deg, None, None, index_base=1, fp32=True,
                        level_blocks=True, identity=[[d != t for d in range(nd)] for t in range(nd)])
    for p in ("fp64", "fp32"):
        if plan.sweep(p)["available"]:  # (1D operators have none)
            plan.set_sweep(p, True)
    fs = [torch.from_numpy(np.random.default_rng(s).standard_normal(plan.dof)).cuda() for s in range(2)]

    def steps():
        TS._SOLVERS.pop(plan, None)
        return sum(TS.backward_euler(plan, f, x * pde.set_dt(pde, 0.01), tol=1e-12)[2] for x in (3, 30, 100) for f in fs)

    scaled = steps()
    monkeypatch.setattr(TS, "scale_power", lambda nd, deg: 0.0)
    assert scaled <= 1.03 * steps()


@pytest.mark.parametrize("power", [-0.75, -0.5, -0.25, 1.0])
def test_stiff_scale_is_a_power_of_the_diagonal(kmx_gpu, power):
    """Against torch, 8 ulps of pow's; in the sweep's order the same values, 0 in absent cells."""
    import torch

    tab = G.refine_random(G.hash_table_sparse_nd([3] * 3, 3, "SG"), 5, 0.5, np.random.default_rng(1))
    pde = K.diffusion_nd(3, 5)
    plan = kmx_gpu.Plan(K.get_coeff_mats(pde, 3), tab.idx1d, 3, None, None, index_base=1, fp32=True, level_blocks=True,
                        identity=[[d != t for d in range(3)] for t in range(3)])
    work = torch.empty(plan.dof, dtype=torch.float64, device="cuda")
    for dt in (-3.0, 0.0, 100 * pde.set_dt(pde, 0.01)):
        want = (1.0 - dt * plan.diagonal()).clamp(min=1.0).pow(power)
        got = plan.stiff_scale(dt, power, work, torch.empty_like(work))
        assert float(((got - want) / want).abs().max()) <= 8 * 2.3e-16
        assert torch.equal(plan.stiff_scale(dt, power, work, work), got)
        for p in ("fp64", "fp32"):
            plan.set_sweep(p, True)
            nb = plan.box_values(p)
            assert nb > plan.dof
            box = plan.stiff_scale(dt, power, work, torch.full((nb,), 7.0, dtype=torch.float64, device="cuda"), p)
            assert torch.equal(box, plan.to_box(got, torch.empty_like(box), p))
            plan.set_sweep(p, False)
    with pytest.raises(ValueError):
        plan.stiff_scale(1.0, power, work, work[:-1].clone())
    with pytest.raises(ValueError):
        plan.stiff_scale(1.0, power, work, torch.empty_like(work), "fp32")  # no sweep on
