"""The factored FP64 apply (kmx_factor.hip) against the CPU oracle and the pair kernels,
at sizes below the rule that picks it (KMX_FACTOR_MIN_FMA=0), through the C ABI.

Bars: 1e-13 relative (2-norm) to the oracle, the bar of every FP64 apply (sums of at most
P T deg^d products, random operands: a few eps (P T deg^d / N)^(1/2), below 1e-14 here)."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def everywhere(monkeypatch):
    monkeypatch.setenv("KMX_FACTOR_MIN_FMA", "0")


def rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def case(nd, lev, deg, T, conn, seed, shared=False):
    rng = np.random.default_rng(seed)
    if conn:
        h = O.hash_table_nd(nd, lev, "SG")
        rp, cols = O.connect_nd(nd, lev, "SG", lev, lev)
    else:
        h = O.hash_table_sparse_nd([lev] * nd, max(lev, 1), "SG")
        rp = cols = None
    n = deg * 2 ** lev
    mats = [[rng.standard_normal((n, n)) for _ in range(nd)] for _ in range(T)]
    if shared:  # terms acting in one dimension each, one matrix per dimension in all the others
        common = [rng.standard_normal((n, n)) for _ in range(nd)]
        mats = [[m if d == t % nd else common[d] for d, m in enumerate(tm)] for t, tm in enumerate(mats)]
    idx = np.asarray(h["idx1d"])
    return mats, idx, rp, cols, rng.standard_normal(idx.shape[0] * deg ** nd)


SHAPES = [
    (2, 3, 2, 2, True), (2, 4, 3, 3, False), (2, 5, 4, 2, True), (2, 3, 5, 1, False), (2, 7, 2, 4, False),
    (3, 3, 2, 3, True), (3, 4, 3, 3, True), (3, 2, 4, 2, False), (3, 5, 2, 2, False),
    (4, 3, 2, 4, True), (4, 2, 2, 1, False), (5, 2, 2, 5, True), (5, 3, 2, 2, False), (6, 2, 2, 6, True),
    (6, 1, 2, 3, False),
]


@pytest.mark.parametrize("nd,lev,deg,T,conn", SHAPES)
@pytest.mark.parametrize("shared", [False, True])
def test_matches_oracle_forward_and_adjoint(kmx_gpu, nd, lev, deg, T, conn, shared):
    import torch

    mats, idx, rp, cols, x = case(nd, lev, deg, T, conn, nd * 100 + lev * 10 + deg, shared)
    plan = kmx_gpu.Plan(mats, idx, deg, rp, cols, index_base=1, adjoint=True)
    scales = np.random.default_rng(1).uniform(0.5, 2.0, size=T)
    for t, s in enumerate(scales):
        plan.set_term_scale(t, s)
    scaled = [[scales[t] * m if d == 0 else m for d, m in enumerate(tm)] for t, tm in enumerate(mats)]
    xd = torch.from_numpy(x).cuda()
    y = plan.apply(xd).cpu().numpy()
    assert rel(y, O.apply_A(O.ApplyInputs(scaled, idx, deg, rp, cols), x, nthreads=8)) <= 1e-13
    # the adjoint is the operator of the transposed matrices over the transposed (symmetric) pair list
    tr = [[np.ascontiguousarray(m.T) for m in tm] for tm in scaled]
    yt = plan.apply_transpose(xd).cpu().numpy()
    assert rel(yt, O.apply_A(O.ApplyInputs(tr, idx, deg, rp, cols), x, nthreads=8)) <= 1e-13
    # a new matrix (its class of equal prefixes may change), then the old one again
    new = np.random.default_rng(2).standard_normal(mats[0][0].shape)
    plan.update_term(0, 0, new)
    scaled[0][0] = scales[0] * new
    y2 = plan.apply(xd).cpu().numpy()
    assert rel(y2, O.apply_A(O.ApplyInputs(scaled, idx, deg, rp, cols), x, nthreads=8)) <= 1e-13
    plan.update_term(0, 0, mats[0][0])
    assert np.array_equal(plan.apply(xd).cpu().numpy(), y)


def test_lists_that_are_no_product_run_pair_by_pair(kmx_gpu):
    """One pair taken out of, or repeated in, a product list; and elements given twice."""
    import torch

    mats, idx, rp, cols, x = case(2, 4, 2, 2, True, 5)
    rp, cols = np.asarray(rp).copy(), np.asarray(cols).copy()
    drop, dup = 7, 11
    c1, r1 = np.delete(cols, drop), rp - (rp > drop)
    c2, r2 = np.insert(cols, dup, cols[dup]), rp + (rp > dup)
    for rr, cc in ((r1, c1), (r2, c2)):
        y = kmx_gpu.Plan(mats, idx, 2, rr, cc, index_base=1).apply(torch.from_numpy(x).cuda()).cpu().numpy()
        assert rel(y, O.apply_A(O.ApplyInputs(mats, idx, 2, rr, cc), x)) <= 1e-13
    twice = np.vstack([idx, idx[:3]])
    x2 = np.random.default_rng(3).standard_normal(twice.shape[0] * 4)
    y = kmx_gpu.Plan(mats, twice, 2, None, None, index_base=1).apply(torch.from_numpy(x2).cuda()).cpu().numpy()
    assert rel(y, O.apply_A(O.ApplyInputs(mats, twice, 2), x2)) <= 1e-13


@pytest.mark.parametrize("nd,lev,deg,conn", [(2, 4, 3, True), (3, 3, 3, True), (6, 1, 2, True), (2, 4, 4, False)])
@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
def test_non_finite_inputs_reach_connected_rows_only(kmx_gpu, monkeypatch, nd, lev, deg, conn, value):
    """y is not finite exactly where the pair kernels' is, with the same values there, and
    elsewhere equal to 1e-13."""
    import torch

    mats, idx, rp, cols, x = case(nd, lev, deg, 2, conn, 9)
    x[(idx.shape[0] - 1) * deg ** nd + 1] = value  # in the last element: a high level, few connections
    xd = torch.from_numpy(x).cuda()
    y = kmx_gpu.Plan(mats, idx, deg, rp, cols, index_base=1).apply(xd).cpu().numpy()
    monkeypatch.setenv("KMX_FACTOR_MIN_FMA", "1e300")
    ref = kmx_gpu.Plan(mats, idx, deg, rp, cols, index_base=1).apply(xd).cpu().numpy()
    fin = np.isfinite(ref)
    assert np.array_equal(fin, np.isfinite(y)) and np.array_equal(y[~fin], ref[~fin], equal_nan=True)
    assert not fin.all() and (not fin.any() or rel(y[fin], ref[fin]) <= 1e-13)


def test_streams_threads_and_capture(kmx_gpu):
    """Applies of one plan from two streams and two threads, interleaved, and under graph
    capture, each against its own result alone (the workspace is the plan's)."""
    import threading

    import torch

    mats, idx, rp, cols, _ = case(3, 4, 3, 3, True, 4)
    plan = kmx_gpu.Plan(mats, idx, 3, rp, cols, index_base=1)
    xs = [torch.randn(plan.dof, dtype=torch.float64, device="cuda") for _ in range(2)]
    want = [plan.apply(x).clone() for x in xs]
    torch.cuda.synchronize()
    out = [[torch.empty_like(x) for _ in range(20)] for x in xs]

    def work(k):
        st = torch.cuda.Stream()
        with torch.cuda.stream(st):
            for y in out[k]:
                plan.apply(xs[k], y)
        st.synchronize()

    th = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    for k in range(2):
        assert all(torch.equal(y, want[k]) for y in out[k])
    y = torch.empty_like(xs[0])
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        plan.apply(xs[0], y)
    for x in (xs[1], xs[1] * 2):
        xs[0].copy_(x)
        ref = plan.apply(x)
        g.replay()
        torch.cuda.synchronize()
        assert float((y - ref).norm() / ref.norm()) <= 1e-13


def test_apply_while_the_last_stream_records_a_graph(kmx_gpu):
    """The stream of the last apply records a graph now: an apply on another stream runs at
    once, outside the graph."""
    import torch

    mats, idx, rp, cols, _ = case(3, 3, 2, 2, True, seed=5)
    plan = kmx_gpu.Plan(mats, idx, 2, rp, cols)
    x = torch.from_numpy(np.random.default_rng(1).standard_normal(plan.dof)).cuda()
    ref = plan.apply(x).clone()
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    outs = [torch.zeros_like(x) for _ in range(3)]
    torch.cuda.synchronize()
    with torch.cuda.stream(a):
        plan.apply(x, outs[0])
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=a):
        plan.apply(x, outs[1])
        with torch.cuda.stream(b):
            plan.apply(x, outs[2])
    b.synchronize()
    assert rel(outs[2].cpu().numpy(), ref.cpu().numpy()) <= 1e-13
    assert not outs[1].any()
    for _ in range(3):
        outs[2].zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert rel(outs[1].cpu().numpy(), ref.cpu().numpy()) <= 1e-13
        assert not outs[2].any()


@pytest.mark.parametrize("nd,lev,deg,T,conn", SHAPES + [(2, 4, 3, 2, True), (3, 3, 3, 2, True), (2, 4, 4, 2, False),
                                                        (3, 3, 2, 2, True)])
def test_which_plans_take_the_factored_form(kmx_gpu, monkeypatch, nd, lev, deg, T, conn):
    """The plans of the tests above run the kernels that they are about: every shape but 2D
    deg 5 (which no rule picks), with or without an adjoint; not below the size rule, and not
    while a sweep is on."""
    mats, idx, rp, cols, _ = case(nd, lev, deg, T, conn, 3)
    has = (nd, deg) != (2, 5)
    for adjoint in (False, True):
        plan = kmx_gpu.Plan(mats, idx, deg, rp, cols, index_base=1, adjoint=adjoint)
        assert plan.factored() == has and plan.factored(transpose=True) == (has and adjoint)
        plan.update_term(0, 0, mats[0][0] + 1.0)
        plan.set_term_scale(0, 0.5)
        assert plan.factored() == has
    monkeypatch.setenv("KMX_FACTOR_MIN_FMA", "1e300")
    assert not kmx_gpu.Plan(mats, idx, deg, rp, cols, index_base=1).factored()


def test_which_lists_take_the_factored_form(kmx_gpu):
    mats, idx, rp, cols, _ = case(2, 4, 2, 2, True, 5)
    rp, cols = np.asarray(rp), np.asarray(cols)
    make = lambda i, r, c, **kw: kmx_gpu.Plan(mats, i, 2, r, c, index_base=1, **kw)
    assert make(idx, rp, cols).factored()
    assert not make(idx, rp - (rp > 7), np.delete(cols, 7)).factored()
    assert not make(idx, rp + (rp > 11), np.insert(cols, 11, cols[11])).factored()
    assert make(idx, None, None).factored()
    assert not make(np.vstack([idx, idx[:3]]), None, None).factored()
    general = make(idx, rp, cols, level_blocks=True)  # random factors: a sweep of the general form
    assert general.factored()
    general.set_sweep("fp64", True)
    assert not general.factored()
    general.set_sweep("fp64", False)
    assert general.factored()


def test_the_size_rule_picks_the_large_plans(kmx_gpu, monkeypatch):
    """By the rule itself: a 3D level 7 run's plan is factored, a 2D level 3 one is not."""
    monkeypatch.delenv("KMX_FACTOR_MIN_FMA")
    for nd, lev, deg, T, want in ((3, 7, 2, 6, True), (2, 3, 2, 2, False)):
        mats, idx, _, _, _ = case(nd, lev, deg, T, False, 1)
        assert kmx_gpu.Plan(mats, idx, deg, None, None, index_base=1).factored() == want


def test_autotune_decides_for_its_own_plan(kmx_gpu):
    """A plan on which the pair kernels are faster gives the factored form up; what it leaves
    for later plans of its kind is the pair kernels' variant alone."""
    import torch

    mats, idx, rp, cols, x = case(2, 3, 2, 2, True, 6)  # far below the size rule
    plan, other = (kmx_gpu.Plan(mats, idx, 2, rp, cols, index_base=1, adjoint=True) for _ in range(2))
    xd = torch.from_numpy(x).cuda()
    want = [plan.apply(xd).cpu().numpy(), plan.apply_transpose(xd).cpu().numpy()]
    plan.autotune()
    assert not plan.factored() and not plan.factored(transpose=True)
    assert rel(plan.apply(xd).cpu().numpy(), want[0]) <= 1e-13
    assert rel(plan.apply_transpose(xd).cpu().numpy(), want[1]) <= 1e-13
    plan.update_term(0, 0, mats[0][0])
    plan.autotune()
    assert rel(plan.apply(xd).cpu().numpy(), want[0]) <= 1e-13
    assert other.factored() and other.factored(transpose=True)
    later = kmx_gpu.Plan(mats, idx, 2, rp, cols, index_base=1, adjoint=True)
    assert later.factored() and later.factored(transpose=True)
    assert np.array_equal(later.apply(xd).cpu().numpy(), want[0])


@pytest.mark.parametrize("nd,lev,deg,T,conn", [(3, 3, 3, 3, True), (6, 1, 2, 6, False), (2, 4, 2, 4, True)])
def test_matrices_that_split_and_join_classes(kmx_gpu, nd, lev, deg, T, conn):
    """Terms that share matrices share partial sums.  Matrices replaced one by one until no
    two terms share any, and back: more sums than the plan began with, the same ones again."""
    import torch

    mats, idx, rp, cols, x = case(nd, lev, deg, T, conn, 8, shared=True)
    plan = kmx_gpu.Plan(mats, idx, deg, rp, cols, index_base=1, adjoint=True)
    xd = torch.from_numpy(x).cuda()
    first = [plan.apply(xd).clone(), plan.apply_transpose(xd).clone()]
    rng = np.random.default_rng(4)
    now = [list(tm) for tm in mats]

    def check():
        assert plan.factored() and plan.factored(transpose=True)
        for y, ms in ((plan.apply(xd), now), (plan.apply_transpose(xd), [[m.T.copy() for m in tm] for tm in now])):
            assert rel(y.cpu().numpy(), O.apply_A(O.ApplyInputs(ms, idx, deg, rp, cols), x, nthreads=8)) <= 1e-13

    for t in range(T):
        for d in range(nd):
            if d != t % nd:
                now[t][d] = rng.standard_normal(mats[t][d].shape)
                plan.update_term(t, d, now[t][d])
        check()
    for t in reversed(range(T)):
        for d in range(nd):
            now[t][d] = mats[t][d]
            plan.update_term(t, d, mats[t][d])
    check()
    assert torch.equal(plan.apply(xd), first[0]) and torch.equal(plan.apply_transpose(xd), first[1])


def test_more_streams_than_workspaces(kmx_gpu):
    """Six streams in turn, in blocks and from threads: the bits of an apply alone; again
    after a matrix that splits a class (workspaces made anew), and while a graph is recorded."""
    import threading

    import torch

    mats, idx, rp, cols, _ = case(3, 4, 3, 3, True, 4, shared=True)
    plan = kmx_gpu.Plan(mats, idx, 3, rp, cols, index_base=1, adjoint=True)
    streams = [torch.cuda.Stream() for _ in range(6)]
    xs = [torch.randn(plan.dof, dtype=torch.float64, device="cuda") for _ in streams]
    for split in (False, True):
        if split:
            plan.update_term(2, 0, np.random.default_rng(2).standard_normal(mats[2][0].shape))
        assert plan.factored()
        want = [plan.apply(x).clone() for x in xs]
        wantT = [plan.apply_transpose(x).clone() for x in xs]
        out = [[torch.zeros_like(x) for _ in range(12)] for x in xs]
        torch.cuda.synchronize()
        for q in range(4):  # in turn
            for k, s in enumerate(streams):
                plan.apply(xs[k], out[k][q], stream=s)
        for k, s in enumerate(streams):  # in blocks
            for q in range(4, 8):
                plan.apply_transpose(xs[k], out[k][q], stream=s)

        def work(k):
            for q in range(8, 12):
                plan.apply(xs[k], out[k][q], stream=streams[k])

        torch.cuda.synchronize()
        th = [threading.Thread(target=work, args=(k,)) for k in range(6)]
        for t in th:
            t.start()
        for t in th:
            t.join()
        torch.cuda.synchronize()
        for k in range(6):
            for q in range(12):
                assert torch.equal(out[k][q], wantT[k] if 4 <= q < 8 else want[k]), (split, k, q)
    fresh = kmx_gpu.Plan(mats, idx, 3, rp, cols, index_base=1)
    ref = fresh.apply(xs[0]).clone()
    graph, a, b = torch.cuda.CUDAGraph(), torch.zeros_like(ref), torch.zeros_like(ref)
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        fresh.apply(xs[0], a)
        fresh.apply(xs[0], b, stream=streams[1])  # its first apply there: a workspace of its own
    streams[1].synchronize()
    assert torch.equal(b, ref) and not a.any()
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert float((a - ref).norm() / ref.norm()) <= 1e-13


def test_pair_lists_of_long_runs(kmx_gpu):
    """Rows of whole 64-column runs: a pair listed twice in place of its neighbour, or the next
    word's, is no product; the same columns in another order are one."""
    import torch

    mats, idx, rp, cols, x = case(2, 6, 2, 2, True, 12)
    rp, cols = np.asarray(rp), np.asarray(cols)
    row = int(np.flatnonzero(np.diff(rp) == len(idx))[0])  # connected to every element
    at = int(rp[row])
    assert len(idx) > 192 and np.array_equal(cols[at:at + len(idx)], np.arange(1, len(idx) + 1))
    xd = torch.from_numpy(x).cuda()
    for k, c in ((64, 65), (100, 99), (127, 127), (63, 64), (130, 190)):  # cols[k] is k + 1
        bad = cols.copy()
        bad[at + k] = c + (c == k + 1)
        plan = kmx_gpu.Plan(mats, idx, 2, rp, bad, index_base=1)
        assert not plan.factored()
        y = plan.apply(xd).cpu().numpy()
        assert rel(y, O.apply_A(O.ApplyInputs(mats, idx, 2, rp, bad), x)) <= 1e-13
    want = kmx_gpu.Plan(mats, idx, 2, rp, cols, index_base=1)
    assert want.factored()
    for a, b in ((64, 127), (70, 71), (10, 150)):
        other = cols.copy()
        other[[at + a, at + b]] = other[[at + b, at + a]]
        plan = kmx_gpu.Plan(mats, idx, 2, rp, other, index_base=1)
        assert plan.factored() and torch.equal(plan.apply(xd), want.apply(xd))
