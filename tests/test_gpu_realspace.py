"""GPU wavelet -> real space transform (wavelet_to_realspace.m) against the
oracle's restatement (per element kron_multd with rectangular column blocks,
summed).  FP64 bar 1e-13 relative (2-norm)."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def run_case(kmx, meval, idx, deg, seed):
    import torch

    rng = np.random.default_rng(seed)
    fw = rng.standard_normal(idx.shape[0] * deg ** len(meval))
    ref = O.wavelet_to_realspace(meval, idx, deg, fw)
    rs = kmx.RealSpace(meval, idx, deg)
    fr = rs.apply(torch.from_numpy(fw).cuda()).cpu().numpy()
    rs.destroy()
    return rel(fr, ref)


@pytest.mark.parametrize(
    "nd,lev,deg,oldhash",
    [(1, 8, 7, False), (2, 4, 3, False), (2, 5, 2, True), (3, 3, 4, False), (3, 4, 2, True), (4, 3, 2, False)],
)
def test_realspace_matches_oracle(kmx_gpu, nd, lev, deg, oldhash):
    rng = np.random.default_rng(nd * 100 + lev)
    h = O.hash_table_nd(nd, lev, "SG") if oldhash else O.hash_table_sparse_nd([lev] * nd, lev, "SG")
    n = deg * 2 ** lev
    npts = [max(3, n // (1 + d)) + d for d in range(nd)]  # rectangular, uneven per dim
    meval = [rng.standard_normal((npts[d], n)) for d in range(nd)]
    assert run_case(kmx_gpu, meval, h["idx1d"], deg, seed=lev) <= 1e-13


def test_realspace_adapted_grid(kmx_gpu):
    """Refined grid: level groups with absent cells."""
    from kmx import grid as G

    rng = np.random.default_rng(3)
    base = G.hash_table_sparse_nd([3, 3], 5, "SG")
    table = G.refine_random(base, 5, 0.6, rng)
    lev = int(table.lev.max())
    n = 3 * 2 ** lev
    meval = [rng.standard_normal((40, n)), rng.standard_normal((33, n))]
    assert run_case(kmx_gpu, meval, table.idx1d, 3, seed=4) <= 1e-13


def test_realspace_errors(kmx_gpu):
    rng = np.random.default_rng(0)
    h = O.hash_table_sparse_nd([3, 3], 3, "SG")
    meval = [rng.standard_normal((10, 2 * 8)), rng.standard_normal((10, 2 * 4))]  # dim 2 too narrow for lev 3
    with pytest.raises(kmx_gpu.KmxError):
        kmx_gpu.RealSpace(meval, h["idx1d"], 2)


def test_asgard_mirror_wavelet_to_realspace(kmx_gpu):
    """The reference-named entry (kmx.asgard.wavelet_to_realspace) on a
    continuity2 grid with host vectors."""
    from kmx import asgard as A
    from kmx import coeffs as K
    from kmx import grid as G

    opts = A.OPTS(lev=3, deg=2)
    pde = K.continuity2(3)
    table = G.hash_table_sparse_nd([3, 3], 8, "SG")
    rng = np.random.default_rng(8)
    meval = [rng.standard_normal((12, 16)), rng.standard_normal((9, 16))]
    fw = rng.standard_normal(table.num_elem * 4)
    fr = A.wavelet_to_realspace(pde, opts, meval, fw, table)
    assert rel(fr, O.wavelet_to_realspace(meval, table.idx1d, 2, fw)) <= 1e-13


# gold_wavelet_to_realspace.m:1,3 (lev, deg); max_lev 8 (OPTS.m:24); domains
# pdes/continuity1.m:16, continuity3.m:24-34
@pytest.mark.parametrize("name,deg,lev,doms", [("continuity_1", 7, 8, [(-1, 1)]),
                                               ("continuity_3", 4, 3, [(-1, 1), (-2, 2), (-3, 3)])])
def test_asgard_realspace_matches_gold(kmx_gpu, gold, name, deg, lev, doms):
    """The reference-named entries end to end on the GPU: matrix_plot_D's evaluation
    matrices, then wavelet_to_realspace of f = 2 * (0, 1, ..., N deg^d - 1)
    (gold_wavelet_to_realspace.m:36-42) against the reference's gold vector (the
    3D one stored as every 8th value)."""
    from kmx import asgard as A
    from kmx import coeffs as K
    from kmx import grid as G

    opts = A.OPTS(lev=lev, deg=deg)
    pde = K.PDE(dims=[K.Dimension(a, b, lev) for (a, b) in doms], terms=[])
    table = G.hash_table_sparse_nd([lev] * len(doms), 8, "SG")
    meval = [A.matrix_plot_D(pde, opts, dim)[0] for dim in pde.dims]
    fw = 2.0 * np.arange(table.num_elem * deg ** len(doms))
    fr = A.wavelet_to_realspace(pde, opts, meval, fw, table)
    key = f"transformations/wavelet_to_realspace_{name}"
    ref = gold[key].ravel()
    assert rel(fr[:: int(gold[key + "/stride"][0])], ref) <= 1e-13


@pytest.mark.parametrize(
    "nd,lev,deg,npts",
    [
        (1, 3, 1, [1]), (1, 6, 8, [65]),            # one row of points; a list of 512 k, one tile and a column more
        (2, 4, 1, [64, 63]), (2, 3, 5, [16, 129]),  # exact and ragged tiles, deg without a shift
        (3, 2, 5, [17, 33, 65]),                    # 25 prefix values: more than one 16-row tile
        (3, 3, 2, [70, 9, 70]),                     # several row tiles over >= 8 column tiles (630 values)
        (6, 1, 2, [3, 2, 4, 2, 3, 5]),
    ],
)
def test_realspace_tile_edges(kmx_gpu, nd, lev, deg, npts):
    """Tile edges and remainders of the staged products.  Every result is a sum of at most
    N deg^d products of d + 1 factors ~ N(0, 1): (N deg^d)^(1/2) eps relative, below 1e-13."""
    rng = np.random.default_rng(nd * 10 + deg)
    h = O.hash_table_sparse_nd([lev] * nd, lev, "SG")
    meval = [rng.standard_normal((npts[d], deg * 2 ** lev)) for d in range(nd)]
    assert run_case(kmx_gpu, meval, h["idx1d"], deg, seed=lev) <= 1e-13


def test_realspace_no_elements(kmx_gpu):
    import torch

    rs = kmx_gpu.RealSpace([np.ones((5, 4)), np.ones((3, 4))], np.zeros((0, 2), np.int32), 2)
    out = torch.full((15,), 7.0, dtype=torch.float64, device="cuda")
    rs.apply(torch.empty(0, dtype=torch.float64, device="cuda"), out)
    assert torch.count_nonzero(out) == 0


def _dense(meval, idx, deg, f):
    """The definition with every zero of Meval multiplied (so 0 x inf is a NaN)."""
    B = deg ** len(meval)
    out = np.zeros(int(np.prod([m.shape[0] for m in meval])))
    with np.errstate(invalid="ignore"):
        for e, row in enumerate(np.asarray(idx) - 1):
            M = np.ones((1, 1))
            for m, J in zip(meval, row):
                M = np.kron(M, m[:, J * deg:(J + 1) * deg])
            out += (M * f[e * B:(e + 1) * B]).sum(axis=1)
    return out


@pytest.mark.parametrize("nd,lev,deg,npts", [(1, 6, 3, None), (2, 5, 3, None), (3, 4, 2, (96, 40, 130)),
                                             (2, 5, 2, (65, 64)), (2, 3, 2, (400, 1))])
def test_realspace_children_by_tile(kmx_gpu, nd, lev, deg, npts):
    """Plotting grids of several tiles, where a tile sums over the children that are not zero
    on it: against the definition, with and without values that are not finite, the finite
    call after one that was not, and replayed."""
    import torch
    from kmx import coeffs as K
    from kmx import grid as G

    idx = G.hash_table_sparse_nd([lev] * nd, lev, "SG").idx1d
    meval = [K.matrix_plot_D(deg, lev, -1.0, 1.0)[0] for _ in range(nd)]
    if npts:  # other numbers of points: rows repeated or left out
        meval = [m[np.arange(n) * m.shape[0] // n] for m, n in zip(meval, npts)]
    meval[0] = meval[0].copy()
    meval[0][:, -deg:] = 0.0  # a block that is zero everywhere
    rng = np.random.default_rng(nd + lev)
    f = rng.standard_normal(len(idx) * deg ** nd)
    rs = kmx_gpu.RealSpace(meval, idx, deg, index_base=1)
    want = _dense(meval, idx, deg, f)
    got = rs.apply(torch.from_numpy(f).cuda())
    assert rel(got.cpu().numpy(), want) <= 1e-13
    fd, out = torch.from_numpy(f).cuda(), torch.empty_like(got)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        rs.apply(fd, out)
    last = len(idx) - 1  # (its first index is the finest: perhaps of the zero block)
    for at, v in ((0, np.inf), (f.size // 2, np.nan), (last * deg ** nd, -np.inf), (f.size - 1, np.inf)):
        g = f.copy()
        g[at] = v
        ref = _dense(meval, idx, deg, g)
        bad = rs.apply(torch.from_numpy(g).cuda()).cpu().numpy()
        assert np.array_equal(np.isnan(bad), np.isnan(ref)) and np.array_equal(bad == np.inf, ref == np.inf)
        assert np.array_equal(bad == -np.inf, ref == -np.inf)
        assert torch.equal(rs.apply(torch.from_numpy(f).cuda()), got)
        fd.copy_(torch.from_numpy(g))
        graph.replay()
        assert np.array_equal(np.nan_to_num(out.cpu().numpy(), nan=1.5), np.nan_to_num(bad, nan=1.5))
        fd.copy_(torch.from_numpy(f))
        graph.replay()
        assert torch.equal(out, got)


@pytest.mark.parametrize("nd,lev,deg", [(2, 5, 3), (3, 4, 2)])
@pytest.mark.parametrize("dim", [0, 1])
@pytest.mark.parametrize("value", [1e308, np.inf, np.nan])
def test_realspace_values_lost_in_a_later_stage(kmx_gpu, nd, lev, deg, dim, value):
    """Finite coefficients and, at a few points of one dimension, evaluation values that
    overflow the sum (1e308 times sums over 1e3) or are not finite themselves: nothing is
    finite at those points, and every other point has the bits that it has without them,
    call after call, eager and replayed."""
    import torch
    from kmx import coeffs as K
    from kmx import grid as G

    idx = G.hash_table_sparse_nd([lev] * nd, lev, "SG").idx1d
    rng = np.random.default_rng(nd * 10 + dim)
    # the zeros of real evaluation matrices, 130 points (three tiles), positive values
    meval = []
    for _ in range(nd):
        m = K.matrix_plot_D(deg, lev, -1.0, 1.0)[0]
        m = m[np.arange(130) * m.shape[0] // 130]
        meval.append(np.where(m == 0.0, 0.0, rng.uniform(1.0, 2.0, m.shape)))
    f = torch.from_numpy(rng.uniform(1e3, 2e3, len(idx) * deg ** nd)).cuda()
    want = kmx_gpu.RealSpace(meval, idx, deg).apply(f)
    assert bool(torch.isfinite(want).all())
    points = [70, 129]  # in the second and the third tile
    hit = [m.copy() for m in meval]
    hit[dim][points] = np.where(hit[dim][points] == 0.0, 0.0, value)
    rs = kmx_gpu.RealSpace(hit, idx, deg)
    shape = [130] * nd
    keep = [i for i in range(130) if i not in points]

    def check(out):
        v = out.view(shape).movedim(dim, 0)
        assert not bool(torch.isfinite(v[points]).any())
        assert torch.equal(v[keep], want.view(shape).movedim(dim, 0)[keep])

    for _ in range(8):
        check(rs.apply(f))
    out = torch.empty_like(want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        rs.apply(f, out)
    for _ in range(3):
        graph.replay()
        check(out)
        out.zero_()
        check(rs.apply(f))
