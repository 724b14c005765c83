"""Kronecker chains and batched GEMMs on arguments as callers hold them: row-major
factors (kmx_kronmult_layout), lists of tensors, addresses, numpy sizes."""
import ctypes as C

import numpy as np
import pytest


def test_rowmajor_factors_beyond_the_limit_are_refused():
    from kmx import _lib as L

    lib = L.lib()
    n = (C.c_int * 2)(25, 25)
    one = (C.c_void_p * 2)(8, 8)  # never read: 1250 values are refused before any launch
    args = (2, n, n, one)
    assert lib.kmx_kronmult_layout(*args, bytes([0, 1]), 8, 1, 8, 0, None, None) == L.KMX_E_SHAPE
    assert lib.kmx_kronmult_layout(*args, bytes([0, 1]), 8, 1, 8, 1, None, None) == L.KMX_E_SHAPE
    assert lib.kmx_kronmult_layout(*args, bytes([1, 1]), 8, 0, None, 0, None, None) == L.KMX_E_ARG


@pytest.mark.gpu
@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("shapes,nvec", [([(3, 5)], 1), ([(1, 4), (6, 1), (2, 3)], 7), ([(8, 8)] * 4, 9),
                                         ([(16, 16)] * 3, 5), ([(31, 2), (7, 31), (4, 9)], 33), ([(25, 40)], 3),
                                         ([(25, 40), (2, 3)], 3), ([(500, 1), (1, 400)], 2), ([(2, 2)] * 12, 1),
                                         ([(6, 5)] * 6, 3)])
def test_factor_layouts_give_the_same_bits(kmx_gpu, shapes, nvec, noalloc):
    """Factors by rows, by columns, as strided views, alone and mixed, up to and beyond the
    values taken by rows: the bits of column-major factors (given Y: copies are made)."""
    import torch

    gen = torch.Generator().manual_seed(len(shapes) * 100 + nvec)
    base = [torch.randn(r, c, dtype=torch.float64, generator=gen).cuda() for r, c in shapes]
    ncol, nrow = int(np.prod([c for _, c in shapes])), int(np.prod([r for r, _ in shapes]))
    X = torch.randn(ncol, nvec, dtype=torch.float64, generator=gen).cuda()
    col = [m.t().contiguous().t() for m in base]
    wide = [torch.stack([m, m], dim=2)[:, :, 0] for m in base]
    Y = torch.empty(nrow * nvec, dtype=torch.float64, device="cuda")
    ref = kmx_gpu.kronmult(col, X, noalloc=noalloc, Y=Y).clone()
    mixed = [(base, col, wide)[i % 3][i] for i in range(len(base))]
    for mats in (base, col, wide, mixed):
        assert torch.equal(kmx_gpu.kronmult(mats, X, noalloc=noalloc), ref)
    want = X.cpu().numpy()
    K = np.ones((1, 1))
    if nrow * ncol <= 1 << 22:
        for m in base:
            K = np.kron(K, m.cpu().numpy())
        # a sum of ncol products of k + 1 factors
        bound = 8 * (ncol + len(shapes)) * np.finfo(float).eps * (np.abs(K) @ np.abs(want))
        assert np.all(np.abs(ref.cpu().numpy() - K @ want) <= bound)
    with pytest.raises((RuntimeError, ValueError, IndexError)):
        kmx_gpu.kronmult([base[0][None]] + base[1:], X)


@pytest.mark.gpu
def test_gemm_arguments_as_tensors_addresses_and_iterators(kmx_gpu):
    import torch

    gen = torch.Generator().manual_seed(4)
    n = [5, 17, 64]
    A = [torch.randn(i * i, dtype=torch.float64, generator=gen).cuda() for i in n]
    outs = []
    for kind in range(4):
        Cm = [torch.zeros(i * i, dtype=torch.float64, device="cuda") for i in n]
        size = [n, tuple(n), np.asarray(n), [np.int64(i) for i in n]][kind]
        a = [A, [t.data_ptr() for t in A], (t for t in A), [A[0].data_ptr(), A[1], A[2]]][kind]
        kmx_gpu.gemm_vbatched("N", "T", size, size, size, 1.0, a, size, A, size, 0.0, Cm, size)
        outs.append(torch.cat(Cm))
    assert all(torch.equal(o, outs[0]) for o in outs[1:])
    want = torch.cat([(t.view(i, i).t() @ t.view(i, i)).t().reshape(-1) for t, i in zip(A, n)])
    assert torch.allclose(outs[0], want, rtol=0, atol=1e-12)


@pytest.mark.gpu
def test_batch_state_layouts(kmx_gpu):
    """A longer vector, and one that is not one contiguous vector, as states of a batch."""
    import torch
    from kmx import batch as BT

    s = BT.BatchedSystem(BT.make_instances(count=2, seed=3, lev2d=(4, 5), lev3d=(4, 4)), sweep=("fp64",))
    ref = s.apply(s.f, torch.empty_like(s.f), "fp64").clone()
    long = torch.cat([s.f, s.f])
    y = torch.zeros_like(long)
    s.apply(long, y, "fp64")
    assert torch.equal(y[:s.dof], ref) and not y[s.dof:].any()
    with pytest.raises(ValueError):
        s.apply(long[::2], y, "fp64")


@pytest.mark.gpu
@pytest.mark.parametrize("count", [81, 216, 217])
@pytest.mark.parametrize("ta,tb,beta", [("N", "N", 0.0), ("T", "N", 0.5), ("N", "T", -1.0), ("T", "T", 0.0)])
def test_packed_descriptors_give_the_same_bits(kmx_gpu, ta, tb, beta, count):
    """Batches whose descriptors travel packed (leading dimensions the rows stored): the bits
    of the same products one call each, empty extents and 1 x 1 among them; one leading
    dimension more than its rows takes the other route."""
    import torch

    rng = np.random.default_rng(count)
    gen = torch.Generator().manual_seed(count)
    shapes = [tuple(int(v) for v in rng.integers(1, 70, 3)) for _ in range(count)]
    shapes[3], shapes[4], shapes[5], shapes[6] = (1, 1, 1), (0, 7, 5), (7, 5, 0), (64, 64, 130)

    def rnd(n):
        return torch.randn(max(1, n), dtype=torch.float64, generator=gen).cuda()

    ms, ns, ks = (list(v) for v in zip(*shapes))
    A, B, C0 = [rnd(m * k) for m, _, k in shapes], [rnd(n * k) for _, n, k in shapes], [rnd(m * n) for m, n, _ in shapes]
    lda = [max(1, k if ta == "T" else m) for m, _, k in shapes]
    ldb = [max(1, n if tb == "T" else k) for _, n, k in shapes]
    ldc = [max(1, m) for m, _, _ in shapes]
    many, one = [c.clone() for c in C0], [c.clone() for c in C0]
    kmx_gpu.gemm_vbatched(ta, tb, ms, ns, ks, 1.5, A, lda, B, ldb, beta, many, ldc)
    for i in range(count):
        kmx_gpu.gemm_vbatched(ta, tb, [ms[i]], [ns[i]], [ks[i]], 1.5, [A[i]], [lda[i]], [B[i]], [ldb[i]], beta, [one[i]],
                              [ldc[i]])
    for i in range(count):
        assert torch.equal(many[i], one[i]), (i, shapes[i])
    wide = rnd(71 * 71)
    other = [c.clone() for c in C0]
    lda[0] = 71
    kmx_gpu.gemm_vbatched(ta, tb, ms, ns, ks, 1.5, [wide] + A[1:], lda, B, ldb, beta, other, ldc)
    for i in range(1, count):
        assert torch.equal(other[i], one[i]), (i, shapes[i])


@pytest.mark.gpu
@pytest.mark.parametrize("count", [1, 100, 641])
def test_gemm_on_a_stream_given_is_complete_on_return(kmx_gpu, count):
    """Behind work that keeps that stream busy: C may be read, and A and B given back, on the
    current stream as soon as the call returns.  Recorded into a graph otherwise."""
    import torch

    n = [6] * count
    A = torch.randn(count, 36, dtype=torch.float64, device="cuda")
    Cm = torch.zeros(count, 36, dtype=torch.float64, device="cuda")
    want = torch.matmul(A.view(-1, 6, 6), A.view(-1, 6, 6)).reshape(count, 36)  # row-major: (B A)^T
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        torch.cuda._sleep(20_000_000)
    kmx_gpu.gemm_vbatched("N", "N", n, n, n, 1.0, list(A), n, list(A), n, 0.0, list(Cm), n, stream=side)
    assert side.query()
    assert torch.allclose(Cm, want, rtol=0, atol=1e-13)
    if count <= 640:
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            kmx_gpu.gemm_vbatched("N", "N", n, n, n, 1.0, list(A), n, list(A), n, 0.0, list(Cm), n,
                                  stream=torch.cuda.current_stream())
        for _ in range(3):
            Cm.zero_()
            graph.replay()
            assert torch.allclose(Cm, want, rtol=0, atol=1e-13)
            torch.cuda.synchronize()
