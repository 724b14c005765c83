"""kmx_kronmult_noalloc (the library allocates nothing; intermediates in its fixed
scratch array) against the allocating kmx_kronmult, through the C ABI: two calls
in a row, the second smaller than the first (the scratch keeps the first call's
contents, which the second must not see), bit-for-bit equal results; an
intermediate beyond the scratch limit is refused with KMX_E_SHAPE."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _case(rng, shapes, nvec):
    import torch

    mats = [torch.from_numpy(rng.standard_normal(s)).cuda() for s in shapes]
    ncol = int(np.prod([s[1] for s in shapes]))
    X = torch.from_numpy(rng.standard_normal((ncol, nvec))).cuda()
    return mats, X


def test_kronmult_noalloc_matches_allocating_entry(kmx_gpu):
    import torch

    from kmx import _lib

    rng = np.random.default_rng(17)
    cases = [
        ([(4, 3), (5, 4), (3, 5), (4, 4)], 6),  # k = 4, rectangular factors, 6 vectors
        ([(3, 3), (2, 4), (3, 2)], 2),          # smaller: k = 3
        ([(4, 4), (4, 4)], 1),                  # k = 2, one vector
    ]
    for shapes, nvec in cases:
        mats, X = _case(rng, shapes, nvec)
        ref = kmx_gpu.kronmult(mats, X)
        got = kmx_gpu.kronmult(mats, X, noalloc=True)
        torch.cuda.synchronize()
        assert got.shape == ref.shape
        assert torch.equal(got, ref), (shapes, nvec, float((got - ref).abs().max()))
        # and the closed form, on the host
        K = mats[0].cpu().numpy()
        for m in mats[1:]:
            K = np.kron(K, m.cpu().numpy())
        want = K @ X.cpu().numpy()
        assert np.linalg.norm(got.cpu().numpy() - want) <= 1e-13 * np.linalg.norm(want)
    # an intermediate above KMX_KRON_SCRATCH_ELEMS / 2 values is refused
    big = [(128, 128), (128, 128), (128, 128)]
    mats, X = _case(rng, big, 1)
    assert 128 ** 3 > _lib.KRON_SCRATCH_ELEMS // 2
    with pytest.raises(kmx_gpu.KmxError) as e:
        kmx_gpu.kronmult(mats, X, noalloc=True)
    assert e.value.code == _lib.KMX_E_SHAPE


@pytest.mark.parametrize("shapes,nvec", [
    ([(1, 1)], 1), ([(17, 33)], 5), ([(40, 3), (3, 40)], 7),           # more than 16 rows, one mode
    ([(16, 16), (16, 16), (2, 2)], 3),                                 # 16 rows exactly
    ([(8, 8)] * 4 + [(2, 2)], 2),                                      # 8192 values: the largest power of two in a tile
    ([(9, 9)] * 4 + [(2, 2)], 2),                                      # 13122: two launches, the second strided
    ([(3, 2), (97, 89), (91, 95)], 3),                                 # a mode with ragged runs of the faster values
    ([(2, 9000)], 2), ([(9000, 2), (2, 3)], 1),                        # a mode beyond the tile: launches of its own
    ([(2, 2)] * 16, 1),
])
def test_kronmult_groups(kmx_gpu, shapes, nvec):
    """The grouped launches at the edges of their tile and of their 16-row passes, allocating
    and not, against numpy's products factor by factor: sums of at most 9000 products per
    factor, so well below 1e-13 relative (2-norm); and Y written over X."""
    import torch

    rng = np.random.default_rng(len(shapes) * 100 + nvec)
    mats, X = _case(rng, shapes, nvec)
    want = X.cpu().numpy()
    pre = 1
    for m in mats:
        a = m.cpu().numpy()
        want = np.matmul(a, want.reshape(pre, a.shape[1], -1)).reshape(pre * a.shape[0], -1)
        pre *= a.shape[0]
    want = want.reshape(pre, nvec)
    tol = 1e-13 * np.linalg.norm(want)
    got = kmx_gpu.kronmult(mats, X)
    assert np.linalg.norm(got.cpu().numpy() - want) <= tol
    again = kmx_gpu.kronmult(mats, X, noalloc=True)
    assert torch.equal(again, got)
    if len(shapes) > 1 and pre == X.shape[0]:
        import ctypes as C

        from kmx._lib import check, lib

        k = len(mats)
        xs = X.t().contiguous()
        cm = [m.t().contiguous() for m in mats]
        check(lib().kmx_kronmult(k, (C.c_int * k)(*[s[0] for s in shapes]), (C.c_int * k)(*[s[1] for s in shapes]),
                                 (C.c_void_p * k)(*[m.data_ptr() for m in cm]), C.c_void_p(xs.data_ptr()), nvec,
                                 C.c_void_p(xs.data_ptr()), C.c_void_p(torch.cuda.current_stream().cuda_stream)))
        torch.cuda.synchronize()
        assert torch.equal(xs.view(nvec, -1).t(), got)
