"""Host-side pieces of the time-step harness that need no GPU."""
import numpy as np


def test_gmres_least_squares_update_matches_lstsq():
    """The host side of the device GMRES: Givens rotations applied column by column
    give the minimiser of |beta e1 - H y| and its residual, as numpy's lstsq does."""
    from kmx.timestep import HessenbergLSQ

    rng = np.random.default_rng(0)
    for m in (1, 5, 40):
        H = np.triu(rng.standard_normal((m + 1, m)), -1)
        beta = 2.5
        ls = HessenbergLSQ(beta, m)
        e1 = np.zeros(m + 1)
        e1[0] = beta
        for k in range(m):
            res = ls.add_column(H[: k + 2, k].tolist())
            yk = np.linalg.lstsq(H[: k + 2, : k + 1], e1[: k + 2], rcond=None)[0]
            assert abs(res - np.linalg.norm(H[: k + 2, : k + 1] @ yk - e1[: k + 2])) <= 1e-12 * beta
            assert ls.residual() == res
        assert np.max(np.abs(ls.solve() - yk)) <= 1e-10 * max(1.0, np.abs(yk).max())


def test_gmres_holds_back_chunks_only_when_the_queued_steps_converge():
    """The device GMRES holds the next chunk back when the residual estimates,
    extrapolated at their last chunk's rate, reach the target within the queued
    steps ((depth - 1) chunks), and never for stalling or growing residuals."""
    from types import SimpleNamespace

    from kmx.timestep import DeviceGMRES

    g = SimpleNamespace(chunk=4, depth=2)
    held = DeviceGMRES._converges_in_flight
    rs = [10.0 ** -i for i in range(9)]  # a decade per step, at 1e-8 after 8 steps
    assert held(g, rs, 1e-11)      # 3 more steps: within the 4 queued
    assert held(g, rs, 1e-12)      # exactly 4
    assert not held(g, rs, 1e-13)  # 5: the next chunk is needed
    assert not held(g, [1.0, 1.0, 1.0, 1.0, 1.0], 1e-3)  # stalled
    assert not held(g, [1.0, 2.0, 3.0], 1e-3)            # growing
    assert not held(g, [1.0], 1e-3)                      # no step yet
    assert not held(SimpleNamespace(chunk=4, depth=1), rs, 1e-11)  # nothing queued
    assert not held(g, rs, 0.0)  # tol = 0: never converges by estimate


def test_krylov_vectors_in_the_sweeps_order():
    """Not without a sweep, not much longer ones, and not across the end of the register
    kernels (kmx_gmres.hip: AR_MAX_G workgroups of AR_MIN_CHUNK values)."""
    import os
    import re

    from conftest import ROOT

    from kmx import timestep as TS

    src = open(os.path.join(ROOT, "dg-sparsegrid_amd", "csrc", "kmx_gmres.hip")).read()
    g, c = (int(re.search(rf"constexpr int {n} = (\d+)", src).group(1)) for n in ("AR_MAX_G", "AR_MIN_CHUNK"))
    assert TS.ARNOLDI_SHORT == g * c
    assert not TS.box_order(2304, 0) and TS.box_order(2304, 2304) and TS.box_order(32064, 32064)
    assert TS.box_order(8000, 9000) and not TS.box_order(8000, 9001)
    assert TS.box_order(32512, 32768) and not TS.box_order(32512, 32769) and not TS.box_order(32768, 33728)
    assert TS.box_order(32769, 33728)
