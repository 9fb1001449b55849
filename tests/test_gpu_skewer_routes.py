"""The two routes of the bubble mean free paths: few skewers walk zreion itself, many
a copy with y contiguous.  Both against the oracle's walks on either side of the rule
(64 skewers, N^2 / 1200 from N = 512 on), as in test_gpu_bubble.py; and a call with
one skewer does not pay for the copy.
"""
import time

import numpy as np
import pytest

import bubble as ob
from _cases import box_mpc, lib_params
from conftest import announce
from prc_d2z import D2Z, FUSED_FP32, PLAIN_FP32

pytestmark = pytest.mark.gpu


def _box(N, mode=FUSED_FP32, nscales=6):
    lp = lib_params(N, nscales=nscales, mode=mode, rmax=0.1 * 1.5625 * N)
    d = D2Z(lp)
    d.generate_delta(5)
    d.run()
    return lp, d


@pytest.mark.parametrize("N,counts", [(16, (1, 63, 64)), (32, (1, 63, 64)), (64, (63, 64, 65)), (192, (1, 63, 64)), (512, (217, 218))])
def test_routes_vs_oracle(N, counts):
    lp, d = _box(N)
    with d:
        z = d.zreion()
        hist = D2Z.cumulative_history(d.history(), N)
        for nsk in counts:
            announce(f"skewer routes N={N} nskewers={nsk}")
            mfp, _, dfd = d.bubble_mfp(hist, nskewers=nsk, seed=3)
            mfp_o, _, dfd_o, _, _ = ob.bubble_mfp(z, hist, box_mpc(lp), nskewers=nsk, seed=3)
            assert np.abs(dfd.astype(np.int64) - dfd_o.astype(np.int64)).sum() <= 4
            np.testing.assert_allclose(mfp, mfp_o, rtol=1e-6)


def test_one_skewer_does_not_copy_the_field():
    """At 1024^3 the copy moves 8.6 GB (1.7 ms); the walks of one skewer take about
    0.1 ms, as much as at 64^3 within a small factor."""
    best = {}
    for N in (64, 1024):
        announce(f"one skewer N={N}")
        _, d = _box(N, PLAIN_FP32, 2)
        with d:
            hist = D2Z.cumulative_history(d.history(), N)
            t = []
            for _ in range(15):
                t0 = time.perf_counter()
                d.bubble_mfp(hist, nskewers=1)
                t.append(time.perf_counter() - t0)
            best[N] = min(t[1:])
    assert best[1024] <= 4.0 * best[64], best
