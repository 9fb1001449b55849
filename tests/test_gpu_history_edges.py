"""The history histogram at the edges of its bins and table, and the skewer walks
at grid sizes below, at and between multiples of the wave width.

Counts are integers and compared exactly with the definition in FP64
(bubblehistory_d2z.C:17-28); mean free paths as in test_gpu_bubble.py.
"""
import numpy as np
import pytest
import torch

import bubble as ob
from _cases import box_mpc, field, lib_params
from conftest import announce
from prc_d2z import D2Z, FUSED_FP32, NHISTORY, history_noalloc

pytestmark = pytest.mark.gpu


def _counts(z):
    dz = np.float64(np.float32((0.01 - 49.9) / (NHISTORY - 1)))
    with np.errstate(invalid="ignore"):
        q = (z.astype(np.float64) - 49.9) / dz
        b = q[(q > -1.0) & (q < NHISTORY)].astype(np.int64)
    return np.bincount(b, minlength=NHISTORY)


@pytest.mark.parametrize("n", [1, 3, 1027, (1 << 18) + 5, 3 * (1 << 18) + 2])
def test_history_bin_edges(n):
    announce(f"history bin edges n={n}")
    rng = np.random.default_rng(n)
    dz = np.float64(np.float32((0.01 - 49.9) / (NHISTORY - 1)))
    edge = (49.9 + dz * rng.integers(-3, NHISTORY + 3, n)).astype(np.float32)
    z = np.nextafter(edge, np.float32(np.inf) * rng.choice(np.float32([-1, 1]), n)).astype(np.float32)
    z = np.where(rng.random(n) < 0.4, edge, z)
    wild = np.float32([0.0, -1.0, 49.9, 49.9005, 50.5, 0.01, 0.0095, 1e30, -1e30, np.inf, -np.inf, np.nan])
    z = np.where(rng.random(n) < 0.05, rng.choice(wild, n), z).astype(np.float32)
    t = torch.from_numpy(z).cuda()
    torch.cuda.synchronize()
    assert np.array_equal(history_noalloc(t.data_ptr(), n).astype(np.int64), _counts(z))


@pytest.mark.parametrize("n,value", [(4096, np.nan), (4096, 60.0), (5000, 0.0), (5000, 7.25)])
def test_history_one_value(n, value):
    """No cell in any bin, and every cell in one."""
    announce(f"history of one value {value}")
    z = np.full(n, value, np.float32)
    t = torch.from_numpy(z).cuda()
    torch.cuda.synchronize()
    assert np.array_equal(history_noalloc(t.data_ptr(), n).astype(np.int64), _counts(z))


@pytest.mark.parametrize("N,nsk", [(16, 300), (32, 300), (64, 257), (192, 300)])
def test_skewers_vs_oracle(N, nsk):
    announce(f"skewers N={N} nskewers={nsk}")
    lp = lib_params(N, nscales=8, mode=FUSED_FP32)
    with D2Z(lp) as d:
        d.set_delta(field(N))
        d.run()
        z = d.zreion()
        hist = D2Z.cumulative_history(d.history(), N)
        mfp, _, dfd = d.bubble_mfp(hist, nskewers=nsk, seed=11)
    mfp_o, _, dfd_o, _, _ = ob.bubble_mfp(z, hist, box_mpc(lp), nskewers=nsk, seed=11)
    assert np.abs(dfd.astype(np.int64) - dfd_o.astype(np.int64)).sum() <= 4
    np.testing.assert_allclose(mfp, mfp_o, rtol=1e-6)
