"""The history histogram over the sizes at which its number of blocks changes (2^13
cells a block, 128 blocks from 2^20 cells, one per 2^15 from 2^22, 256 from 2^23), and
the time of a small grid, whose cells must be shared out over the chip.

Counts are integers and compared exactly with the definition in FP64.
"""
import time

import numpy as np
import pytest
import torch

from conftest import announce
from prc_d2z import history_noalloc
from test_gpu_history_edges import _counts

pytestmark = pytest.mark.gpu


def _zreion(n):
    rng = np.random.default_rng(n)
    z = rng.normal(9.0, 2.5, n).astype(np.float32)
    z[rng.random(n) < 0.1] = 0.0
    return z


def _on_device(z):
    t = torch.from_numpy(z).cuda()
    torch.cuda.synchronize()
    return t


@pytest.mark.parametrize("n", [(1 << 13) - 1, (1 << 13) + 1, (1 << 14) + 3, (1 << 20) - 5, (1 << 20) + (1 << 13),
                               (1 << 22) + (1 << 15) + 2, (1 << 23) + 7])
def test_counts(n):
    announce(f"history blocks n={n}")
    z = _zreion(n)
    t = _on_device(z)
    assert np.array_equal(history_noalloc(t.data_ptr(), n).astype(np.int64), _counts(z))


def test_a_small_grid_is_shared_out():
    """64^3 cells cost little more than 16^3: launches and the copy of the counts."""
    t = _on_device(_zreion(64 ** 3))
    best = {}
    for n in (16 ** 3, 64 ** 3):
        announce(f"history time n={n}")
        runs = []
        for _ in range(40):
            t0 = time.perf_counter()
            history_noalloc(t.data_ptr(), n)
            runs.append(time.perf_counter() - t0)
        best[n] = min(runs)
    assert best[64 ** 3] <= 1.6 * best[16 ** 3], best
