"""The search of a corrected history for the first interval that brackets an ionized
fraction (zreioncorrect, bubblehistory_d2z.C:270-299), by bisection where the history
does not decrease and entry by entry where it does: the corrected field is the
oracle's bit for bit, as in test_gpu_bubble.py."""
import numpy as np
import pytest

import bubble as ob
from _cases import field, lib_params
from conftest import announce
from prc_d2z import D2Z, FUSED_FP32, NCHISTORY

pytestmark = pytest.mark.gpu


def _rising():
    return np.linspace(0.0, 1.01, NCHISTORY).astype(np.float32)


def _steps():
    return np.repeat(_rising()[::100], 100)


def _falls_inside():
    c = _rising()
    c[2000:7000] = c[2000:7000][::-1]
    return c


def _falls_at_the_ends():
    c = _rising()
    c[:2] = c[1], c[0]
    c[-2:] = c[-1], c[-2]
    return c


def _one_entry_lower():
    c = _rising()
    c[5000] = c[4000]
    return c


@pytest.mark.parametrize("shape", [_rising, _steps, _falls_inside, _falls_at_the_ends, _one_entry_lower])
def test_search_vs_oracle(shape):
    announce(f"corrected history search {shape.__name__}")
    N, chist = 64, shape()
    lp = lib_params(N, nscales=8, mode=FUSED_FP32)
    with D2Z(lp) as d:
        d.set_delta(field(N))
        d.run()
        z = d.zreion()
        hist = D2Z.cumulative_history(d.history(), N)
        d.correct_zreion(hist, chist)
        got = d.zreion()
    assert np.array_equal(got, ob.correct_zreion(z, hist, chist))
