"""The binned power spectrum at the smallest grids, whose planes kz = 0 and N/2 are
most of its work, and with few and many bins; bounds as in test_gpu_power_spectrum.py."""
import numpy as np
import pytest

import d2z_fp64 as oracle
from _cases import field, lib_params
from conftest import announce
from prc_d2z import D2Z, PLAIN_FP32
from test_gpu_power_spectrum import _bins

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,nk", [(16, 1), (16, 12), (32, 1), (32, 40), (64, 60), (256, 30)])
def test_sizes_vs_oracle(N, nk):
    lp = lib_params(N, mode=PLAIN_FP32)
    kmin, kmax = _bins(N, lp.BoxSize, nk)
    delta = field(N)
    announce(f"power spectrum N={N} nk={nk}")
    with D2Z(lp) as d:
        d.set_delta(delta)
        got = d.power_spectrum(nk, kmin, kmax)
    ref = oracle.power_spectrum(delta, lp.BoxSize, nk, kmin, kmax)
    assert np.array_equal(got["nmodes"], ref["nmodes"])
    for key in ("ps", "ook2", "kmean"):
        np.testing.assert_allclose(got[key], ref[key], rtol=1e-5, equal_nan=True, err_msg=key)
