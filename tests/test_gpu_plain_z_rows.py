"""The plain path's last pass, cell by cell, at N = 16 and 32, where a thread holds a
whole row, at N = 256, and at N = 512, where the rows of the intermediates are stored
permuted.  Its rows are those that smoothed_field() returns: the sums of squares are
theirs, and zreion and the recorded radii follow from them."""
import numpy as np
import pytest

from _cases import lib_params
from conftest import announce
from prc_d2z import D2Z, PLAIN_FP32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rbub", [0, 1])
@pytest.mark.parametrize("N", [16, 32, 256, 512])
def test_rows_sums_and_radii(N, rbub):
    announce(f"plain z pass N={N} rbubble={rbub}")
    lp = lib_params(N, nscales=3, mode=PLAIN_FP32, rbub=rbub, rmax=min(40.0, 0.4 * N))
    with D2Z(lp) as d:
        d.generate_delta(4)
        d.run()
        z, diag = d.zreion(), d.radius_diag()
        rb = d.rbubble() if rbub else None
        best = np.zeros((N, N, N), np.float32)
        at = np.zeros((N, N, N), np.int8)
        for r in range(3):
            f = d.smoothed_field(r)
            # both sum the same floats in double: one rounding of the result to float
            s = np.sqrt(np.mean(np.square(f, dtype=np.float64)))
            assert abs(diag["sigma_grid"][r] - s) <= 2.0 ** -23 * s
            # A (delta_R + B) - 1 in double, rounded to float; strictly greater wins
            zr = (diag["A"][r] * (f.astype(np.float64) + diag["B"][r]) - 1.0).astype(np.float32)
            win = zr > best
            best[win], at[win] = zr[win], r + 1
    assert np.array_equal(z, best)
    if rbub:
        # recorded in Mpc, the table's column in Mpc/h
        for r in range(3):
            R = rb[at == r + 1]
            assert R.size or N < 256
            assert not R.size or np.all(R == R[0]) and np.isclose(R[0] * lp.h, diag["R_mpch"][r], rtol=1e-6)
        assert not rb[at == 0].any()
