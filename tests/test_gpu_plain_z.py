"""The plain path's last pass (c2r, barrier and sum of squares in one kernel): its
rows are those that smoothed_field() returns, for every plan length and with fewer
and more rows than blocks."""
import numpy as np
import pytest

import d2z_fp64 as oracle
from _cases import field, lib_params, oracle_params, zreion_metrics
from conftest import announce
from prc_d2z import D2Z, PLAIN_FP32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rbub", [0, 1])
@pytest.mark.parametrize("N", [16, 32, 64, 128, 192])
def test_rows_and_sums(N, rbub):
    announce(f"plain z pass N={N} rbubble={rbub}")
    f = field(N)
    lp = lib_params(N, nscales=5, mode=PLAIN_FP32, rbub=rbub)
    with D2Z(lp) as d:
        d.set_delta(f)
        d.run()
        z, table = d.zreion(), d.radius_table()
        rb = d.rbubble() if rbub else None
        sums = [np.sqrt(np.mean(d.smoothed_field(r).astype(np.float64) ** 2)) for r in range(5)]
    # both sum the same floats in double: one rounding of the result to float
    np.testing.assert_allclose(table[:, 2], sums, rtol=2.0 ** -23)
    zo, _, _ = oracle.delta2zreion(f, oracle_params(lp))
    assert zreion_metrics(z, zo)["max_abs"] <= 2e-4
    if rbub:
        assert np.array_equal(rb > 0, z > 0)
        # recorded in Mpc, the table's first column in Mpc/h
        assert all(np.isclose(R * lp.h, table[:, 0], rtol=1e-6).any() for R in np.unique(rb[rb > 0]))
