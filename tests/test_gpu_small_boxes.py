"""Small boxes, whose x pass spreads a launch's radii over blocks and whose z pass
spreads a batch's over groups of threads: every batch length, also one that the
groups do not divide or outnumber, gives the same bits, and the default one the
oracle's field."""
import numpy as np
import pytest

import d2z_fp64 as oracle
from _cases import field, lib_params, oracle_params, zreion_metrics
from conftest import announce
from prc_d2z import D2Z, FUSED_FP32, FUSED_HALF, FUSED_MIXED

pytestmark = pytest.mark.gpu
NS = 11


@pytest.mark.parametrize("mode", [FUSED_FP32, FUSED_MIXED, FUSED_HALF])
@pytest.mark.parametrize("N", [16, 32, 64, 128])
def test_batch_lengths(N, mode):
    announce(f"small box N={N} mode={mode}")
    f = field(N)
    lp = lib_params(N, nscales=NS, mode=mode)
    with D2Z(lp) as d:
        d.set_delta(f)
        d.run()
        z, table = d.zreion(), d.radius_table()
        d.run()
        assert np.array_equal(d.zreion(), z)
    for rpl in (1, 2, 3, 5, 7):
        with D2Z(lib_params(N, nscales=NS, mode=mode, rpl=rpl)) as d:
            d.set_delta(f)
            d.run()
            assert np.array_equal(d.zreion(), z), rpl
            np.testing.assert_allclose(d.radius_table(), table, rtol=1e-6)
    zo, _, _ = oracle.delta2zreion(f, oracle_params(lp))
    assert zreion_metrics(z, zo)["max_abs"] <= (0.02 if mode == FUSED_HALF else 2e-4)
