"""The paired FP16 planes of N = 1024: the vector and the matrix form of the x and
of the z pass, in each combination, read and write the same layout."""
import numpy as np
import pytest

from conftest import announce
from prc_d2z import D2Z, D2ZParams, FUSED_HALF, PLAN_MATRIX, PLAN_VECTOR

pytestmark = pytest.mark.gpu

# The forms round delta_R differently, each within the half path's 2e-3 of its rms;
# z = A delta_R - A B - 1 with sigma_R A below about 1 for these radii, so two forms
# are within 2 x 2e-3 rms.  A misplaced column would move z by its own rms (> 0.1).
RMS = 4e-3


@pytest.mark.parametrize("rbub", [0, 1])
def test_plans_share_a_layout(rbub):
    lp = D2ZParams(N=1024, BoxSize=2000.0, Nscales=3, Rmax=120.0, zeta=40.0, M_min=1.4706e8, mode=FUSED_HALF,
                   RecordBubbleSizes=rbub)
    planes = slice(0, 1024, 73)  # of both parities
    with D2Z(lp) as d:
        d.generate_delta(3)
        ref = None
        for x in (PLAN_MATRIX, PLAN_VECTOR):
            for z in (PLAN_MATRIX, PLAN_VECTOR):
                announce(f"half planes x={x} z={z} rbub={rbub}")
                d.set_plan(x, z, 2)
                d.run()
                got = d.zreion()[planes].astype(np.float64)
                if ref is None:
                    ref = got
                    assert ref.std() > 0.1
                assert np.sqrt(np.mean((got - ref) ** 2)) <= RMS, (x, z)
