"""The x passes with the longest W(x) tables their LDS takes (3584 intervals, 3184 for
the split matrix-core pass): the largest radius is set so that the table ends within
20 intervals of that.

Reference: the plain path on the same field, which evaluates W(x) itself.  The table
at h = 1/4 errs by at most 8.7e-7 (9.6e-8 at 1/8) of a mode's amplitude; with cells
of rms 2.4 that is 1.3e-5 of delta_R at six sigma, and z = A delta_R + .. with A below
1: 2e-5 with the FP32 transforms' rounding.  FP16 storage: the 0.02 of the half path.
"""
import math

import numpy as np
import pytest
import torch

from _cases import box_for, lib_params
from conftest import announce
from prc_d2z import D2Z, FUSED_FP32, FUSED_HALF, FUSED_MIXED, Group, PLAIN_FP32, PLAN_MATRIX, PLAN_VECTOR

pytestmark = pytest.mark.gpu


def _rmax(N, entries, h):
    """Rmax whose table has 6 to 20 intervals fewer than `entries`: x = dk R sqrt(3) N/2 1.001 + 1."""
    x = (entries - 10) * h
    rmax = (x - 1.0) / 1.001 / (math.sqrt(3.0) * N / 2) / (2.0 * math.pi) * box_for(N)
    got = math.ceil((2.0 * math.pi / box_for(N) * rmax * math.sqrt(3.0) * N / 2 * 1.001 + 1.0) / h) + 1
    assert entries - 20 <= got <= entries - 6
    return rmax


class _Field:
    def __init__(self, d):
        self.__cuda_array_interface__ = {"shape": (d.N, d.N, d.N), "typestr": "<f4",
                                         "data": (d.zreion_device_ptr(), False), "version": 2}


def _zreion(lp, plan=None):
    """Every 16th x plane of one run's zreion."""
    with D2Z(lp) as d:
        d.generate_delta(2)
        if plan:
            d.set_plan(*plan, 16)
        d.run()
        return torch.as_tensor(_Field(d), device="cuda")[::16].clone()


@pytest.mark.parametrize("N,entries,h,runs", [
    (256, 3584, 0.125, [(FUSED_FP32, None, 2e-5), (FUSED_HALF, None, 0.02)]),
    (512, 3584, 0.25, [(FUSED_FP32, None, 2e-5), (FUSED_HALF, None, 0.02)]),
    (1024, 3584, 0.25, [(FUSED_FP32, None, 2e-5), (FUSED_HALF, (PLAN_VECTOR, PLAN_VECTOR), 0.02),
                        (FUSED_HALF, (PLAN_MATRIX, PLAN_VECTOR), 0.02)]),
    (1024, 3184, 0.25, [(FUSED_MIXED, (PLAN_MATRIX, PLAN_VECTOR), 2e-5), (FUSED_MIXED, (PLAN_VECTOR, PLAN_VECTOR), 2e-5)]),
    (2048, 3584, 0.25, [(FUSED_FP32, None, 2e-5), (FUSED_HALF, (PLAN_MATRIX, PLAN_VECTOR), 0.02),
                        (FUSED_HALF, (PLAN_VECTOR, PLAN_VECTOR), 0.02)]),
])
def test_longest_table(N, entries, h, runs):
    def lp(mode):
        return lib_params(N, nscales=2, mode=mode, rmax=_rmax(N, entries, h))

    announce(f"long W table N={N} plain")
    ref = _zreion(lp(PLAIN_FP32))
    assert float(ref.max()) > 1.0  # cells above the barrier
    for mode, plan, tol in runs:
        announce(f"long W table N={N} mode={mode} plan={plan}")
        dz = float((_zreion(lp(mode), plan) - ref).abs().max())
        print(f"N={N} mode={mode} plan={plan}: max |dz| {dz:.2e}")
        assert dz <= tol


def test_longest_table_in_a_group():
    """Group launches take the longest table of their boxes; each box's bits are its own run's."""
    announce("long W table, group")
    boxes, alone = [], []
    for N in (64, 256, 256):
        d = D2Z(lib_params(N, nscales=3, mode=FUSED_FP32, rmax=_rmax(256, 3584, 0.125) if N == 256 else 20.0))
        d.generate_delta(N + len(boxes))
        d.run()
        alone.append(d.zreion())
        boxes.append(d)
    with Group(boxes) as g:
        g.run()
        for d, z in zip(boxes, alone):
            assert np.array_equal(d.zreion(), z)
    for d in boxes:
        d.close()
