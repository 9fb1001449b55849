"""bench.py describes the arithmetic and the traffic of the FFT plans that ran, on the CPU."""
import json
import sys

import pytest

from conftest import ROOT

sys.path.insert(0, str(ROOT))
import bench  # noqa: E402

PLANS = [{"x": x, "z": z} for x in ("vector", "matrix") for z in ("vector", "matrix")]


@pytest.mark.parametrize("mode", ["mixed", "half"])
@pytest.mark.parametrize("plans", PLANS)
def test_dtype_follows_the_plans(mode, plans):
    on = [a for a in ("x", "z") if plans[a] == "matrix"]
    text = bench.dtype_of(mode, plans)
    assert ("matrix" in text) == bool(on)
    assert ("split hi/lo" in text) == (mode == "mixed" and bool(on))
    if on:
        assert f"stages of {' and '.join(on)} " in text
    assert text.startswith("f16" if mode == "half" else "f32")


def test_dtype_without_plans():
    assert bench.dtype_of("plain", None) == bench.dtype_of("fused", PLANS[0]) == "f32"


def test_plan_names():
    assert bench.plan_names({"x_plan": 1, "z_plan": 0, "x_radii_per_launch": 16}) == {"x": "matrix", "z": "vector"}
    assert bench.plan_names(None) is None


@pytest.mark.parametrize("mode", ["mixed", "fused", "half"])
@pytest.mark.parametrize("plans", PLANS)
def test_traffic_is_the_plans_own(mode, plans):
    """A profile is used only for the plans it was taken with, which its commands fix."""
    prof = bench.traffic_profile("c3_1024", mode, plans)
    if not prof:
        return
    about = prof["_about"]
    assert about["fft_plans"] == plans
    flag = f"--plan {plans['x']},{plans['z']}"
    for c in ("fetch_command", "write_command"):
        assert f"--mode {mode}" in about[c]
        # without the flag and the tuner: the fused mode, which has the vector plans only
        assert flag in about[c] or (mode == "fused" and "--plan" not in about[c] and "--no-tune" in about[c])


def test_traffic_of_the_measured_plans():
    """The mixed step's two x passes and the half path's matrix passes have a profile each; the
    split z pass has none."""
    v, m = PLANS[0], {"x": "matrix", "z": "vector"}
    mixed = [bench.traffic_profile("c3_1024", "mixed", p) for p in (v, m)]
    assert all(mixed) and mixed[0] != mixed[1]
    assert bench.traffic_profile("c3_1024", "mixed") == mixed[0]
    assert bench.traffic_profile("c3_1024", "half", {"x": "matrix", "z": "matrix"})
    assert bench.traffic_profile("c3_1024", "mixed", {"x": "matrix", "z": "matrix"}) == {}
    assert bench.traffic_profile("no_such_workload", "mixed", v) == {}
    assert json.loads((ROOT / "profiles" / "traffic_c3_1024_mixed_matrix_x.json").read_text())["_about"]["fft_plans"] == m
