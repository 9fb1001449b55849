"""The autotuner's cache file on the CPU: a choice is reused by the build of the library
that stored it, and by no other."""
import json
from types import SimpleNamespace

import prc_d2z
from prc_d2z import D2Z

TUNED = {"radii_per_launch": 32, "z_blocks": 1024, "x_plan": 0, "z_plan": 0, "x_radii_per_launch": 16}


class _Lib:
    """Stands for a loaded library whose file is `path`; counts the tuner's runs."""

    def __init__(self, path):
        self._name = str(path)
        self.runs = 0
        self.set = []

    def prc_d2z_autotune(self, ctx, t):
        self.runs += 1
        for k, v in TUNED.items():
            setattr(t._obj, k, v)
        return 0

    def prc_d2z_set_plan(self, ctx, *a):
        self.set.append(a)
        return 0

    def prc_d2z_set_launch_config(self, ctx, *a):
        self.set.append(a)
        return 0


def _context(lib):
    d = D2Z.__new__(D2Z)
    d.lib, d._ctx, d.N = lib, None, 1024
    d.params = SimpleNamespace(device=0, mode=prc_d2z.FUSED_MIXED)
    return d


def test_a_choice_belongs_to_its_build(tmp_path):
    cache, so = tmp_path / "plans.json", tmp_path / "lib.so"
    # a file of an earlier format: its key names no build
    cache.write_text(json.dumps({"0:N1024:mode2": dict(TUNED, x_plan=1, z_plan=1, ms_per_radius=1.0)}))
    so.write_bytes(b"one build")
    a = _Lib(so)
    t = _context(a).autotune(cache)
    assert a.runs == 1 and not t["cached"] and (t["x_plan"], t["z_plan"]) == (0, 0)
    t = _context(a).autotune(cache)
    assert a.runs == 1 and t["cached"] and a.set == [(0, 0, 16), (32, 1024)]
    so.write_bytes(b"another build")
    b = _Lib(so)
    assert not _context(b).autotune(cache)["cached"] and b.runs == 1
    assert _context(b).autotune(cache)["cached"] and b.runs == 1
    assert len(json.loads(cache.read_text())) == 3


def test_no_cache_tunes_each_time(tmp_path):
    a = _Lib(tmp_path / "missing.so")
    d = _context(a)
    assert not d.autotune()["cached"] and not d.autotune()["cached"] and a.runs == 2
