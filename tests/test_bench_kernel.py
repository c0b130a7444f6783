"""bench.py names and prices the kernel that a plain render ran in: path launches,
whichever statistics fields the library counts them in."""
import importlib.util
import os

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def bench():
    spec = importlib.util.spec_from_file_location("bench_module", os.path.join(ROOT, "bench.py"))
    m = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(m)
    return m


def totals(**kw):
    t = dict(segments=3_000_000, paths=1_000_000, trace_ms=0.0, shade_ms=0.0, trace_launches=0, shade_launches=0,
             tail_segments=0, tail_ms=0.0, tail_launches=0)
    t.update(kw)
    return t


@pytest.mark.parametrize("t", [
    totals(tail_segments=3_000_000, tail_ms=40.0, tail_launches=4),  # constant textures, one light
    totals(trace_ms=40.0, trace_launches=4),                         # textures, media, light lists, general walk
])
def test_path_launches_are_named_and_priced_as_such(bench, t):
    assert bench.timed_kernel(t) == ("k_paths", 40.0, 4)
    r = bench.roofline("no_such_scene", 100, t)
    assert r["kernel"] == "k_paths" and r["avg_launch_ms"] == 10.0
    assert r["bytes_per_launch"] == 12 * 1_000_000 / 4
    assert r["hbm"]["achieved"] == pytest.approx(12 * 1_000_000 / 0.04 / 1e9, abs=0.01)
    assert r["achieved"] is None and r["traffic"] is None  # no counter profile of that frame


def test_headline_rate_is_of_the_kernel_that_ran(bench):
    t = totals(tail_segments=3_000_000, tail_ms=1.0, tail_launches=1)
    r = bench.roofline("cornell555", 1200, t)
    ops = r["executed_lane_ops_per_segment"]
    assert r["bound"] == "valu" and ops > 100
    assert r["achieved"] == pytest.approx(ops * 3e6 / 1e-3 / 1e12, rel=1e-3)
    assert 0 < r["traffic"] < 200 * t["paths"]
