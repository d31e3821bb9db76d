"""bench.py's `roofline` object: the bytes behind `achieved` are bytes that the launch moves."""

import pytest
import torch

import bench


def _diag(members, launches):
    i = lambda v: torch.full((members,), v, dtype=torch.int32)  # noqa: E731
    return {"numIters": i(100), "outerIters": i(4), "launches": i(launches)}


@pytest.mark.parametrize("precision,ms", [("mixed", 7.0), ("fp64", 9.5)])
def test_resident_launch_counts_what_it_moves(precision, ms):
    """A resident launch is bound by latency; its achieved bandwidth is the measured traffic over the time (null for another
    number of members, which is not measured), the recurrence's bytes stand beside it."""
    r = bench.roofline_of(precision, ms, _diag(128, 0), None, 128, "auto")
    assert r["bound"] == "latency" and r["kernel"] == ("mx" if precision == "mixed" else "cg2d") + "_resident_kernel"
    assert r["achieved"] == pytest.approx(r["traffic"] / ms * 1e-6)
    assert r["frac"] == pytest.approx(r["achieved"] / r["peak"]) and r["frac"] < 0.5
    assert r["algorithmic_GBs"] == pytest.approx(r["algorithmic_bytes"] / ms * 1e-6)
    r = bench.roofline_of(precision, ms, _diag(32, 0), None, 32, "auto")
    assert r["bound"] == "latency" and r["traffic"] is None and r["achieved"] is None and r["frac"] is None


@pytest.mark.parametrize("precision,launches,launch", [("mixed", 300, "phases"), ("fp64", 200, "phases"),
                                                       ("fp64", 0, "persistent")])
def test_streaming_launches_count_the_recurrence(precision, launches, launch):
    r = bench.roofline_of(precision, 20.0, _diag(128, launches), None, 128, launch)
    assert r["bound"] == "hbm"
    assert r["achieved"] == pytest.approx(r["algorithmic_bytes"] / 20.0 * 1e-6)
    assert r["frac"] == pytest.approx(r["achieved"] / r["peak"])
