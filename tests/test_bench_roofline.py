"""The roofline record of bench.py: the rate achieved is that of the bytes that
moved, and the algorithmic bytes' rate stands beside it under its own name."""
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402


def test_achieved_is_the_measured_traffic():
    r = bench.roofline_of(10.8e9, 21.4e9, 5.6)
    assert r["achieved"] == round(10.8e9 / 5.6e-3 / 1e9, 1) and r["frac"] == round(r["achieved"] / 8000.0, 4)
    assert r["algorithmic"]["rate"] == round(21.4e9 / 5.6e-3 / 1e9, 1) and r["traffic"] == 10800000000


def test_nothing_is_claimed_without_a_profile():
    r = bench.roofline_of(None, 21.4e9, 5.6)
    assert r["achieved"] is None and r["frac"] is None and r["traffic"] is None
    assert r["algorithmic"]["rate"] > 0
