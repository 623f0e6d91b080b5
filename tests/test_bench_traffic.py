"""The measured traffic that bench.py reports beside a launch's algorithmic bytes."""
import os
import sys

import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402


def test_traffic_of_another_launch_is_not_reported():
    """6.63 GB must move in a launch of three fields: 2.25 GB was measured per field"""
    rows = [("z_s2x_dual", 8, 8 * 3.2, 8 * 6.6255e9)]
    assert bench._roofline(rows, {"z_s2x_dual": 2.246e9})["traffic"] is None
    assert bench._roofline(rows, {})["traffic"] is None
    assert bench._roofline(rows, {"z_s2x_dual": 6.75e9})["traffic"] == 6750000000


# bytes one launch must move at 512 x 512 x (512 + 25), d = 5: all fields of a pass
CB = 16 * 537 * 512 * 257          # a float64 spectral field
XP = {"mixed": 8, "fp64": 16}      # bytes of an xy-stage value, of 512 * 257 * 512


@pytest.mark.parametrize("mode", ["mixed", "fp64"])
def test_committed_traffic_is_per_launch_of_all_fields(mode):
    xp = XP[mode] * 512 * 512 * 257
    t = bench._measured_traffic("hd512", mode)
    assert t["z_s2x_dual"] > 0.95 * 3 * (CB + 2 * xp)
    assert t["y_dual"] > 0.95 * 15 * xp
    assert t["xgrad_fused"] > 0.95 * 12 * xp
    assert t["z_x2s"] > 0.95 * 3 * (xp + CB * XP[mode] / 16)
