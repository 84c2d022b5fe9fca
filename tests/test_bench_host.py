"""bench.py's account of the dominant kernel, without a GPU: which kernel a
persistent solve ran on, its milliseconds and its share of the attempts, also
when no cell was handed off (the hand-off's statistics are then zero)."""
import sys
from pathlib import Path

import pytest

sys.path.insert(0, str(Path(__file__).resolve().parent.parent))
import bench  # noqa: E402


@pytest.mark.parametrize("cfg,ho,name,ms,away", [
    ({"wave_per_cell": 1, "variant": 7}, (0, 0, 0.0, 0.0), "k_wave", 593.0, 0),
    ({"wave_per_cell": 1, "variant": 7}, None, "k_wave", 593.0, 0),
    ({"wave_per_cell": 0, "variant": 4}, None, "k_persist", 593.0, 0),
    ({"wave_per_cell": 0, "variant": 4}, (0, 0, 0.0, 0.0), "k_persist", 593.0, 0),
    ({"wave_per_cell": 0, "variant": 4}, (98304, 700000, 400.0, 150.0), "k_persist", 400.0, 700000),
])
def test_dominant_kernel(cfg, ho, name, ms, away):
    kernel, kms, other = bench.dominant_kernel(cfg, 593.0, ho)
    assert kernel.startswith(name) and kms == ms and other == away


def test_no_hand_off_is_reported_as_none():
    assert bench.handoff_report(98304, (0, 0, 0.0, 0.0), 593.0) is None
    assert bench.handoff_report(0, None, 593.0) is None
    r = bench.handoff_report(98304, (1000.0, 5000.0, 400.0, 150.0), 560.0)
    assert r == {"max_cells": 98304, "cells_handed_off": 1000, "cell_per_wave_attempts": 5000,
                 "lane_launch_ms": 400.0, "cell_per_wave_launch_ms": 150.0, "integrate_ms": 560.0}


def test_split_is_named_only_where_there_is_one():
    assert "lane kernel" in bench.split_report({"wave_per_cell": 0}, 4096)
    assert "lane kernel" not in bench.split_report({"wave_per_cell": 1}, 4096)
    assert bench.split_report({"wave_per_cell": 0}, 0) == "one persistent kernel, class order"
