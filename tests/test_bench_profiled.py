"""bench.py finds the committed counters of the sub-sweep and measuring-stage kernels that a lattice's
size picks, and of no others."""
import json
import os
import sys

import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402

N = (8, 8, 8, 8)
FIGURES = {"waves": 1.0, "valu_per_wave": 2.0, "traffic_bytes": 3.0}


@pytest.mark.parametrize("name, found", [("metropolis_kernel<float, 2, 3>", True),
                                         ("metropolis_kernel<float, 2, 8>", True),
                                         ("metropolis_small_kernel<float, 2, 3, 5>", True),
                                         ("metropolis_kernel<float, 3, 4>", False),
                                         ("metropolis_kernel<double, 3, 2>", False),
                                         ("metropolis_learned_kernel<float, 2, 3>", False)])
def test_sweep_kernel(tmp_path, monkeypatch, name, found):
    os.makedirs(tmp_path / "profiles")
    with open(tmp_path / "profiles" / "counters_8x8x8x8.json", "w") as f:
        json.dump({"kernels": {name: FIGURES, "flow_stage_kernel<float, 2, 1, false>": FIGURES}}, f)
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))
    assert bench.profiled(N, [bench.sweep_kernel(2)]) == (FIGURES if found else None)


@pytest.mark.parametrize("name, found", [("flow_stage_kernel<float, 2, 0, true>", True),
                                         ("flow_stage_kernel<float, 2, 0, true, 3u, false>", True),
                                         ("flow_measure_wide_kernel<float, 2>", True),
                                         ("flow_stage_kernel<float, 2, 0, false>", False),
                                         ("flow_measure_wide_kernel<double, 3>", False)])
def test_measuring_stage(tmp_path, monkeypatch, name, found):
    os.makedirs(tmp_path / "profiles")
    with open(tmp_path / "profiles" / "counters_8x8x8x8.json", "w") as f:
        json.dump({"kernels": {name: FIGURES}}, f)
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))
    assert bench.profiled(N, [bench.stage0_kernel(2)]) == (FIGURES if found else None)


def test_committed_counters():
    n = (32, 32, 32, 32)
    assert bench.profiled(n, [bench.sweep_kernel(2)])["waves"] == 8192
    assert bench.profiled(n, [bench.plain_stage_kernel(2, k) for k in (1, 2)])["waves"] == 65536
    assert bench.profiled(n, [bench.stage0_kernel(2)])["waves"] == 65536
    assert bench.profiled(n, [bench.plain_stage_kernel(3, 1)]) is None
