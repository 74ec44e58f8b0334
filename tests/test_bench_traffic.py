"""The bench reports measured HBM traffic only for the launch that it was
measured on: same workload, state and sweep, same algorithmic bytes, same
tile shape."""
import json
import os
import types

import pytest

import bench


@pytest.fixture
def args(tmp_path):
    path = tmp_path / "traffic.json"
    path.write_text(json.dumps({"operational:fp32:sweep_z": {
        "tile": "4/1", "algorithmic_bytes": 684288000, "bytes_per_launch": 776000000}}))
    return types.SimpleNamespace(traffic=str(path))


@pytest.mark.parametrize("key,alg,tile,expected", [
    ("operational:fp32:sweep_z", 684288000.0, "4/1", 776000000),
    ("operational:fp32:sweep_z", 684288000.0, "8/2", None),
    ("operational:fp32:sweep_z", 684288000.0, "8/1", None),
    ("operational:fp32:sweep_z", 684300000.0, "4/1", None),
    ("operational:fp32:sweep_y", 684288000.0, "4/1", None),
])
def test_traffic_only_for_the_measured_launch(args, key, alg, tile, expected):
    assert bench._traffic(args, key, alg, tile) == expected


def test_every_committed_entry_names_its_shape():
    with open(os.path.join(bench.ROOT, "profiles", "traffic.json")) as f:
        entries = json.load(f)
    assert entries
    for key, e in entries.items():
        axis = "xyz".index(key[-1])
        assert e["tile"].count("/") == (0 if axis == 0 else 1), key
        assert e["algorithmic_bytes"] <= e["bytes_per_launch"], key


def test_tile_is_what_set_tiling_takes():
    g = types.SimpleNamespace(tiling=lambda axis: ((6, 4), (2, 8), (1, 4))[axis])
    assert [bench._tile(g, d) for d in range(3)] == ["6", "8/2", "4/1"]
