"""The bench reports counted HBM traffic only for the kernels as they were counted."""
import json
import os

import pytest

import bench

W, K = "w", "k_radix_pass<u32 key, u32 value>"


@pytest.fixture
def tree(tmp_path, monkeypatch):
    src = tmp_path / "libsais_amd" / "csrc"
    os.makedirs(src)
    os.makedirs(tmp_path / "profiles")
    for name in ("radix.hip", "rounds.hip", "engine.h", "common.h"):
        (src / name).write_text(f"int a;  // {name}\n")
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))
    (tmp_path / "profiles" / "pmc_traffic.json").write_text(
        json.dumps({"workload": W, "code": {K: bench.kernel_code(K)}, "bytes_per_launch": {K: 7, "k_round_tile": 8}}))
    return src


def test_traffic_of_counted_code(tree):
    assert bench.measured_traffic(W, K) == 7
    assert bench.measured_traffic("other", K) is None
    assert bench.measured_traffic(W, "k_round_tile") is None      # no record of its code


@pytest.mark.parametrize("name,text,want", [
    ("radix.hip", "int a;\n// another comment\n", 7),
    ("rounds.hip", "int b;\n", 7),
    ("radix.hip", "int b;\n", None),
    ("engine.h", "int a, c;\n", None),
])
def test_traffic_after_a_change(tree, name, text, want):
    (tree / name).write_text(text)
    assert bench.measured_traffic(W, K) == want


def test_every_timed_kernel_has_a_source():
    for k in bench.KERNELS:
        assert len(bench.kernel_code(k)) == 16
