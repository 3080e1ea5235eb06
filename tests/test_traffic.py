"""``bench.measured_traffic``: the counter summaries hold every kernel the
bench can name as dominant, and count for their own build alone."""

from __future__ import annotations

import json
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


@pytest.mark.parametrize("config", [2, 5])
def test_traffic_of_a_build(config, tmp_path, monkeypatch):
    import bench
    name = f"c{config}_traffic.json"
    d = json.loads((ROOT / "profiles" / name).read_text())
    assert {"k_pretok", "k_bpe_pack"} <= set(d["kernels"])
    (tmp_path / "profiles").mkdir()
    (tmp_path / "profiles" / name).write_text(json.dumps(d))
    lib = tmp_path / "toktier_amd" / "_lib"
    lib.mkdir(parents=True)
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))
    (lib / "manifest.json").write_text(json.dumps({"build_key": d["build_key"]}))
    for k, v in d["kernels"].items():
        assert bench.measured_traffic(config, k) == v["fetch_bytes"] + v["write_bytes"] > 0
    assert bench.measured_traffic(config, "k_other") is None
    (lib / "manifest.json").write_text(json.dumps({"build_key": "another"}))
    assert bench.measured_traffic(config, "k_pretok") is None
