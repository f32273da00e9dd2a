"""The benchmark quotes committed counters of the very kernel it runs, or none."""

from __future__ import annotations

import json

import bench


def test_counters_are_those_of_the_kernel_that_runs(tmp_path, monkeypatch):
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))
    (tmp_path / "profiles").mkdir()
    table = {"sw_affine_scaled_fused_kernel<4, 8>": 1, "sw_affine_scaled_fused_kernel<4, 16, true>": 2,
             "sw_affine_scaled_forward_kernel<true, 8, 8, true>": 3}
    (tmp_path / "profiles" / "x.md").write_text("text\n\ntag: " + json.dumps(table) + "\n")
    assert bench._profiled("x.md", "tag", "fused", (4, 16))[0] == 2
    assert bench._profiled("x.md", "tag", "forward", (8, 8))[0] == 3
    for shape in ((4, 8), (8, 16), None):  # another template, another shape, no shape
        assert bench._profiled("x.md", "tag", "fused", shape) == (None, None)
    assert bench._profiled("y.md", "tag", "fused", (4, 16)) == (None, None)
