"""bench.py quotes a committed traffic figure only for the kernels it was measured on."""

from __future__ import annotations

import importlib


def test_traffic_is_null_when_the_kernels_have_changed(tmp_path):
    bench = importlib.import_module("bench")
    none = {"traffic": None, "traffic_kernel": None, "traffic_commit": None}
    assert bench._traffic_from_profiles("x", tmp_path) == none
    body = "# a comment: with a colon\ndominant_kernel: k<1>\ncommit: abc\ntraffic_bytes_per_launch: 12\n"
    (tmp_path / "traffic_x.txt").write_text(body)
    assert bench._traffic_from_profiles("x", tmp_path) == none
    (tmp_path / "traffic_x.txt").write_text(body + "sources: 0123\n")
    assert bench._traffic_from_profiles("x", tmp_path) == none
    (tmp_path / "traffic_x.txt").write_text(body + f"sources: {bench._kernel_sources_hash()}\n")
    assert bench._traffic_from_profiles("x", tmp_path) == {
        "traffic": 12.0, "traffic_kernel": "k<1>", "traffic_commit": "abc"}


def test_hash_follows_code_and_not_comments(tmp_path):
    bench = importlib.import_module("bench")
    src = tmp_path / "a.hip"
    src.write_text("int x;  // one\n")
    first = bench._kernel_sources_hash(tmp_path)
    src.write_text("// two\nint  x;\n")
    assert bench._kernel_sources_hash(tmp_path) == first
    src.write_text("int y;\n")
    assert bench._kernel_sources_hash(tmp_path) != first
