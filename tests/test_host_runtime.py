"""The C ABI's host side against a HIP runtime in host memory (defined in
tests/cpp/host_runtime_check.cpp, which needs no GPU): what is allocated when,
what happens when an allocation fails, and that what is freed was allocated."""

from __future__ import annotations

import subprocess
from pathlib import Path

import pytest

from rasterizer_amd import build

PROG = Path(__file__).resolve().parent / "_bin" / "host_runtime_check"


@pytest.mark.parametrize("check", ["blocking_calls", "error_left_behind", "failed_creation", "scratch",
                                   "scene_box_sizes", "no_host_memory", "failed_growth", "failed_plans",
                                   "view_answers", "growing_calls"])
def test_host_runtime(check):
    if not PROG.exists():
        build.build()
    r = subprocess.run([str(PROG), check], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
