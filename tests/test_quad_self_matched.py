"""Decomposition of meshes with triangles that repeat an index (which are their
own neighbours, and which the matching can pair with themselves): the search
for augmenting paths ends wherever it meets them, and every triangle is in one
quad at most.  On the host in a process with a time and memory limit; on the
device with the same quads."""

from __future__ import annotations

import os
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest

from rasterizer_amd import QuadDecomposition, Rasterizer

ROOT = Path(__file__).resolve().parent.parent


def meshes():
    V = np.ones((4, 4), np.float32)
    V[:, :3] = [[0, 0, 0], [0.3, 0, 0], [0, 0, 0.3], [0.2, 0, 0.2]]
    yield np.array([[3, 0, 0], [0, 0, 3], [3, 2, 0]]), V
    for seed in range(200):
        rng = np.random.default_rng(seed)
        nv, nt = int(rng.integers(3, 30)), int(rng.integers(2, 120))
        V = np.ones((nv, 4), np.float32)
        V[:, :3] = rng.uniform(-0.4, 0.4, (nv, 3))
        tri = rng.integers(0, nv, (nt, 3))
        if seed % 2:  # a few such triangles among proper ones
            tri = np.argsort(rng.random((nt, nv)), axis=1)[:, :3]
            k = rng.random(nt) < 0.15
            tri[k, 2] = tri[k, 0]
        yield tri, V


def check(tri, V):
    quads = QuadDecomposition.decompose(tri, V).size // 4
    repeats = (tri[:, 0] == tri[:, 1]) | (tri[:, 1] == tri[:, 2]) | (tri[:, 2] == tri[:, 0])
    # Only a triangle that is matched with itself is in no quad.
    assert len(tri) - int(repeats.sum()) <= 2 * quads and quads <= len(tri)


def test_search_ends():
    code = ("import resource; resource.setrlimit(resource.RLIMIT_AS, (8 << 30, 8 << 30))\n"
            "import test_quad_self_matched as t\n"
            "for m in t.meshes(): t.check(*m)\n"
            "print('done')")
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT / "tests", env={**os.environ,
                       "PYTHONPATH": str(ROOT)}, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "done" in r.stdout, r.stderr[-2000:]


@pytest.mark.gpu
def test_device_gives_the_same():
    r = Rasterizer(64, 64)
    for tri, V in meshes():
        assert np.array_equal(r.quad_decompose_device(tri, V), QuadDecomposition.decompose(tri, V))
