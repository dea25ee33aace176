"""The device bake around the size up to which an occluder is baked in LDS
(1,024 quads), alone and mixed with larger and smaller ones in one call,
against the host bake bit for bit."""

from __future__ import annotations

import numpy as np
import pytest

from rasterizer_amd import Occluder, Rasterizer

pytestmark = pytest.mark.gpu


def _mesh(rng, quads, clusters):
    """Quads facing a few directions, so that k-means moves some of them."""
    n = rng.normal(size=(clusters, 3))
    f = n[rng.integers(0, clusters, quads)] + 0.4 * rng.normal(size=(quads, 3))
    u = np.cross(f, rng.normal(size=(quads, 3)))
    w = np.cross(f, u)
    c = rng.uniform(-50, 50, (quads, 3))
    v = np.ones((quads, 4, 4), np.float32)
    for k, (a, b) in enumerate(((-1, -1), (1, -1), (1, 1), (-1, 1))):
        v[:, k, :3] = c + a * u + b * w
    return v.reshape(-1, 4)


@pytest.mark.parametrize("sizes", [[8], [64], [72], [1016], [1024], [1032], [2048, 8, 1024], [1024, 3000, 512, 64]])
def test_sizes_match_host_bake(sizes):
    rng = np.random.default_rng(len(sizes) * 1000 + sizes[0])
    meshes = [_mesh(rng, n, k % 3 * 4 + 2) for k, n in enumerate(sizes)]
    lo = [m.min(axis=0) - 1 for m in meshes]
    hi = [m.max(axis=0) + 1 for m in meshes]
    got = Rasterizer(64, 64).bake_device(meshes, lo, hi)
    for m, a, b, g in zip(meshes, lo, hi, got):
        h = Occluder.bake(m, a, b)
        assert np.array_equal(g.packets, h.packets)
        for f in ("m_boundsMin", "m_boundsMax", "m_center"):
            assert np.array_equal(getattr(g, f).view(np.uint32), getattr(h, f).view(np.uint32)), f
