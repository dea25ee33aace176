"""The device bake of many small occluders, whose launch takes the LDS that the
largest one needs: alone, with a few that are larger, and with ones that are
baked outside the LDS, against the host bake bit for bit."""

from __future__ import annotations

import numpy as np
import pytest

from rasterizer_amd import Occluder, Rasterizer
from test_gpu_bake_sizes import _mesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [[8] * 700, [8, 16, 24] * 100, [8] * 300 + [1024] + [16] * 300, [1032] * 3,
                                   [1032] + [8] * 300, [40] * 50 + [1600, 1016]])
def test_small_occluders_match_host_bake(sizes):
    rng = np.random.default_rng(sum(sizes))
    meshes = [_mesh(rng, n, k % 3 * 4 + 2) for k, n in enumerate(sizes)]
    lo = [m.min(axis=0) - 1 for m in meshes]
    hi = [m.max(axis=0) + 1 for m in meshes]
    for m, a, b, g in zip(meshes, lo, hi, Rasterizer(64, 64).bake_device(meshes, lo, hi)):
        h = Occluder.bake(m, a, b)
        assert np.array_equal(g.packets, h.packets)
        for f in ("m_boundsMin", "m_boundsMax", "m_center"):
            assert np.array_equal(getattr(g, f).view(np.uint32), getattr(h, f).view(np.uint32)), f
