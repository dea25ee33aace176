"""The device decomposition's adjacency lists where their order matters:
triangles that repeat, that hold an edge and its reverse, edges shared by many
triangles in both directions, and vertex counts around a power of two (the
width of a half-edge's key), against the host decomposition; and calls of
different sizes in turn on one context, whose working memory is kept between
them."""

from __future__ import annotations

import numpy as np
import pytest

from rasterizer_amd import QuadDecomposition, Rasterizer, scenes
from test_gpu_sah import _same_occluders

pytestmark = pytest.mark.gpu


def _mesh(vertices, triangles):
    rng = np.random.default_rng(vertices * 1000 + triangles)
    V = np.ones((vertices + 3, 4), np.float32)
    V[:, :3] = rng.uniform(-0.4, 0.4, (vertices + 3, 3))  # near enough for most plane tests to pass
    V[rng.random(vertices + 3) < 0.2, 1] += 5.0
    tri = np.argsort(rng.random((triangles, vertices)), axis=1)[:, :3]
    # Triangles that are their own neighbours, on vertices of their own: the
    # matching pairs each with itself.
    own = np.array([[0, 1, 0], [2, 2, 2]]) + vertices
    return np.insert(tri, triangles // 2, own, axis=0).astype(np.uint32), V


@pytest.mark.parametrize("vertices", [3, 4, 5, 6, 13, 61, 62, 254])
@pytest.mark.parametrize("triangles", [1, 3, 86, 700])
def test_shared_edges(vertices, triangles):
    tri, V = _mesh(vertices, triangles)
    got = Rasterizer(64, 64).quad_decompose_device(tri, V)
    assert np.array_equal(got, QuadDecomposition.decompose(tri, V))


def test_sizes_in_turn():
    r = Rasterizer(64, 64)
    for n in (40, 200, 3, 90, 200, 40):
        tri, V = scenes.triangulated_boxes(np.random.default_rng(n), n)
        assert np.array_equal(r.quad_decompose_device(tri, V), QuadDecomposition.decompose(tri, V))
        want = scenes.bake_scene(scenes.decompose_mesh(tri, V), vertex_buffer=V).occluders
        _same_occluders(r.prepare_mesh_device(tri, V), want)
