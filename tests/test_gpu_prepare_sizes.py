"""Scene preparation on one context in calls of very different size: one that
uses more working memory than is kept between calls, a small one after it, the
large one again.  Each gives what a context of its own gives."""

from __future__ import annotations

import numpy as np
import pytest

from rasterizer_amd import Rasterizer, scenes

pytestmark = pytest.mark.gpu


def _boxes(n):
    rng = np.random.default_rng(n)
    unit = scenes.box_quads(np.zeros(3), np.ones(3))[None, :, :, :3]
    q = np.ones((n, 6, 4, 4), np.float32)
    q[..., :3] = rng.uniform(-300, 300, (n, 1, 1, 3)) + unit * rng.uniform(0.5, 5.0, (n, 1, 1, 3))
    return q.reshape(-1, 4, 4)


def _prepared(r, quads):
    occ = r.prepare_scene_device(quads)
    return (np.concatenate([o.packets.ravel() for o in occ]),
            np.array([[*o.m_boundsMin, *o.m_boundsMax, *o.m_center] for o in occ]))


def test_large_small_large():
    scenes_ = {n: _boxes(n) for n in (250000, 30)}
    want = {n: _prepared(Rasterizer(64, 64), q) for n, q in scenes_.items()}
    r = Rasterizer(64, 64)
    for n in (250000, 30, 250000, 30):
        got = _prepared(r, scenes_[n])
        assert all(np.array_equal(a, b) for a, b in zip(got, want[n])), f"{n} boxes"
