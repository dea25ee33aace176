"""Query answers of multi-view steps as they come back to the host: in any order
of the views and more than once, several views a copy, views without queries and
one with more than the pinned buffer holds among them, after another step and
after a view's number of queries changed.  Each view against a context of its own
that draws the same frames (clear leaves the depth, which queries of blocks not
drawn since read)."""

from __future__ import annotations

import numpy as np
import pytest

from rasterizer_amd import Rasterizer, Views, scenes

pytestmark = pytest.mark.gpu

W, H = 128, 64
COUNTS = [0, 1, 63, 64, 0, 0, 1100000, 65, 1000] + [30000 + k for k in range(40)] + [0, 70000, 0]


class World:
    def __init__(self):
        sc = scenes.config1(seed=11, n_boxes=40, width=W, height=H, n_queries=4096)
        self.pool = np.tile(sc.meta["queries"], (300, 1))
        self.occluders = sc.occluders
        self.singles = [Rasterizer(W, H) for _ in COUNTS]
        self.views = Views(self.singles[0], [(W, H)] * len(COUNTS))
        self.views.set_query_gated(True)
        self.counts = list(COUNTS)
        for k, n in enumerate(COUNTS):
            self.views.set_occluders(k, sc.occluders)
            self.set_count(k, n)

    def set_count(self, k, n):
        self.counts[k] = n
        self.views.set_queries(k, self.pool[k:k + n])

    def step(self, step):
        for k in range(len(COUNTS)):
            a = 10.0 * ((k + step) % 4)
            mvp = scenes.view_projection([a, 5.0, -60.0], [0.2 - 0.01 * a, -0.05, 1.0], [0.0, 1.0, 0.0], np.pi / 3, W / H)
            self.views.set_mvp(k, mvp)
            self.singles[k].clear()
            self.singles[k].setModelViewProjection(mvp)
            self.singles[k].draw_frame(self.occluders, want_status=False)
        self.views.run()
        self.views.sync()

    def want(self, k):
        n = self.counts[k]
        return self.singles[k].query_batch(self.pool[k:k + n]) if n else (np.zeros(0, bool), np.zeros(0, bool))


def _same(got, want, what):
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1]), what


def test_answers_in_any_order():
    w = World()
    rng = np.random.default_rng(3)
    views = np.arange(len(COUNTS))
    for step, order in enumerate((views, rng.permutation(views), np.repeat(views, 2), views[::-1],
                                  np.concatenate([views[:20], views[:3], views[10:]]))):
        w.step(step)
        want = {int(k): w.want(k) for k in order}
        for k in order:
            _same(w.views.queries(int(k)), want[int(k)], f"step {step}, view {k}")
        assert any(v.any() and not v.all() for v, _ in want.values())


def test_changed_count():
    w = World()
    changed = 12
    assert not any(a.any() for a in w.views.queries(changed)), "before any step"
    for step, count in enumerate((40, 0, 1200000, COUNTS[changed])):
        w.step(step)
        _same(w.views.queries(changed), w.want(changed), f"step {step}")
        w.set_count(changed, count)
        # Until the next step: none for the view, the others' as they were.
        _same(w.views.queries(changed), (np.zeros(count, bool),) * 2, "changed")
        for k in (13, 11, 20):
            _same(w.views.queries(k), w.want(k), f"step {step}, view {k} after the change")
    w.step(5)
    for k in range(8, 24):
        _same(w.views.queries(k), w.want(k), f"view {k}")
