"""The block loop's counters: the (quad, block) pairs that a draw visits do not
depend on the order of the occluders or on what earlier ones cover (so reject
rates of different orders can be compared), each is rejected or written, and the
written ones are the reference's.  Single frames count the same as the same
frames as views, on both sides of the number of items from which a tile tests
item boxes."""

from __future__ import annotations

import math

import numpy as np
import pytest

from rasterizer_amd import Rasterizer, Views, scenes
from test_gpu_item_rounds import H, W, _occluders

pytestmark = pytest.mark.gpu

MVP = scenes.view_projection((0.0, 0.0, 0.0), np.array([0.0, 0.0, 1.0]), (0, 1, 0), math.pi / 8, W / H)


def _step(items, tile_w, waves, gated, order=None):
    V = Views(Rasterizer(64, 64), [(W, H)])
    V.set_config(waves, 0, tile_w)
    V.set_query_gated(gated)
    V.enable_stats(True)
    V.set_occluders(0, items)
    V.set_mvp(0, MVP)
    if order is not None:
        V.set_batch_order(0, order.permutation(V.n_batches(0)))
    V.run()
    V.sync()
    return V.stats()


@pytest.mark.parametrize("tile_w,waves", [(8, 8), (8, 2), (16, 8), (16, 4)])
def test_visited_pairs_do_not_depend_on_the_order(oracle_mod, tile_w, waves):
    items = _occluders(400, np.random.default_rng(5))
    for order in (items, items[::-1]):
        s = _step(order, tile_w, waves, False)
        o = oracle_mod.OracleRasterizer(W, H)
        o.clear()
        o.setModelViewProjection(MVP)
        before = o.stats()
        o.draw_frame(order, gated=False)
        written = o.stats()["written"] - before["written"]
        assert s["visited"] == s["rejected"] + s["written"] and s["written"] == written
        if order is items:
            first = s["visited"]
        assert s["visited"] == first
    s = _step(items, tile_w, waves, False, np.random.default_rng(6))
    assert s["visited"] == first and s["visited"] == s["rejected"] + s["written"]


@pytest.mark.parametrize("tile_w,waves", [(8, 8), (8, 4), (16, 8), (16, 2)])
@pytest.mark.parametrize("n", [500, 2047, 2048, 4300])
def test_frames_count_as_views(oracle_mod, report, n, tile_w, waves):
    rng = np.random.default_rng(n)
    kinds = _occluders(40, rng)
    items = [kinds[i] for i in rng.integers(0, len(kinds), n)]
    g, o = Rasterizer(W, H), oracle_mod.OracleRasterizer(W, H)
    g.set_config(tile_w, waves)
    g.frame_stats(True)
    for r in (g, o):
        r.clear()
        r.setModelViewProjection(MVP)
    assert np.array_equal(g.draw_frame(items), o.draw_frame(items))
    (dg, hg), (do, ho) = g.raw(), o.raw()
    assert np.array_equal(hg, ho), f"hiZ {report(hg, ho)}"
    assert np.array_equal(dg, do), f"depth {report(dg, do)}"
    s = g.frame_stats_read().astype(np.int64).sum(axis=0)
    v = _step(items, tile_w, waves, True)
    assert (s[13], s[14], s[15]) == (v["visited"], v["rejected"], v["written"])
