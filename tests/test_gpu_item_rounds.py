"""The tiles' walk over their items at the edges of its rounds, against the
oracle bit for bit: as many small occluders in one tile as a block of 64 item
slots holds, one more, as many as a window holds, one more, and more
candidates than one window tests; among them one with more 64-quad groups than
an item's group mask has bits.  Query-gated (front to back and back to front)
and without gating, in every tile size and wave count."""

from __future__ import annotations

import math

import numpy as np
import pytest

from rasterizer_amd import Occluder, Rasterizer, Views, scenes

pytestmark = pytest.mark.gpu

W = H = 120


def _occluders(n, rng):
    """n boxes in front of the eye and all around it, a dense one among them."""
    c = np.stack([rng.uniform(-9, 9, n), rng.uniform(-9, 9, n), rng.uniform(40, 90, n)], axis=1)
    c[n // 2::7, 2] *= -1.0  # some are behind the eye
    h = np.exp(rng.uniform(math.log(0.05), math.log(2.5), (n, 3)))
    out = []
    for i in range(n):
        if i == n // 3:
            k = 27  # 6 * 27 * 27 = 4,374 quads: 69 groups
            g = np.linspace(-1.0, 1.0, k + 1)
            parts = [scenes.box_quads(c[i] + h[i] * np.array([(g[a] + g[a + 1]) / 2, (g[b] + g[b + 1]) / 2, 0.0]),
                                      h[i] * np.array([1.0 / k, 1.0 / k, 1.0])) for a in range(k) for b in range(k)]
            q = np.concatenate(parts)
        else:
            q = scenes.box_quads(c[i], h[i])
        v = scenes.pad_to_batches(q).reshape(-1, 4)
        out.append(Occluder.bake(v, v.min(axis=0), v.max(axis=0)))
    order = np.argsort(np.linalg.norm(c, axis=1))
    return [out[i] for i in order]


@pytest.mark.parametrize("tile_w,waves", [(8, 2), (8, 4), (8, 8), (16, 2), (16, 8)])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 128, 129, 530])
def test_rounds_match_oracle(oracle_mod, report, n, tile_w, waves):
    occ = _occluders(n, np.random.default_rng(n))
    mvp = scenes.view_projection((0.0, 0.0, 0.0), np.array([0.0, 0.0, 1.0]), (0, 1, 0), math.pi / 8, W / H)
    for items in (occ, occ[::-1]):
        g, o = Rasterizer(W, H), oracle_mod.OracleRasterizer(W, H)
        g.set_config(tile_w, waves)
        for r in (g, o):
            r.clear()
            r.setModelViewProjection(mvp)
        st_g, st_o = g.draw_frame(items), o.draw_frame(items)
        assert np.array_equal(st_g, st_o), f"statuses differ at {np.flatnonzero(st_g != st_o)[:10]}"
        (dg, hg), (do, ho) = g.raw(), o.raw()
        assert np.array_equal(hg, ho), f"hiZ {report(hg, ho)}"
        assert np.array_equal(dg, do), f"depth {report(dg, do)}"
    V = Views(g, [(W, H)] * 2)
    V.set_config(waves, 0, tile_w)
    V.set_query_gated(False)
    for k in range(2):
        V.set_occluders(k, items)
        V.set_mvp(k, mvp)
    V.run()
    V.sync()
    got = V.raw(1)
    v = oracle_mod.OracleRasterizer(W, H)
    v.clear()
    v.setModelViewProjection(mvp)
    v.draw_frame(items, gated=False)
    want = v.raw()
    assert np.array_equal(got[1], want[1]) and np.array_equal(got[0], want[0])


@pytest.mark.parametrize("tile_w", [8, 16])
@pytest.mark.parametrize("low", [0, 1, 2, 3, 40000])
def test_quads_behind_what_is_there(oracle_mod, report, low, tile_w):
    """Small quads over a buffer whose blocks' smallest depth is 0, 1 (which
    reads as cleared), 2, 3 or nearer than most of them, drawn after others: the
    tests that leave out quads that every block rejects."""
    rng = np.random.default_rng(low)
    occ = _occluders(300, rng)
    mvp = scenes.view_projection((0.0, 0.0, 0.0), np.array([0.0, 0.0, 1.0]), (0, 1, 0), math.pi / 8, W / H)
    depth = rng.integers(low, 50000, (W // 8 * (H // 8), 64)).astype(np.uint16)
    depth[:, 0] = low
    hiz = np.concatenate([depth.min(axis=1), np.zeros(8, np.uint16)]).astype(np.uint16)
    g, o = Rasterizer(W, H), oracle_mod.OracleRasterizer(W, H)
    g.set_config(tile_w, 8)
    g.upload_raw(depth, hiz)
    o.set_raw(depth, hiz)
    for r in (g, o):
        r.setModelViewProjection(mvp)
    assert np.array_equal(g.draw_frame(occ), o.draw_frame(occ))
    (dg, hg), (do, ho) = g.raw(), o.raw()
    assert np.array_equal(hg, ho), f"hiZ {report(hg, ho)}"
    assert np.array_equal(dg, do), f"depth {report(dg, do)}"


@pytest.mark.parametrize("tile_w,waves", [(8, 8), (16, 8), (16, 2)])
@pytest.mark.parametrize("n", [2047, 2048, 2049, 4300])
def test_many_items(oracle_mod, report, n, tile_w, waves):
    """Around the number of items from which a tile tests their boxes, four a
    thread, with most of them outside any one tile."""
    rng = np.random.default_rng(n)
    kinds = _occluders(40, rng)
    occ = [kinds[i] for i in rng.integers(0, len(kinds), n)]
    occ[::50] = occ[: len(occ[::50])]
    mvp = scenes.view_projection((0.0, 0.0, 0.0), np.array([0.0, 0.0, 1.0]), (0, 1, 0), math.pi / 8, 4 * W / H)
    g, o = Rasterizer(4 * W, H), oracle_mod.OracleRasterizer(4 * W, H)
    g.set_config(tile_w, waves)
    for r in (g, o):
        r.clear()
        r.setModelViewProjection(mvp)
    assert np.array_equal(g.draw_frame(occ), o.draw_frame(occ))
    (dg, hg), (do, ho) = g.raw(), o.raw()
    assert np.array_equal(hg, ho), f"hiZ {report(hg, ho)}"
    assert np.array_equal(dg, do), f"depth {report(dg, do)}"
