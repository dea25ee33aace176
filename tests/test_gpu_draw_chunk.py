"""The tiles' draw of a staged chunk at the edges of its tables, against the
oracle bit for bit: chunks whose quads need more fold-table rows than one
pass holds, more than 64 (block, quad) pairs in one block, single-block
quads, and quads that reach far outside the tile, in every tile size and
wave count."""

from __future__ import annotations

import math

import numpy as np
import pytest

from rasterizer_amd import Occluder, Rasterizer, scenes

pytestmark = pytest.mark.gpu

W, H = 328, 200


def _boxes(kind, rng):
    if kind == "rows":        # every quad spans whole tiles: 64 quads need all rows
        n, spread, lo, hi = 96, 6.0, 4.0, 30.0
    elif kind == "one block":  # a cluster about 8 px across: hundreds of pairs in a block
        n, spread, lo, hi = 400, 0.15, 0.02, 0.3
    elif kind == "small":     # a block or two each, all over the buffer
        n, spread, lo, hi = 700, 12.0, 0.05, 0.3
    else:                     # from single pixels to most of the buffer
        n, spread, lo, hi = 300, 10.0, 0.02, 20.0
    c = rng.uniform(-spread, spread, (n, 3))
    c[:, 2] = 60.0 + rng.uniform(-20.0, 20.0, n)
    h = np.exp(rng.uniform(math.log(lo), math.log(hi), (n, 3)))
    h[:, 2] = np.minimum(h[:, 2], 5.0)
    return np.concatenate([scenes.box_quads(c[i], h[i]) for i in range(n)])


@pytest.mark.parametrize("tile_w,waves", [(t, n) for t in (8, 16) for n in (2, 4, 8)])
@pytest.mark.parametrize("kind", ["rows", "one block", "small", "mixed"])
def test_chunks_match_oracle(oracle_mod, report, kind, tile_w, waves):
    rng = np.random.default_rng(17)
    quads = scenes.pad_to_batches(rng.permutation(_boxes(kind, rng)))
    v = quads.reshape(-1, 4)
    occ = [Occluder.bake(v[k:k + 4 * 512], v.min(axis=0), v.max(axis=0)) for k in range(0, v.shape[0], 4 * 512)]
    eye, d = (0.0, 0.0, 0.0), np.array([0.02, -0.03, 1.0])
    mvp = scenes.view_projection(eye, d / np.linalg.norm(d), (0, 1, 0), math.pi / 6, W / H)
    g, o = Rasterizer(W, H), oracle_mod.OracleRasterizer(W, H)
    g.set_config(tile_w, waves)
    for r in (g, o):
        r.clear()
        r.setModelViewProjection(mvp)
        for k in occ:
            r.rasterize(k, False)
    (dg, hg), (do, ho) = g.raw(), o.raw()
    assert np.count_nonzero(do) > 1000 or kind == "one block"
    assert np.array_equal(hg, ho), f"{kind}: hiZ {report(hg, ho)}"
    assert np.array_equal(dg, do), f"{kind}: depth {report(dg, do)}"
