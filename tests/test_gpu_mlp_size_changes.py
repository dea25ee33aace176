"""Gradients on one model in calls of changing size, from a large one down,
with pairs in every work-group's 128 samples: what a larger call left in the
kept rows of partial sums is in no later result.  Each sample is in one pair at
most, so each score's gradient is a single addition and the gradient is the same
bytes whichever model computes it."""

from __future__ import annotations

import numpy as np
import pytest

from rasterizer_amd import Mlp

pytestmark = pytest.mark.gpu


def _case(n):
    rng = np.random.default_rng(n)
    pairs = rng.permutation(n)[: n // 2 * 2].reshape(-1, 2)
    return rng.normal(size=(n, 16)).astype(np.float32), pairs.astype(np.uint32)


@pytest.mark.parametrize("sizes", [(40000, 300, 40000, 2), (32768, 127, 129, 33000, 128), (2048, 2, 2049)])
def test_sizes_down_and_up(sizes):
    rng = np.random.default_rng(8)
    w = rng.normal(scale=0.25, size=Mlp.N_PARAMS).astype(np.float32)
    kept = Mlp(seed=3)
    kept.set_params(w)
    for n in sizes:
        x, pairs = _case(n)
        fresh = Mlp(seed=3)
        fresh.set_params(w)
        want, loss = fresh.gradients(x, pairs)
        # Every row counts: with one work-group's pairs left out the gradient is
        # another one.
        if n > 256:
            rest, _ = fresh.gradients(x, pairs[(pairs >= 128).all(axis=1)])
            assert not np.array_equal(rest, want)
        g, l = kept.gradients(x, pairs)
        assert np.array_equal(g, want), f"{n} samples"
        # The pairs' losses are added by one atomic a wave, n / 128 of them in any
        # order: each rounds by 2^-24 of the sum at most, in both results.
        assert abs(l - loss) <= 2.0 * (n / 128 + 8) * 2.0**-24 * abs(loss)
    g, l = kept.gradients(_case(300)[0], np.zeros((0, 2), np.uint32))
    assert l == 0.0 and not g.any()
