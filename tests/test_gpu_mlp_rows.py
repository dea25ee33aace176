"""Gradients at the sample counts where the backward pass's partial sums
change: one work-group's 128 samples and one more, every work-group (32,768)
and one more (a second round), against the CPU oracle; repeated calls on one
model of changing size return the same bytes as the first of that size."""

from __future__ import annotations

import numpy as np
import pytest

from oracle import mlp as ref
from rasterizer_amd import Mlp

pytestmark = pytest.mark.gpu


def _case(n):
    rng = np.random.default_rng(n)
    x = rng.normal(size=(n, 16)).astype(np.float32) * 2 + 0.5
    i = rng.integers(0, n, n // 2 + 1)
    return x, np.stack([i, (i + 1 + rng.integers(0, n - 1, i.size)) % n], 1).astype(np.uint32)


@pytest.fixture(scope="module")
def model():
    rng = np.random.default_rng(8)
    m = Mlp(seed=3)
    w = rng.normal(scale=0.25, size=Mlp.N_PARAMS).astype(np.float32)
    norm = np.concatenate([np.full(16, 0.5), np.full(16, 0.5)]).astype(np.float32)
    m.set_params(w, norm)
    return m, w, norm


@pytest.mark.parametrize("n", [2, 127, 128, 129, 2049, 32768, 32769, 33000])
def test_gradients(model, n):
    m, w, norm = model
    x, pairs = _case(n)
    g, loss = m.gradients(x, pairs)
    lw, gw = ref.gradients(w, norm, x, pairs, bf16_ops=True)
    assert abs(loss - lw) <= 1e-4 * (1 + abs(lw))
    # The oracle rounds to bf16 where the kernels do; what remains is rounding
    # that falls the other way in single terms (2^-8 of a term).
    floor = 1e-3 * np.abs(gw).max()  # b3's gradient is a sum of +-pairs
    for name, a, b in (("W1", 0, 1024), ("b1", 1024, 1088), ("W2", 1088, 5184), ("b2", 5184, 5248),
                       ("W3", 5248, 5312), ("b3", 5312, 5313)):
        scale = max(np.abs(gw[a:b]).max(), floor)
        err = np.abs(g[a:b] - gw[a:b]).max() / scale
        assert err < 2e-2, f"{name}: max error {err:.3e} of the block's largest gradient"


def test_sizes_in_turn(model):
    m, _, _ = model
    one = np.array([[0, 1]], np.uint32)  # a single pair: no addition's order can differ
    first = {}
    for n in (300, 40000, 2, 300, 40000, 2, 129):
        g, loss = m.gradients(_case(n)[0], one)
        want = first.setdefault(n, (g, loss))
        assert np.array_equal(g, want[0]) and loss == want[1]
    g, loss = m.gradients(_case(300)[0], np.zeros((0, 2), np.uint32))
    assert loss == 0.0 and not g.any()
