"""SAH batching on the device where ties decide the batches: centres on
coarse grids, so that most splits fall between equal centres and the order
left by earlier sorts matters, at sizes around the work-groups' and the
chunks' edges, against the restatement of the reference's recursion."""

from __future__ import annotations

import numpy as np
import pytest

from rasterizer_amd import Rasterizer, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [17, 33, 511, 513, 2049, 9001])
@pytest.mark.parametrize("cells", [(2, 3, 5), (1, 40, 1), (9, 1, 9), (30, 30, 30)])
@pytest.mark.parametrize("target,gran", [(17, 8), (64, 8), (512, 8), (9, 1), (40, 7)])
def test_tied_centres_match_reference(n, cells, target, gran):
    rng = np.random.default_rng(n * 7 + gran)
    c = np.stack([rng.integers(0, k, n) - k // 2 for k in cells], axis=1).astype(np.float32)
    h = rng.integers(1, 4, (n, 3)).astype(np.float32) * np.float32(0.25)
    mn, mx = c - h, c + h
    got = Rasterizer(64, 64).sah_batches_device(mn, mx, target, gran)
    want = scenes.sah_batches(mn, mx, target, gran)
    assert [b.tolist() for b in got] == [np.asarray(b).tolist() for b in want]
