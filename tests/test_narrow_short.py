"""Products with one side of at most 16 and a short K (the one-pass small GEMM
instead of the streaming rows kernel), against float64."""
from __future__ import annotations

import numpy as np
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("w,n,k", [(256, 1, 1028), (256, 10, 508), (300, 7, 64), (2001, 16, 508), (70000, 9, 256), (4099, 3, 72)])
def test_short_narrow_products(fg, hip, w, n, k):
    r = np.random.default_rng(w + n + k)
    x, wt = r.standard_normal((w, k)).astype(np.float32), r.standard_normal((n, k)).astype(np.float32)
    b = r.standard_normal(n).astype(np.float32)
    a = fg.Tensor.new(x, [w, k], hip)
    m, c = fg.Tensor.new(wt, [n, k], hip), fg.Tensor.new(b, [n], hip)
    got = a.relu().matmul(m.permute([1, 0])).add(c.reshape([1, n]).expand([w, n])).numpy()
    x64 = np.maximum(x, 0).astype(np.float64)
    scale = x64 @ np.abs(wt.T).astype(np.float64) + np.abs(b)
    # At most 16 waves of four 16-k groups, each term rounded about 40 times: 40 * 2^-24.
    assert np.max(np.abs(got - (x64 @ wt.T.astype(np.float64) + b)) / scale) <= 2.5e-6
