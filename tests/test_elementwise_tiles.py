"""Elementwise kernels over a transposed operand (LDS tiles): tile edges, short
sides, several operands and types, bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

SHAPES = [(4000, 131), (9, 30001), (64, 4097), (513, 2044), (1025, 1023), (33000, 31), (2, 140001), (140001, 2),
          (65, 4100)]


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES)
def test_transposed_operands(fg, hip, shape):
    r, c = shape
    rng = np.random.default_rng(r + c)
    a, b = rng.standard_normal((r, c)).astype(np.float32), rng.standard_normal((c, r)).astype(np.float32)
    ta, tb = fg.Tensor.new(a, [r, c], hip), fg.Tensor.new(b, [c, r], hip)
    bits = lambda t, w: np.array_equal(t.numpy().reshape(w.shape), w)  # noqa: E731
    assert bits(ta.permute([1, 0]).contiguous(), a.T)
    assert bits(ta.permute([1, 0]).add(tb), a.T + b)
    assert bits(ta.narrow(0, 1, r - 1).permute([1, 0]).contiguous(), a[1:].T)
    p = ta.permute([1, 0])
    assert bits(p.mul(p).add(tb).relu(), np.maximum(a.T * a.T + b, np.float32(0)))
    i = (a * 1000).astype(np.int32)
    assert bits(fg.Tensor.new(i, [r, c], hip).permute([1, 0]).contiguous(), i.T)
    assert bits(fg.Tensor.new(a > 0, [r, c], hip).permute([1, 0]).contiguous(), (a > 0).T)


@pytest.mark.gpu
@pytest.mark.parametrize("order", [(2, 1, 0), (1, 0, 2), (0, 2, 1), (2, 0, 1), (1, 2, 0)])
def test_permuted_copies_of_three_axes(fg, hip, order):
    a = np.random.default_rng(3).standard_normal((7, 130, 501)).astype(np.float32)
    got = fg.Tensor.new(a, list(a.shape), hip).permute(list(order)).contiguous().numpy()
    assert np.array_equal(got, np.transpose(a, order))
