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


# Batches of small transposes: both sides short, one short side, sides at the
# least tile, odd ones.
BATCHES = [(70000, 2, 2), (30001, 3, 3), (5000, 8, 8), (2000, 16, 16), (1500, 24, 16), (1300, 31, 17), (700, 20, 20), (900, 10, 40),
           (900, 40, 10), (1100, 4, 64), (600, 2, 300), (300, 700, 2), (70, 65, 67)]


def ints(fg, dev, shape):
    a = np.random.default_rng(sum(shape)).integers(-1000, 1000, shape).astype(np.float32)
    return fg.Tensor.new(a, list(shape), dev), a


@pytest.mark.gpu
@pytest.mark.parametrize("shape", BATCHES)
def test_batches_of_small_transposes(fg, hip, shape):
    x, a = ints(fg, hip, shape)
    want = a.transpose(0, 2, 1)
    p = x.permute([0, 2, 1])
    assert np.array_equal(p.contiguous().numpy(), want)
    y, b = ints(fg, hip, want.shape)
    assert np.array_equal(p.mul(p).add(y).numpy(), want * want + b)


@pytest.mark.parametrize("shape", [(262144, 2, 2), (100000, 3, 3), (65536, 8, 8), (65536, 16, 16), (16384, 32, 32), (30000, 31, 17),
                                   (20000, 10, 40), (8192, 100, 2), (2000, 1000, 2), (700, 65, 65), (9, 300, 300)])
def test_tiles_stay_near_their_outputs(fg, cpu, shape):
    """Tiles only from 384 elements on, and staging (whole steps of 256) no
    more than four times the outputs: a tile ends where its sides end."""
    n, r, c = shape
    x = fg.Tensor.zeros(list(shape), cpu).add(fg.Tensor.scalar(1.0, cpu)).realize()
    (item,) = fg.debug_plan([x.permute([0, 2, 1]).contiguous()], fuse=True, render_hip=True)["items"]
    assert item["class"] == "elementwise"
    assert ("__shared__" in item["source"]) == (r * c >= 384)
    if r * c >= 384:
        steps = int(item["source"].split("in0[")[1].split("]")[0])
        assert item["grid"][0] * steps * 256 <= 4 * n * r * c
