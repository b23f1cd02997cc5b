"""Row reductions read by a whole row of outputs (softmax-like kernels): each
row is folded once; step and lane remainders, several shared ranges, against
float64 and (maxima) bit for bit."""
from __future__ import annotations

import numpy as np
import pytest


def softmax(x):
    """Row softmax without the max shift (inputs are small)."""
    e = x.exp()
    return e.mul(e.sum([1]).expand(list(x.shape)).reciprocal())


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(4096, 1000), (3, 64), (257, 65), (1000, 1001), (5, 40000), (70000, 68)])
def test_rows_of_outputs(fg, hip, shape):
    r = np.random.default_rng(shape[1])
    a = r.standard_normal(shape).astype(np.float32)
    z = fg.Tensor.new(a, list(shape), hip).with_requires_grad(True)
    t = r.dirichlet(np.ones(8), shape[0]).astype(np.float32) @ np.eye(8, shape[1], dtype=np.float32)
    loss = z.cross_entropy(fg.Tensor.new(t, list(shape), hip))
    (g,) = loss.gradient([z])
    fg.Tensor.realize_many([g, loss])
    a64, t64 = a.astype(np.float64), t.astype(np.float64)
    e = np.exp(a64 - a64.max(1, keepdims=True))
    p = e / e.sum(1, keepdims=True)
    want = (p * t64.sum(1, keepdims=True) - t64) / shape[0]
    # About ten roundings and two row sums of at most 160 steps: 1e-5 of the
    # terms. The gradient of the max shift adds the row's sum of p - t, which
    # cancels, at the row's maximum: its terms sum to 2 in magnitude.
    terms = p + t64 + 2.0 * (a64 == a64.max(1, keepdims=True))
    assert np.max(np.abs(g.numpy() - want) / (terms / shape[0])) <= 1e-5
    x = fg.Tensor.new(a, list(shape), hip)
    m = x.sub(x.max([1]).expand(list(shape)))
    assert np.array_equal(m.numpy(), a - a.max(1, keepdims=True))
    s = softmax(fg.Tensor.new(a, list(shape), hip)).numpy()
    assert np.max(np.abs(s - p) / p) <= 1e-5


@pytest.mark.gpu
def test_rows_shared_by_two_ranges(fg, hip):
    a = np.random.default_rng(5).standard_normal((6, 7, 100)).astype(np.float32)
    b = np.random.default_rng(6).standard_normal((6, 9, 12)).astype(np.float32)
    rows = fg.Tensor.new(a, [6, 7, 100], hip).max([1, 2])
    got = fg.Tensor.new(b, [6, 9, 12], hip).mul(rows.expand([6, 9, 12])).numpy()
    assert np.array_equal(got, b * a.max((1, 2), keepdims=True))


def test_softmax_gradient_folds_each_row_once(fg, cpu):
    z = fg.Tensor.new(np.zeros((512, 1000), np.float32), [512, 1000], cpu).with_requires_grad(True)
    (g,) = z.cross_entropy(fg.Tensor.new(np.zeros((512, 1000), np.float32), [512, 1000], cpu)).gradient([z])
    items = fg.debug_plan([g], fuse=True, render_hip=True)["items"]
    last = items[-1]
    assert last["class"] == "row_reduce" and last["out_shape"] == [512, 1000]
    assert last["grid"][0] == 512 // 4 and "for (int b = rlane;" in last["source"]


# Output shape, the reduced operand's shape (its last axis is summed) and the
# shape that the sums take beside the output: one group, few groups, groups
# broadcast over the rows (their outputs lie apart) and over outer and inner
# axes, short and long folds, ragged outputs and cuts.
BROADCASTS = [([4096, 4096], (1, 256), [1, 1]), ([1025, 4099], (1, 64), [1, 1]), ([4096, 1024], (1, 4096), [1, 1]),
              ([16, 4096], (16, 64), [16, 1]), ([9, 30001], (9, 100), [9, 1]), ([262144, 16], (16, 64), [1, 16]),
              ([20001, 16], (16, 300), [1, 16]), ([4096, 4096], (4096, 130), [1, 4096]), ([4096, 64, 4], (64, 128), [1, 64, 1]),
              ([33, 64, 1000], (64, 128), [1, 64, 1]), ([8, 131072], (8, 4000), [8, 1])]


def broadcast(fg, dev, out, terms, shape):
    r = np.random.default_rng(len(out) + terms[1])
    x, s = r.standard_normal(out).astype(np.float32), r.uniform(0.5, 1.5, terms).astype(np.float32)
    t = fg.Tensor.new(s, list(terms), dev).sum([1]).reshape([terms[0]]).reshape(shape).expand(out)
    return fg.Tensor.new(x, out, dev).mul(t), x * s.astype(np.float64).sum(1).reshape(shape)


@pytest.mark.gpu
@pytest.mark.parametrize("out,terms,shape", BROADCASTS)
def test_broadcast_sums(fg, hip, out, terms, shape):
    got, want = broadcast(fg, hip, out, terms, shape)
    # Positive terms, at most 4096 / 256 steps of a thread and a tree of 8 levels, and the product.
    assert np.max(np.abs(got.numpy() - want) / np.abs(want)) <= 4e-6


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(8, 131072), (3, 200003), (255, 65536), (1, 300000)])
def test_few_long_rows(fg, hip, shape):
    a = np.random.default_rng(shape[0]).standard_normal(shape).astype(np.float32)
    x = fg.Tensor.new(a, list(shape), hip)
    assert np.array_equal(x.sub(x.max([1]).expand(list(shape))).numpy(), a - a.max(1, keepdims=True))


def test_few_groups_fill_the_chip(fg, cpu):
    """Workgroups of kernels with few groups of outputs."""
    grid = {}
    for out, terms, shape in BROADCASTS:
        t, _ = broadcast(fg, cpu, out, terms, shape)
        (item,) = fg.debug_plan([t], fuse=True, render_hip=True)["items"]
        assert item["class"] == "row_reduce"
        grid[tuple(out), terms] = item["grid"][0], "for (int b = " in item["source"]
    assert grid[(4096, 4096), (1, 256)] == (1024, True)
    assert grid[(4096, 1024), (1, 4096)] == (1024, True)
    assert grid[(4096, 64, 4), (64, 128)] == (512, True)  # cuts of 2048 outputs
    assert grid[(8, 131072), (8, 4000)] == (8 * 64, True)
    # Sums of 64 broadcast over the rows are folded for each output.
    assert grid[(262144, 16), (16, 64)] == (65536, False)
    assert grid[(4096, 4096), (4096, 130)] == (4096, True)
