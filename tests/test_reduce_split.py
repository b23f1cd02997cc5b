"""Row reductions over few outputs, split over workgroups: chunk and step
remainders, merged and unmerged reduce ranges, one chunk, against float64."""
from __future__ import annotations

import numpy as np
import pytest


# shape, axes, narrowed first (rows of a narrowed view keep their two ranges)
CASES = [((16384,), [0], False), ((65539,), [0], False), ((8200, 3), [0, 1], False), ((513, 127), [0, 1], False),
         ((3, 70001), [1], False), ((511, 17000), [1], False), ((7, 64, 1024), [1, 2], False),
         ((90, 2, 1000), [0, 2], False), ((100001, 5), [0, 1], True), ((40, 30), [0, 1], True)]


@pytest.mark.gpu
@pytest.mark.parametrize("shape,axes,narrowed", CASES)
def test_split_row_reductions(fg, hip, shape, axes, narrowed):
    a = np.random.default_rng(sum(shape)).standard_normal(shape).astype(np.float32)
    x = fg.Tensor.new(a, list(shape), hip)
    if narrowed:
        x, a = x.narrow(1, 1, shape[1] - 1), a[:, 1:]
    one = fg.Tensor.scalar(1.0, hip)
    got = x.mul(x).sum(axes).add(one).numpy()
    b = a.astype(np.float64) ** 2
    want = b.sum(tuple(axes), keepdims=True) + 1.0
    # A term is added at most 8200 / 256 + 8 + 8 + 12 times on its way to the
    # total (its thread's steps, the waves' trees, the chunks): 64 * 2^-24.
    assert np.max(np.abs(got - want) / want) <= 4e-6
    assert np.array_equal(x.max(axes).numpy(), a.max(tuple(axes), keepdims=True))
    i = (a * 100).astype(np.int32)
    got = fg.Tensor.new(i, list(i.shape), hip).sum(axes).numpy()
    assert np.array_equal(got, i.sum(tuple(axes), keepdims=True, dtype=np.int32))


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(60000, 17), (5000, 784), (3001, 66), (70000, 4), (9000, 1), (20, 3000, 18), (4097, 500)])
def test_split_column_reductions(fg, hip, shape):
    """Sums over the rows, split in chunks: ragged outputs of the second pass."""
    a = np.random.default_rng(len(shape) + shape[-1]).standard_normal(shape).astype(np.float32)
    axis = len(shape) - 2
    x = fg.Tensor.new(a, list(shape), hip)
    got = x.mul(x).sum([axis]).add(fg.Tensor.scalar(1.0, hip)).numpy()
    want = (a.astype(np.float64) ** 2).sum(axis, keepdims=True) + 1.0
    # At most 1100 rows of a thread's share and 40 more additions: 2^-24 each.
    assert np.max(np.abs(got - want) / want) <= 1e-5
    assert np.array_equal(x.max([axis]).numpy(), a.max(axis, keepdims=True))
    i = (a * 100).astype(np.int32)
    assert np.array_equal(fg.Tensor.new(i, list(shape), hip).sum([axis]).numpy(), i.sum(axis, keepdims=True, dtype=np.int32))


def test_split_row_reduction_launches(fg, cpu):
    """[5000, 3001] summed whole: one merged range, several chunks."""
    x = fg.Tensor.zeros([5000, 3001], cpu).add(fg.Tensor.scalar(1.0, cpu))
    k = fg.debug_plan([x.realize().sum([0, 1])], fuse=True, render_hip=True)["items"][0]
    assert k["class"] == "row_reduce" and "_part(" in k["source"] and 1024 < k["grid"][0] <= 2048
    # An empty reduction keeps its one pass and its identity.
    e = fg.Tensor.zeros([0, 3], cpu).sum([0, 1])
    assert "_part(" not in fg.debug_plan([e], fuse=True, render_hip=True)["items"][0]["source"]


@pytest.mark.parametrize("shape,split", [((1, 65536), False), ((1, 1 << 20), True), ((3, 70000), False), ((64, 1 << 18), True),
                                         ((300, 20001), False), ((100, 100001), True), ((500, 65536), False), ((256, 1 << 18), False),
                                         ((511, 40000), False)])
def test_rows_are_split_where_a_second_launch_pays(fg, cpu, shape, split):
    x = fg.Tensor.zeros(list(shape), cpu).add(fg.Tensor.scalar(1.0, cpu)).realize()
    (item,) = fg.debug_plan([x.mul(x).sum([1])], fuse=True, render_hip=True)["items"]
    assert item["class"] == "row_reduce" and ("_part(" in item["source"]) == split
