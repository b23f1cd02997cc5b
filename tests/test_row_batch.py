"""Row batches: consecutive kernels over the same rows in one launch on
replayed plans, bit for bit what the kernels compute on their own."""
from __future__ import annotations

import numpy as np
import pytest


def cross_entropy(fg, dev, shape, seed):
    r = np.random.default_rng(seed)
    z = fg.Tensor.new(r.standard_normal(shape).astype(np.float32), list(shape), dev).with_requires_grad(True)
    t = fg.Tensor.new(np.eye(shape[1], dtype=np.float32)[r.integers(0, shape[1], shape[0])], list(shape), dev)
    return z, t


def loss_and_grad(fg, z, t):
    loss = z.cross_entropy(t)
    (g,) = loss.gradient([z])
    fg.Tensor.realize_many([g, loss])
    return loss, g


# rows a multiple of the rows per workgroup and not; rows folded by a wave, by
# part of one, and across the waves of a workgroup; aligned and not.
@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(4096, 1000), (513, 1001), (8193, 33), (600, 5000), (1030, 4099), (512, 68)])
def test_replayed_batches_give_the_same_bits(fg, hip, shape):
    z, t = cross_entropy(fg, hip, shape, 1)
    fg.clear_caches()
    first = [x.numpy().copy() for x in loss_and_grad(fg, z, t)]  # kernel by kernel
    for _ in range(3):
        got = loss_and_grad(fg, z, t)
        assert all(np.array_equal(a.numpy(), b) for a, b in zip(got, first))
    z2, t2 = cross_entropy(fg, hip, shape, 2)  # other buffers, the same plan
    got = [x.numpy() for x in loss_and_grad(fg, z2, t2)]
    a64, t64 = z2.numpy().astype(np.float64), t2.numpy().astype(np.float64)
    e = np.exp(a64 - a64.max(1, keepdims=True))
    p = e / e.sum(1, keepdims=True)
    terms = p + t64 + 2.0 * (a64 == a64.max(1, keepdims=True))  # see test_row_outputs.py
    assert np.max(np.abs(got[1] - (p - t64) / shape[0]) / (terms / shape[0])) <= 1e-5


def test_row_batches_of_a_plan(fg, cpu):
    from hipcompile import compile_sources

    z, t = cross_entropy(fg, cpu, (2048, 300), 3)
    loss = z.cross_entropy(t)
    plan = fg.debug_plan([loss.gradient([z])[0], loss], fuse=True, render_hip=True)
    items = plan["items"]
    assert [(b["first"], b["count"]) for b in plan["row_batches"]] == [(0, len(items) - 1)]  # all but the loss's mean
    src = plan["row_batches"][0]["source"]
    for it in items[:-1]:
        assert f"{it['name']}_row" in src  # every stage under its own name
    assert "FGKERNELNAME" not in src
    compile_sources({src: plan["row_batches"][0]["name"]}, limit_s=120)


def test_kernels_that_read_other_rows_stay_apart(fg, cpu):
    # exp(x) is materialised; its row sums read it by row, its column
    # sums and its transpose read every row.
    x = fg.Tensor.new(np.zeros((700, 700), np.float32), [700, 700], cpu)
    y = x.exp()
    rows, cols, both = y.sum([1]), y.sum([0]), y.add(y.permute([1, 0]))
    plan = fg.debug_plan([y, rows, cols, both], fuse=True, render_hip=True)
    runs = [(b["first"], b["count"]) for b in plan["row_batches"]]
    names = [it["out_shape"] for it in plan["items"]]
    assert all(names[i] != [1, 700] and i != len(names) - 1 for f, c in runs for i in range(f, f + c)), (runs, names)
    # Fewer rows than CUs: no batch.
    z, t = cross_entropy(fg, cpu, (500, 300), 4)
    loss = z.cross_entropy(t)
    assert fg.debug_plan([loss.gradient([z])[0]], fuse=True, render_hip=True)["row_batches"] == []
