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


# Programs whose second kernel reads the first one's output both in its own row
# and in every row (or the first one reads so what the second one writes): the
# result of (fg, device, a [n, k], m [n, n]) and the float64 value.
def outer_sum(fg, dev, a, m):
    n = len(a)
    d = fg.Tensor.new(a, list(a.shape), dev)
    d = d.mul(d).sum([1])
    d64 = (a.astype(np.float64) ** 2).sum(1, keepdims=True)
    return d.expand([n, n]).add(d.permute([1, 0]).expand([n, n])), d64 + d64.T


def normalised_adjacency(fg, dev, a, m):
    n = len(a)
    t = fg.Tensor.new(m, [n, n], dev)
    d = t.sum([1]).reciprocal()
    d64 = 1.0 / m.astype(np.float64).sum(1, keepdims=True)
    return t.mul(d.expand([n, n])).mul(d.permute([1, 0]).expand([n, n])), m * d64 * d64.T


def first_row_added(fg, dev, a, m):
    x = fg.Tensor.new(m, list(m.shape), dev)
    e = x.exp().contiguous()
    e64 = np.exp(m.astype(np.float64))
    return e.add(e.narrow(0, 0, 1).expand(list(m.shape))), e64 + e64[:1]


MIXED = {f.__name__: f for f in (outer_sum, normalised_adjacency, first_row_added)}


def mixed_inputs(n):
    r = np.random.default_rng(n)
    return r.uniform(0.5, 1.5, (n, 300)).astype(np.float32), r.uniform(0.5, 1.5, (n, n)).astype(np.float32)


def together(plan):
    """The pairs of plan items that share a row batch."""
    runs = [range(b["first"], b["first"] + b["count"]) for b in plan["row_batches"]]
    return {(i, j) for r in runs for i in r for j in r if i < j}


@pytest.mark.parametrize("name", MIXED)
def test_reads_by_row_and_of_every_row_stay_apart(fg, cpu, name):
    """A buffer read in the kernel's own row and without the row is not by row."""
    out, _ = MIXED[name](fg, cpu, *mixed_inputs(1024))
    plan = fg.debug_plan([out], fuse=True, render_hip=True)
    assert len(plan["items"]) == 2 and together(plan) == set(), plan["row_batches"]


def test_every_row_read_before_an_update_stays_apart(fg, cpu):
    """y reads w[r] and all of w; the update of w in the same schedule is by row."""
    n = 1024
    w = fg.Tensor.new(np.ones((n, 1), np.float32), [n, 1], cpu)
    y = w.expand([n, n]).add(w.permute([1, 0]).expand([n, n]))
    w.assign(fg.Tensor.new(np.ones((n, 300), np.float32), [n, 300], cpu).sum([1]))
    plan = fg.debug_plan([y, w], fuse=True, render_hip=True)
    assert len(plan["items"]) == 2 and together(plan) == set(), plan["row_batches"]


@pytest.mark.gpu
@pytest.mark.parametrize("name", MIXED)
@pytest.mark.parametrize("n", [1024, 2050])
def test_replays_of_mixed_reads(fg, hip, name, n):
    fg.clear_caches()
    a, m = mixed_inputs(n)
    first = None
    for _ in range(4):
        out, want = MIXED[name](fg, hip, a, m)
        got = out.numpy()
        # At most 300 or n positive terms, 2^-24 each, and a few roundings.
        assert np.max(np.abs(got - want) / want) <= 2e-4
        assert first is None or np.array_equal(got, first)
        first = got.copy()


def column_sums_added(fg, dev, a, m):
    """A reduction broadcast over the rows of square outputs: its kernel reads
    what the first one writes."""
    n = len(a)
    e = fg.Tensor.new(m, [n, n], dev).exp()
    s = fg.Tensor.new(a, list(a.shape), dev).sum([1])
    out = e.add(s.permute([1, 0]).expand([n, n]))
    e64 = np.exp(m.astype(np.float64))
    return [e, out], [e64, e64 + a.astype(np.float64).sum(1)[None, :]]


def exp_of_column_sums(fg, dev, a, m):
    """The same kernel as the writer of what the second one reads by row."""
    n = len(a)
    s = fg.Tensor.new(a, list(a.shape), dev).mul(fg.Tensor.scalar(0.01, dev)).sum([1])
    o = fg.Tensor.new(m, [n, n], dev).add(s.permute([1, 0]).expand([n, n]))
    o64 = m + (a.astype(np.float64) * float(np.float32(0.01))).sum(1)[None, :]
    return [o, o.exp()], [o64, np.exp(o64)]


BROADCAST = {f.__name__: f for f in (column_sums_added, exp_of_column_sums)}


@pytest.mark.parametrize("name", BROADCAST)
def test_reductions_broadcast_over_the_rows_stay_apart(fg, cpu, name):
    roots, _ = BROADCAST[name](fg, cpu, *mixed_inputs(1024))
    plan = fg.debug_plan(roots, fuse=True, render_hip=True)
    reduces = [i for i, it in enumerate(plan["items"]) if it["class"] == "row_reduce"]
    assert len(plan["items"]) == 2 and len(reduces) == 1 and together(plan) == set(), plan["row_batches"]


@pytest.mark.gpu
@pytest.mark.parametrize("name", BROADCAST)
@pytest.mark.parametrize("n", [1024, 2050])
def test_replays_of_reductions_broadcast_over_the_rows(fg, hip, name, n):
    fg.clear_caches()
    a, m = mixed_inputs(n)
    first = None
    for _ in range(4):
        roots, want = BROADCAST[name](fg, hip, a, m)
        fg.Tensor.realize_many(roots)
        got = [t.numpy() for t in roots]
        for g, w in zip(got, want):
            # Sums of 300 positive terms (of about 3 before exp), 2^-24 each.
            assert np.max(np.abs(g - w) / w) <= 1e-4
        assert first is None or all(np.array_equal(x, y) for x, y in zip(got, first))
        first = [g.copy() for g in got]


def test_long_rows_batch_while_they_stay_in_the_caches(fg, cpu):
    def runs(rows, cols):
        x = fg.Tensor.zeros([rows, cols], cpu).add(fg.Tensor.scalar(1.0, cpu)).realize()
        e = x.exp()
        plan = fg.debug_plan([e, e.mul(x)], fuse=True, render_hip=True)
        assert len(plan["items"]) == 2
        return [(b["first"], b["count"]) for b in plan["row_batches"]]

    # Three buffers of rows x cols: up to 8192 columns, or 256 MiB in all.
    assert runs(4096, 8192) == [(0, 2)] and runs(600, 32768) == [(0, 2)]
    assert runs(1024, 32768) == [] and runs(512, 131072) == [] and runs(4096, 8196) == []
