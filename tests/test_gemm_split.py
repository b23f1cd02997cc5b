"""The tiled GEMM's bfloat16 split on HIP: operands of any f32 magnitude,
infinities, NaN, sums past the split's scaled range, and accuracy against the
rounding of f32 sums, in every orientation of a Linear's products."""
from __future__ import annotations

import numpy as np
import pytest

from test_gemm_tiles import products

# (B, in, out): ragged rows and columns; k a multiple of 16, of 4 and of neither.
SHAPES = [(520, 608, 300), (600, 620, 301), (515, 601, 333)]


def data(shape, seed):
    B, fi, fo = shape
    r = np.random.default_rng(seed)
    return (r.standard_normal((B, fi)).astype(np.float32), r.standard_normal((fo, fi)).astype(np.float32),
            r.standard_normal((B, fo)).astype(np.float32))


def run(fg, dev, x, w, g):
    p = products(fg, dev, x, w, g)
    fg.Tensor.realize_many(list(p.values()))
    with np.errstate(all="ignore"):
        x, w, g = (a.astype(np.float64) for a in (x, w, g))
        ax, aw, ag = np.abs(x), np.abs(w), np.abs(g)
        want = {"fwd": (x @ w.T, ax @ aw.T), "dx": (g @ w, ag @ aw), "dw": (g.T @ x, ag.T @ ax)}
    return {k: (t.numpy().astype(np.float64).reshape(want[k][0].shape), *want[k]) for k, t in p.items()}


def test_products_a_comparison_reads_keep_the_f32_mfma(fg, cpu):
    """A train step's hidden layers feed relu masks; their input and weight
    gradients, and a product nothing compares, are split."""
    t = lambda *s: fg.Tensor.new(np.ones(s, np.float32), list(s), cpu)  # noqa: E731
    w1, w2 = t(700, 600).with_requires_grad(True), t(650, 700).with_requires_grad(True)
    x = t(640, 600)
    z1 = x.matmul(w1.permute([1, 0]))
    z2 = z1.relu().matmul(w2.permute([1, 0]))
    grads = z2.mul(t(640, 650)).sum([0, 1]).gradient([w1, w2])
    items = fg.debug_plan([z2, *grads], fuse=True, render_hip=True)["items"]
    kinds = [("32x32x16_bf16" in i["source"], i["out_shape"]) for i in items if i["class"] == "gemm_mfma_f32"]
    assert kinds[0] == (False, [640, 700, 1]), kinds  # z1, under relu
    assert len(kinds) == 5 and all(split for split, _ in kinds[1:]), kinds


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES)
def test_split_is_as_accurate_as_f32_sums(fg, hip, shape):
    for name, (got, want, _) in run(fg, hip, *data(shape, 1)).items():
        # 620 terms summed one by one in f32 measure about 4.4e-7 here.
        assert np.linalg.norm(got - want) / np.linalg.norm(want) <= 5e-7, name


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES)
def test_operands_of_any_magnitude(fg, hip, shape):
    x, w, g = data(shape, 2)
    scale = np.float32(2.0) ** np.arange(-140, -140 + 4 * 64, 4, dtype=np.float32)  # subnormal to 2^112
    x = (x * scale[np.arange(len(x)) % 64, None]).astype(np.float32)
    w = (w * np.float32(2.0 ** 3)).astype(np.float32)
    g = (g * np.float32(2.0 ** -120)).astype(np.float32)
    for name, (got, want, terms) in run(fg, hip, x, w, g).items():
        # Each term's products are exact to about 2^-22 and below 2^-149 not at all.
        bound = 1e-5 * terms + 1024 * 2.0 ** -149
        assert np.all(np.abs(got - want) <= bound), name


def check_not_finite(fg, dev, shape, big=3.4e38):
    x, w, g = data(shape, 3)
    x[5, 7], x[9, 3], x[11, 2] = np.inf, np.nan, -np.inf
    w[2, 2], w[40, 40] = np.inf, big
    x[300:303] *= np.float32(1e33)  # finite sums of 1e34 and more
    g[4, 4], g[6, 100] = np.inf, big
    for name, (got, want, terms) in run(fg, dev, x, w, g).items():
        assert np.array_equal(np.isnan(got), np.isnan(want)), name
        over = ~np.isnan(want) & (np.abs(want) > 3.3e38)
        assert np.array_equal(got[over & np.isinf(want)], want[over & np.isinf(want)]), name
        fine = ~np.isnan(want) & ~over & (terms < 3.3e38)
        assert np.all(np.abs(got[fine] - want[fine]) <= 1e-5 * terms[fine]), name


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES)
def test_infinities_nan_and_overflow(fg, hip, shape):
    check_not_finite(fg, hip, shape)


# The largest finite value without products beyond f32: one of those beside an
# infinity of the other sign is NaN in f32, but not in float64.
BIG = 5e37


@pytest.mark.gpu
def test_infinities_nan_and_overflow_of_larger_products(fg, hip):
    check_not_finite(fg, hip, (2050, 1030, 1000), BIG)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES)
def test_zero_sums_are_positive(fg, hip, shape):
    """Zero rows and zero columns of operands (a dead unit, a padded batch)
    give +0 wherever they fall in a tile, as sums that start from +0 do."""
    x, w, g = data(shape, 4)
    x[::3], x[:, ::7], w[::5], g[1::4], g[:, 2::6] = 0.0, 0.0, 0.0, 0.0, 0.0
    for name, (got, want, terms) in run(fg, hip, x, w, g).items():
        assert np.any(terms == 0), name
        assert np.all(got[terms == 0] == 0) and not np.any(np.signbit(got[terms == 0])), name


# (B, in, out) whose forward product has K from 100 to 1030, where chains of
# f32 sums are short; errors of the f32 tiles' sums of the same products, of
# normal and of positive operands (2-norm, measured). From K 1024 on, where
# every 2nd stage is folded, sums of positive operands may be a tenth above
# (K 1030: 2.62e-7, the f32 tiles' 2.45e-7).
SHORT = [((1030, 100, 1010), 1.8e-7, 1.4e-7), ((1030, 256, 1010), 2.0e-7, 1.3e-7), ((1030, 320, 1010), 1.5e-7, 7.5e-8),
         ((1030, 512, 1010), 1.65e-7, 7.1e-8), ((4096, 784, 1024), 3.5e-7, 1.95e-7), ((4096, 1030, 1024), 4.0e-7, 2.7e-7)]


@pytest.mark.gpu
@pytest.mark.parametrize("shape,normal,positive", SHORT)
def test_short_products_are_as_accurate_as_f32_sums(fg, hip, shape, normal, positive):
    x, w, _ = data(shape, 5)
    for a, b, bound in ((x, w, normal), (np.abs(x), np.abs(w), positive)):
        t = fg.Tensor.new(a, list(a.shape), hip).matmul(fg.Tensor.new(b, list(b.shape), hip).permute([1, 0]))
        want = a.astype(np.float64) @ b.astype(np.float64).T
        got = t.numpy().reshape(want.shape)
        assert np.linalg.norm(got - want) / np.linalg.norm(want) <= bound


@pytest.mark.gpu
@pytest.mark.parametrize("shape,normal,positive", SHORT)
def test_cancelling_sums(fg, hip, shape, normal, positive):
    """Products whose second half of k cancels the first: an error within the
    rounding of the terms' own sums, for each element."""
    x, w, _ = data(shape, 6)
    h = shape[1] // 2
    x[:, h:2 * h] = -x[:, :h]
    w[:, h:2 * h] = w[:, :h] * (1.0 + 1e-3 * np.random.default_rng(7).standard_normal((len(w), h)).astype(np.float32))
    t = fg.Tensor.new(x, list(x.shape), hip).matmul(fg.Tensor.new(w, list(w.shape), hip).permute([1, 0]))
    x64, w64 = x.astype(np.float64), w.astype(np.float64)
    terms = np.abs(x64) @ np.abs(w64).T
    # The largest of the f32 tiles' sums is 2.7e-7 of the terms (K 128).
    assert np.max(np.abs(t.numpy().reshape(terms.shape) - x64 @ w64.T) / terms) <= 2.7e-7


# The same with the tile fixed, in a process of its own (FG_GEMM_TILE holds for
# every product): the largest tile, a 160-wide one as stream-K, two stages with
# K splits, splits that end inside a 16-k stage.
FORCED = """
import sys
sys.path.insert(0, sys.argv[1]); sys.path.insert(0, sys.argv[1] + "/tests")
import ferrograd_amd as fg
import test_gemm_split as t
t.check_not_finite(fg, "hip", (1000, 785, 601), t.BIG)
"""


@pytest.mark.gpu
@pytest.mark.parametrize("tile", ["256,256,32,4,2,1,3", "256,160,32,8,1,0,3", "128,256,32,2,2,2,2", "64,64,8,2,2,3,3"])
def test_infinities_nan_and_overflow_in_forced_tiles(tile):
    import os
    import subprocess
    import sys

    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", FORCED, root], env=dict(os.environ, FG_GEMM_TILE=tile), capture_output=True,
                       text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.gpu
def test_not_finite_products_take_a_few_times_as_long(fg, hip):
    """A NaN in every tile makes each workgroup compute its tile again on the
    f32 MFMA, a good half of the split's rate: 2.2 times as long in all, where
    loads of every element by itself took eleven."""
    import time

    n = 4096
    r = np.random.default_rng(8)
    x, w = (r.standard_normal((n, n)).astype(np.float32) for _ in range(2))
    bad = x.copy()
    bad[::16, ::16] = np.nan
    wt = fg.Tensor.new(w, [n, n], hip)
    us = []
    for a in (x, bad):
        t = fg.Tensor.new(a, [n, n], hip)
        runs = []
        for _ in range(5):
            fg.synchronize(hip)
            t0 = time.perf_counter()
            for _ in range(5):
                t.matmul(wt.permute([1, 0])).realize()
            fg.synchronize(hip)
            runs.append(time.perf_counter() - t0)
        us.append(min(runs))
    assert us[1] <= 4.0 * us[0], us
