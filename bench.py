#!/usr/bin/env python3
"""Benchmark of ferrograd's realize path on one MI355X (configs C1-C5).

Primary line (the `value`): C2, the pure elementwise bandwidth config
`(a*b + c).relu()` over 2^26 f32 elements, as HBM GB/s of algorithmic traffic
(3 reads + 1 write). A step is one realise of that lazy graph (schedule,
lowering-cache lookup, launch) with the inputs resident in HBM.

Also measured and reported under "secondary": C1 (fused elementwise + row
reduction, GB/s), C3 (Linear forward x@W^T+b, MFMA fp32 TFLOP/s), C4 and C5
(MLP train steps/s plus the GEMM kernels' share of the fp32 MFMA peak; products
split for the bfloat16 matrix cores can pass it).

Kernel durations come from HIP events recorded around every launch on the
device's own stream during the timed region (fg_hip_profile_*). The CPU
baseline is the oracle's restated reference clang backend on one pinned core.

Usage: python bench.py [--gpus 1] [--steps K] [--warmup W] [--only c2] [--no-cpu]
"""
from __future__ import annotations

import argparse
import json
import os
import subprocess
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "fused-kernel HBM GB/s & MFMA fp32 TFLOP/s; MLP train steps/s (1 GPU)"
HBM_PEAK_GBS = 8000.0           # MI355X HBM3E
FP32_MFMA_PEAK_TFLOPS = 157.3   # MI355X dense fp32 matrix
# An f32 product split into six bfloat16 products (C3's GEMM): a sixth of the dense bfloat16 matrix peak.
SPLIT_MFMA_PEAK_TFLOPS = 2500.0 / 6


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def timed(fg, ctx, step, steps: int, warmup: int):
    """Run `step` warmup times untimed, then time `steps` steps between two
    device synchronisations (the step rate), then run `steps` more with
    dispatch-attached events on every launch (the per-kernel durations; the
    events add host work, so they are kept out of the step-rate region).
    Returns (ms/step, profile)."""
    for _ in range(warmup):
        step()
    fg.synchronize()
    h0 = fg.stats()["host_ms"]
    t0 = time.perf_counter()
    for _ in range(steps):
        step()
    fg.synchronize()
    t1 = time.perf_counter()
    h1 = fg.stats()["host_ms"]
    timed.host_ms = {k: (h1[k] - h0[k]) / steps for k in h1}  # host pipeline phases per timed step
    ctx.profile_read()  # drop anything recorded before
    ctx.profile(True)
    for _ in range(steps):
        step()
    fg.synchronize()
    ctx.profile(False)
    prof = ctx.profile_read()
    return (t1 - t0) * 1000.0 / steps, prof


def by_kernel(prof, steps):
    """Average per-step device ms per kernel symbol."""
    agg = {}
    for r in prof:
        agg.setdefault(r["kernel"], []).append(r["ms"])
    return {k: {"calls_per_step": len(v) / steps, "avg_ms": float(np.mean(v)), "total_ms_per_step": float(np.sum(v)) / steps}
            for k, v in agg.items()}


def dominant(kern):
    name = max(kern, key=lambda k: kern[k]["total_ms_per_step"])
    return name, kern[name]


def cpu_baseline(config: str):
    try:
        r = subprocess.run([sys.executable, "-m", "oracle.cpu_bench", config], cwd=ROOT, capture_output=True,
                           text=True, timeout=300)
        if r.returncode != 0:
            log(f"cpu baseline {config} failed: {r.stderr[-2000:]}")
            return None
        return json.loads(r.stdout.strip().splitlines()[-1])
    except Exception as e:  # noqa: BLE001
        log(f"cpu baseline {config} failed: {e}")
        return None


def pmc_traffic(kernel: str):
    """HBM bytes per launch of `kernel` from the committed rocprofv3 --pmc
    FETCH_SIZE / WRITE_SIZE measurements (profiles/pmc_traffic.json), each
    scaled by the factor a plain 1 GiB copy kernel calibrates. Kernel symbols
    are content hashes of the generated source, so a kernel whose source
    changed since it was measured gets None (unmeasured), never a stale
    figure."""
    try:
        with open(os.path.join(ROOT, "profiles", "pmc_traffic.json")) as f:
            t = json.load(f)
    except (OSError, ValueError):
        return None
    k = t.get("kernels", {}).get(kernel)
    if not k:
        return None
    return (k["fetch_kib"] * t["fetch_factor"] + k["write_kib"] * t["write_factor"]) * 1024.0


def bench_c2(fg, ctx, steps, warmup):
    from ferrograd_amd import Tensor

    n = 1 << 26
    r = np.random.default_rng(2)
    host = [r.uniform(-1, 1, n).astype(np.float32) for _ in range(3)]
    a, b, c = (Tensor.new(h, [n], "hip") for h in host)
    holder = {}

    def step():
        holder["out"] = a.mul(b).add(c).relu().realize()

    ms, prof = timed(fg, ctx, step, steps, warmup)
    kern = by_kernel(prof, steps)
    name, dk = dominant(kern)
    alg = 4 * n * 4
    # The timed kernel's last output against float32 numpy rounding each op
    # once, as the reference's one-statement-per-op C does; relu as its
    # Where(0 < t, t, 0) (tensor.rs:517-531).
    t = host[0] * host[1] + host[2]
    want = np.where(np.float32(0) < t, t, np.float32(0))
    got = holder["out"].numpy().reshape(n)
    check = {"against": "float32 numpy, each op rounded once; relu as Where(0 < t, t, 0)",
             "elements": n, "bit_exact": bool(np.array_equal(got.view(np.uint32), want.view(np.uint32)))}
    return {"ms_per_step": ms, "gbs": alg / (ms / 1e3) / 1e9, "kernels": kern, "dominant": name, "check": check,
            "host_ms_per_step": timed.host_ms,
            "roofline": {"bound": "hbm", "achieved": alg / (dk["avg_ms"] / 1e3) / 1e9, "peak": HBM_PEAK_GBS,
                         "unit": "GB/s", "frac": alg / (dk["avg_ms"] / 1e3) / 1e9 / HBM_PEAK_GBS,
                         "traffic": pmc_traffic(name), "kernel": name, "algorithmic_bytes": alg,
                         "kernel_avg_ms": dk["avg_ms"]}}


def bench_c2_pcie(fg, steps):
    """C2 with the host handing over its buffers: upload a, b, c from
    (pageable) host memory, realise, read the result back. Reported beside the
    HBM-resident rate, never as the headline value."""
    from ferrograd_amd import Tensor

    n = 1 << 26
    r = np.random.default_rng(2)
    host = [r.uniform(-1, 1, n).astype(np.float32) for _ in range(3)]
    out = np.empty(n, np.float32)

    import ctypes

    def step():
        a, b, c = (Tensor.new(h, [n], "hip") for h in host)
        y = a.mul(b).add(c).relu().realize()
        # Device::copy_to_host straight into the caller's buffer.
        if fg.lib().fg_tensor_read(y._h, out.ctypes.data_as(ctypes.c_void_p), out.nbytes) != 0:
            raise fg.FerrogradError(fg.lib().fg_last_error().decode())

    step()
    fg.synchronize()
    t0 = time.perf_counter()
    for _ in range(steps):
        step()
    ms = (time.perf_counter() - t0) * 1000.0 / steps
    return {"ms_per_step": ms, "gbs": 4 * n * 4 / (ms / 1e3) / 1e9,
            "note": "3 x 256 MiB host->device + kernel + 256 MiB device->host per step, pageable host buffers "
                    "(copied through pinned 16 MiB chunks by several host threads while the other chunk's DMA runs)",
            "check": {"bit_exact": bool(np.array_equal(out, np.where(0 < (t := host[0] * host[1] + host[2]), t, 0)))}}


def bench_c1(fg, ctx, steps, warmup):
    from ferrograd_amd import Tensor

    # Six distinct inputs (6 x 64 MiB > the 256 MB Infinity Cache) rotate so
    # every step streams from HBM.
    x0 = np.random.default_rng(1).standard_normal((4096, 4096)).astype(np.float32)
    xs = [Tensor.new(x0 if i == 0 else np.random.default_rng(1 + i).standard_normal((4096, 4096)).astype(np.float32),
                     [4096, 4096], "hip") for i in range(6)]
    s0, s1 = Tensor.scalar(0.5, "hip"), Tensor.scalar(1.0, "hip")
    it = {"i": 0, "out": None}

    def step():
        x = xs[it["i"] % len(xs)]
        it["i"] += 1
        it["out"] = x.mul(s0).add(s1).relu().sum([1]).realize()

    ms, prof = timed(fg, ctx, step, steps, warmup)
    kern = by_kernel(prof, steps)
    name, dk = dominant(kern)
    alg = 4096 * 4096 * 4 + 4096 * 4
    ach = alg / (dk["avg_ms"] / 1e3) / 1e9
    # The timed kernel on the first input against float64: every term is >= 0,
    # so the bound 1e-4 * sum|terms| is a relative bound.
    got = xs[0].mul(s0).add(s1).relu().sum([1]).numpy().reshape(4096)
    want = np.maximum(x0.astype(np.float64) * 0.5 + 1.0, 0.0).sum(axis=1)
    rel = float(np.max(np.abs(got - want) / np.maximum(want, 1e-30)))
    check = {"against": "float64 row sums", "max_rel_err": rel, "tol": 1e-4, "ok": rel <= 1e-4}
    # Host pipeline phases per step (schedule key, plan lookup, launch, ...):
    # the gap between the kernel's rate and the per-realise rate.
    return {"ms_per_step": ms, "gbs": alg / (ms / 1e3) / 1e9, "kernels": kern, "check": check,
            "host_ms_per_step": timed.host_ms, "kernel_ms_per_step": dk["total_ms_per_step"],
            "roofline": {"bound": "hbm", "achieved": ach, "peak": HBM_PEAK_GBS, "unit": "GB/s",
                         "frac": ach / HBM_PEAK_GBS, "traffic": pmc_traffic(name), "kernel": name,
                         "algorithmic_bytes": alg, "kernel_avg_ms": dk["avg_ms"]}}


def bench_c3(fg, ctx, steps, warmup):
    from ferrograd_amd import Tensor

    r = np.random.default_rng(5)
    xh = r.standard_normal((4096, 4096)).astype(np.float32)
    wh = np.random.default_rng(6).uniform(-1 / 64, 1 / 64, (4096, 4096)).astype(np.float32)
    x = Tensor.new(xh, [4096, 4096], "hip")
    w = Tensor.new(wh, [4096, 4096], "hip")
    b = Tensor.zeros([4096], "hip")
    holder = {}

    def step():
        holder["y"] = x.matmul(w.permute([1, 0])).add(b).realize()

    ms, prof = timed(fg, ctx, step, steps, warmup)
    kern = by_kernel(prof, steps)
    gemm = [k for k in kern if k.endswith("_gemm")]  # 4096^3 fills the chip: no K split
    flops = 2 * 4096 ** 3
    g = kern[gemm[0]] if gemm else dominant(kern)[1]
    tf = flops / (g["avg_ms"] / 1e3) / 1e12
    # 64 sampled rows of the timed kernel's last output against float64, per
    # element within 1e-4 * sum_k |x w| (b is zero).
    rows = np.random.default_rng(7).choice(4096, 64, replace=False)
    got = holder["y"].numpy().reshape(4096, 4096)[rows]
    x64, w64 = xh[rows].astype(np.float64), wh.astype(np.float64)
    bound = 1e-4 * (np.abs(x64) @ np.abs(w64).T)
    worst = float(np.max(np.abs(got - x64 @ w64.T) / bound))
    check = {"against": "float64, 64 sampled rows", "max_err_over_bound": worst, "ok": worst <= 1.0}
    return {"ms_per_step": ms, "tflops_step": flops / (ms / 1e3) / 1e12, "kernels": kern, "check": check,
            "host_ms_per_step": timed.host_ms,
            "roofline": {"bound": "mfma", "achieved": tf, "peak": SPLIT_MFMA_PEAK_TFLOPS, "unit": "TFLOP/s",
                         "frac": tf / SPLIT_MFMA_PEAK_TFLOPS, "kernel": gemm[0] if gemm else None,
                         "traffic": pmc_traffic(gemm[0]) if gemm else None, "algorithmic_flops": flops,
                         "kernel_avg_ms": g["avg_ms"]}}


def mlp_gemm_flops(batch, dims):
    """Forward + backward GEMM FLOPs of one step (x needs no gradient)."""
    f = 0
    for i in range(len(dims) - 1):
        k, n = dims[i], dims[i + 1]
        f += 2 * batch * k * n          # forward
        f += 2 * batch * k * n          # dW
        if i > 0:
            f += 2 * batch * k * n      # dX
    return f


def bench_batched_loop(fg, model, opt, batch, dims, steps, nbatches=234):
    """examples/mnist.rs:84-98 as written: a resident training set of
    `nbatches` whole batches (234 of 256 rows: MNIST's 60,000 images), a new
    narrow()ed batch every step, run by fg_mlp_train_batches. Synthetic
    U(0,1) images and one-hot labels; the upload is outside the timing."""
    from ferrograd_amd.mlp import synthetic_batch, train_batches_native

    xs, ts = synthetic_batch(batch * nbatches, dims[0], dims[-1], 17, 18)
    x = fg.Tensor.new(xs, list(xs.shape), "hip")
    t = fg.Tensor.new(ts, list(ts.shape), "hip")
    train_batches_native(model, opt, x, t, batch, 8)
    fg.synchronize()
    s0 = fg.stats()
    t0 = time.perf_counter()
    losses = train_batches_native(model, opt, x, t, batch, steps, first_batch=8)
    fg.synchronize()
    ms = (time.perf_counter() - t0) * 1000.0 / steps
    s1 = fg.stats()
    return {"ms_per_step": ms, "steps_per_s": 1e3 / ms, "steps": steps,
            "steps_from_capture": s1["steps_replayed"] - s0["steps_replayed"],
            "dataset_rows": batch * nbatches, "losses_finite": bool(np.all(np.isfinite(losses))),
            "caller": "fg_mlp_train_batches: examples/mnist.rs:84-98 with batch i = rows narrow(0, 256*i, 256) of a "
                      "resident [59904, 784] set, one call for all timed steps; captured steps take the batch start "
                      "as a kernel argument of their replayed launches"}


def bench_mlp(fg, ctx, steps, warmup, batch, dims, native_steps=None, batched=False):
    from ferrograd_amd.mlp import mlp_setup, train_steps_native

    # The first step runs while the biases still hold allocate()'s zeros (a
    # plan of its own); the steady-state plan then schedules and compiles, and
    # is replayed (its block kernels batched and compiled on the first replay;
    # with FG_HIP_GRAPHS=1 recorded as a HIP graph on the second). Six steps
    # keep all of that out of the timed region, and the native warm-up call
    # also captures its step and replays it, compiling the captured
    # sequence's batches.
    warmup = max(warmup, 6)
    step, (model, opt, x, t) = mlp_setup(fg, "hip", batch=batch, dims=dims, with_state=True)
    losses = []
    ms, prof = timed(fg, ctx, lambda: losses.append(step()), steps, warmup)
    # The same loop body run from native code (fg_mlp_train_steps), as the
    # reference's compiled callers run it (examples/mnist.rs:84-101): one call
    # for all timed steps, each step still reading its loss back.
    train_steps_native(model, opt, x, t, warmup)
    fg.synchronize()
    s0 = fg.stats()
    t0 = time.perf_counter()
    native_steps = native_steps or steps
    native_losses = train_steps_native(model, opt, x, t, native_steps)
    fg.synchronize()
    ms_native = (time.perf_counter() - t0) * 1000.0 / native_steps
    s1 = fg.stats()
    h0, h1 = s0["host_ms"], s1["host_ms"]
    host_native = {k: (h1[k] - h0[k]) / native_steps for k in h1}
    # Steps of the timed call launched from its step capture (the call's
    # first steps record the plans and its last step runs in full).
    replayed = s1["steps_replayed"] - s0["steps_replayed"]
    host = timed.host_ms
    narrowed = bench_batched_loop(fg, model, opt, batch, dims, native_steps) if batched else None
    kern = by_kernel(prof, steps)
    check = check_mlp_step_on_device(fg, model, opt, x, t, batch, dims)
    check["losses_finite"] = bool(np.all(np.isfinite(losses + native_losses)))
    check["ok"] = check["ok"] and check["losses_finite"]
    # MFMA kernels: `_gemm`, or the `_gemm_part` / `_gemm_fin` pair of a split-K GEMM.
    gemm_ms = sum(v["total_ms_per_step"] for k, v in kern.items() if "_gemm" in k)
    dev_ms = sum(v["total_ms_per_step"] for v in kern.values())
    flops = mlp_gemm_flops(batch, dims)
    tf = lambda t: flops / (t / 1e3) / 1e12 / FP32_MFMA_PEAK_TFLOPS if t else None  # noqa: E731
    return {"ms_per_step": ms_native, "steps_per_s": 1e3 / ms_native,
            "caller": "native loop on one fixed resident batch (fg_mlp_train_steps: the loop body of "
                      "examples/mnist.rs:90-98, one call for all timed steps; steps after the first repeated ones "
                      "launch from the step capture as one sequence of direct launches, or one HIP graph with "
                      "FG_HIP_GRAPHS=1); *_python: the same steps driven op by op "
                      "from Python; narrowed_batches: the mnist.rs loop with a new narrow()ed batch every step",
            "narrowed_batches": narrowed,
            "native_steps": native_steps, "native_steps_from_capture": replayed,
            "ms_per_step_python": ms, "steps_per_s_python": 1e3 / ms,
            "device_ms_per_step": dev_ms, "host_ms_per_step": host_native, "host_ms_per_step_python": host,
            "kernels_per_step": sum(v["calls_per_step"] for v in kern.values()),
            "gemm_flops_per_step": flops, "gemm_ms_per_step": gemm_ms,
            # All of the step's GEMM FLOPs over the MFMA kernels' time (the narrow
            # N=10 products, 0.2% of C5's FLOPs, run as row/column reductions and
            # are counted in the numerator only), and over all device time.
            "mfma_frac_of_gemm_kernels": tf(gemm_ms), "mfma_frac_of_device_time": tf(dev_ms),
            "loss_first_last": [losses[0], native_losses[-1]] if losses else None,
            "check": check, "kernels": kern}


def check_mlp_step_on_device(fg, model, opt, x, t, batch, dims):
    """One more train step of the timed kernels (the same programs; the
    step holds its pre-activations, which the reference partition
    materialises anyway), checked product by product against float64 on the
    device's own values (tests/f64ref.py check_mlp_step): every forward
    product on 64 sampled batch rows, the loss, and each parameter's
    effective gradient (p0 - p1)/lr, for 64 sampled rows of each hidden
    layer's weight and every row of the last layer's."""
    sys.path.insert(0, os.path.join(ROOT, "tests"))
    import f64ref
    from ferrograd_amd.mlp import synthetic_batch, train_step

    xs, ts = synthetic_batch(batch, dims[0], dims[-1], 7, 8)  # the inputs mlp_setup made
    params = model.parameters()
    p0 = [p.numpy().copy() for p in params]
    zs = []
    loss = train_step(model, opt, x, t, zs).to_vec()[0]
    p1 = [p.numpy() for p in params]
    hidden = [z.numpy().reshape(batch, -1) for z in zs[:-1]]
    logits = zs[-1].numpy().reshape(batch, -1)
    r = np.random.default_rng(12)
    rows = [r.choice(d, min(d, 64), replace=False) for d in dims[1:-1]]
    t0 = time.perf_counter()
    rep = f64ref.check_mlp_step(xs, ts, p0, p1, loss, hidden, logits, rows=rows,
                                batch_rows=r.choice(batch, min(batch, 64), replace=False))
    rep["against"] = ("float64 on the device's own forward values: forward products on 64 batch rows, loss, "
                      "effective gradients (p0-p1)/lr on 64 sampled rows per hidden layer, 1e-4 of sum|terms|")
    rep["check_s"] = time.perf_counter() - t0
    return rep


COPY_SRC = r"""
extern "C" __global__ void __launch_bounds__(256) fg_copy_probe(float4* __restrict__ dst, const float4* __restrict__ src, int n4) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n4) dst[i] = src[i];
}
typedef float fg_probe_f4 __attribute__((ext_vector_type(4)));
extern "C" __global__ void __launch_bounds__(256) fg_copy_probe_nt(fg_probe_f4* __restrict__ dst, const fg_probe_f4* __restrict__ src, int n4) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n4) __builtin_nontemporal_store(__builtin_nontemporal_load(src + i), dst + i);
}
extern "C" __global__ void __launch_bounds__(256) fg_read_probe(float* __restrict__ dst, const fg_probe_f4* __restrict__ src, int n4) {
  // 16 non-temporal 16-byte loads per thread, all issued before the sum; one float written per thread.
  const int base = blockIdx.x * 4096 + threadIdx.x;
  fg_probe_f4 v[16];
  #pragma unroll
  for (int j = 0; j < 16; j++)
    v[j] = base + 256 * j < n4 ? __builtin_nontemporal_load(src + base + 256 * j) : fg_probe_f4{0.f, 0.f, 0.f, 0.f};
  float s = 0.f;
  #pragma unroll
  for (int j = 0; j < 16; j++) s += v[j].x + v[j].y + v[j].z + v[j].w;
  dst[blockIdx.x * 256 + threadIdx.x] = s;
}"""


def copy_probe(nbytes: int = 1 << 30, reps: int = 5) -> None:
    """Launch a plain copy of `nbytes` (read + write) `reps` times: the
    reference kernel whose FETCH_SIZE / WRITE_SIZE counters calibrate the
    byte counts of the generated kernels under rocprofv3 --pmc. Also times it,
    a non-temporal copy and a non-temporal read of `nbytes` with events: the
    practical streaming ceilings the HBM-bound kernels are compared with (3
    source/destination pairs rotate so the 256 MB Infinity Cache cannot hold a
    launch's data)."""
    from ferrograd_amd.hip import Arg, Context

    ctx = Context(0)
    pairs = [(ctx.alloc(nbytes), ctx.alloc(nbytes)) for _ in range(3)]
    prog = ctx.compile(COPY_SRC, "fg_copy_probe", 3)
    n4 = nbytes // 16
    grid, block = ((n4 + 255) // 256, 1, 1), (256, 1, 1)
    for _ in range(reps):
        src, dst = pairs[0]
        ctx.launch(prog, [Arg.ptr(dst), Arg.ptr(src), Arg.i32(n4)], grid=grid, block=block)
    ctx.sync()
    rates = {}
    for name in ("fg_copy_probe", "fg_copy_probe_nt", "fg_read_probe"):
        p = ctx.compile(COPY_SRC, name, 3)
        # The read probe's grid covers 16 float4 per thread; it writes one float
        # per thread (1/64 of the bytes read) into the destination.
        g = ((n4 + 4095) // 4096, 1, 1) if name == "fg_read_probe" else grid
        moved = nbytes if name == "fg_read_probe" else 2 * nbytes
        ms = []
        for i in range(3 + 20):
            src, dst = pairs[i % 3]
            ctx.record(0)
            ctx.launch(p, [Arg.ptr(dst), Arg.ptr(src), Arg.i32(n4)], grid=g, block=block)
            ctx.record(1)
            if i >= 3:
                ms.append(ctx.elapsed_ms(0, 1))
        rates[name + "_us"] = float(np.mean(ms)) * 1e3
        rates[name + "_gbs"] = moved / (float(np.mean(ms)) / 1e3) / 1e9
    print(json.dumps({"copy_probe_bytes_read": nbytes, "copy_probe_bytes_written": nbytes, "launches": reps, **rates}))


def library_compare() -> None:
    """Reference points from the vendor libraries on the same GPU: torch's fp32
    matmul (hipBLASLt / rocBLAS, TF32 off) at C3's 4096^3, and torch's add over
    2^26 f32 elements (2 reads + 1 write). Not part of the ferrograd path."""
    import torch

    torch.backends.cuda.matmul.allow_tf32 = False
    x, w = torch.randn(4096, 4096, device="cuda"), torch.randn(4096, 4096, device="cuda")
    a, b = torch.rand(1 << 26, device="cuda"), torch.rand(1 << 26, device="cuda")
    o = torch.empty_like(a)

    def time_ms(fn, reps=20):
        for _ in range(5):
            fn()
        torch.cuda.synchronize()
        s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        s.record()
        for _ in range(reps):
            fn()
        e.record()
        torch.cuda.synchronize()
        return s.elapsed_time(e) / reps

    mm = time_ms(lambda: torch.mm(x, w.t()))
    add = time_ms(lambda: torch.add(a, b, out=o))
    print(json.dumps({"torch_fp32_mm_4096_ms": mm, "torch_fp32_mm_tflops": 2 * 4096 ** 3 / mm / 1e9,
                      "torch_add_2^26_ms": add, "torch_add_gbs": 3 * 4 * (1 << 26) / add / 1e6}))


def shard_sweep(steps: int) -> None:
    """C5 (784->4096->4096->10) at B = 8192/p for p = 1, 2, 4, 8: the shape one
    GPU runs under p-way data parallelism, before the gradient all-reduce
    (which one GPU cannot show). One JSON line per p."""
    import ferrograd_amd as fg
    from ferrograd_amd.hip import Context

    ctx = Context.of_device()
    dims = (784, 4096, 4096, 10)
    for p in (1, 2, 4, 8):
        b = 8192 // p
        r = bench_mlp(fg, ctx, max(4, steps // 4), 2, b, dims)
        log(f"p={p} B={b}: {r['steps_per_s']:.1f} steps/s, device {r['device_ms_per_step']:.3f} ms, "
            f"gemm {r['mfma_frac_of_gemm_kernels']:.3f} of peak")
        print(json.dumps({"p": p, "batch": b, "ms_per_step": r["ms_per_step"], "steps_per_s": r["steps_per_s"],
                          "device_ms_per_step": r["device_ms_per_step"],
                          "gemm_ms_per_step": r["gemm_ms_per_step"],
                          "mfma_frac_of_gemm_kernels": r["mfma_frac_of_gemm_kernels"],
                          "samples_per_s": r["steps_per_s"] * b}), flush=True)


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--only", default=None, help="run one config: c1,c2,c3,c4,c5")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--kernels", action="store_true", help="include per-kernel tables")
    ap.add_argument("--copy-probe", action="store_true", help="only run the 1 GiB copy calibration kernel")
    ap.add_argument("--probe-mib", type=int, default=1024, help="bytes the copy probe copies, in MiB")
    ap.add_argument("--library-compare", action="store_true", help="only time torch's fp32 mm and add for reference")
    ap.add_argument("--shard-sweep", action="store_true",
                    help="only time the C5 step at the per-GPU batch of 1, 2, 4 and 8-way data parallelism")
    args = ap.parse_args()
    if args.copy_probe:
        copy_probe(args.probe_mib << 20)
        return
    if args.library_compare:
        library_compare()
        return
    if args.shard_sweep:
        shard_sweep(args.steps)
        return
    if args.gpus != 1:
        print(f"bench.py measures one MI355X; --gpus {args.gpus} is not supported in this build "
              "(every config here runs on one GPU; sharding across GPUs is not built)", file=sys.stderr)
        sys.exit(2)

    import ferrograd_amd as fg
    from ferrograd_amd.hip import Context

    ctx = Context.of_device()
    info = ctx.info()
    log(f"device: {info}")
    only = set(args.only.split(",")) if args.only else {"c1", "c2", "c3", "c4", "c5"}
    sec = {}
    t_start = time.time()
    if "c2" in only:
        c2 = bench_c2(fg, ctx, args.steps, args.warmup)
        log(f"c2: {c2['gbs']:.1f} GB/s per step, kernel {c2['roofline']['achieved']:.1f} GB/s "
            f"({100 * c2['roofline']['frac']:.1f}% of HBM peak), bit-exact: {c2['check']['bit_exact']}")
        sec["c2_pcie_inclusive"] = bench_c2_pcie(fg, 3)
        log(f"c2 with host buffers: {sec['c2_pcie_inclusive']['gbs']:.1f} GB/s")
    if "c1" in only:
        sec["c1"] = bench_c1(fg, ctx, args.steps, args.warmup)
        log(f"c1: {sec['c1']['gbs']:.1f} GB/s, kernel {sec['c1']['roofline']['achieved']:.1f} GB/s")
    if "c3" in only:
        # Ten warmup GEMMs (10 ms): after three, the clock was still ramping and
        # the first timed steps ran 9% slower than steady state.
        sec["c3"] = bench_c3(fg, ctx, max(5, args.steps // 2), max(10, args.warmup))
        log(f"c3: gemm {sec['c3']['roofline']['achieved']:.1f} TFLOP/s ({100 * sec['c3']['roofline']['frac']:.1f}%)")
    if "c4" in only:
        # The native call records its capture in its first steps and runs its
        # last in full; 200 steps (about 12 ms) make that a realistic loop's share.
        sec["c4"] = bench_mlp(fg, ctx, args.steps, args.warmup, 256, (784, 128, 10),
                              native_steps=max(args.steps, 200), batched=True)
        log(f"c4: {sec['c4']['steps_per_s']:.1f} steps/s (native loop, fixed batch), "
            f"{sec['c4']['narrowed_batches']['steps_per_s']:.1f} (native loop, narrowed batches), "
            f"{sec['c4']['steps_per_s_python']:.1f} from Python")
    if "c5" in only:
        sec["c5"] = bench_mlp(fg, ctx, max(3, args.steps // 4), 2, 8192, (784, 4096, 4096, 10))
        log(f"c5: {sec['c5']['steps_per_s']:.2f} steps/s (native loop), {sec['c5']['steps_per_s_python']:.2f} from Python, "
            f"gemm {sec['c5']['mfma_frac_of_gemm_kernels']}")
    log(f"gpu legs took {time.time() - t_start:.1f}s")

    cpu = {}
    if not args.no_cpu:
        for c in sorted(only & {"c1", "c2", "c3", "c4", "c5"}):
            cpu[c] = cpu_baseline(c)
            log(f"cpu {c}: {cpu[c]}")
    for c, v in cpu.items():
        if c in sec and v:
            sec[c]["cpu_baseline"] = v
    if not args.kernels:
        for v in sec.values():
            v.pop("kernels", None)

    if "c2" in only:
        c2cpu = cpu.get("c2")
        line = {
            "metric": METRIC, "value": c2["gbs"], "unit": "GB/s", "n_gpus": 1, "steps": args.steps,
            "warmup": args.warmup, "ms_per_step": c2["ms_per_step"], "higher_is_better": True, "scaling": "weak",
            "vs_baseline": None, "dtype": "f32", "data": "synthetic (seeded U(-1,1))",
            "config": {"workload": "C2: out = (a*b + c).relu(), a,b,c f32[2^26], one fused kernel (3 reads + 1 write)",
                       "elements": 1 << 26, "algorithmic_bytes_per_step": 4 * (1 << 26) * 4},
            "roofline": c2["roofline"], "check": c2["check"],
            "cpu_baseline": ({"value": c2cpu["value"], "unit": "GB/s", "cores": c2cpu["cores"], "kind": c2cpu["kind"],
                              "sample": c2cpu["sample"], "host": c2cpu.get("host")} if c2cpu else None),
            "device": info, "secondary": sec,
        }
    else:
        k = sorted(sec)[0]
        line = {"metric": METRIC, "value": None, "unit": None, "n_gpus": 1, "steps": args.steps,
                "warmup": args.warmup, "config": {"workload": ",".join(sorted(only))}, "secondary": sec,
                "device": info}
    print(json.dumps(line))


if __name__ == "__main__":
    main()
