"""Throughput of the int8 NHWC convolution on one MI355X.

    python bench.py [--steps K] [--warmup W] [--config r50_3x3] [--cache cold|warm] [--all]
    python bench.py --bmm [--config r50_3x3_im2col]      # the int32 matrix product instead
    python bench.py --fp32 [--config resnet_like_56x56]  # the fp32 convolution (conv_bench suite)
    python bench.py --fp32 --blocked [--op bprop]        # the blocked fp32 convolution (blocked suite)
    python bench.py --fallback                           # v_dot4 kernel against the MFMA kernels on thin layers
    python bench.py --qi32 [--config r50_3x3]            # the reference's float-code API

One step = one fused conv + bias + requantize (+ ReLU) pass of libmiq_qconv over one batch
of synthetic int8 input, with inputs already resident in HBM.  Every BASELINE.json config is
timed; the headline (configs[1]: ResNet-50 conv2_x 3x3, N=32) is the line's `value`, the
others are in its "configs" block.  Prints ONE JSON line (the driver's contract).

Timing: W untimed warmup steps, then exactly K steps bracketed by device synchronisation,
timed with HIP events on the stream the kernels run on.  The K launches are recorded once
into a HIP graph and replayed, so host launch cost does not gap the GPU; `--eager` times
plain back-to-back launches instead.  A bounded spin kernel queued before the start event
holds the GPU while the host submits the replay, so the region times the K steps' execution
and not the replay's submission latency (a fixed ~30 us that would otherwise be spread over
the K steps and dominate at small K).  With --cache cold (default) every timed step reads and
writes its own buffer set (a pooled buffer of up to 4 GiB, filled by one copy kernel), and a
512 MiB read just before the timed region leaves no step's data in L2 or the 256 MiB
Infinity Cache (MALL); --cache warm reuses one set.

cpu_baseline: the reference's own CPU path (cpu_ref.cpp compiled in oracle/_ref, -O3, one
thread, float codes as the reference stores them) on the full workload, else this
repository's C restatement of it.
"""
from __future__ import annotations

import argparse
import json
import os
import platform
import sys
import time
from pathlib import Path

ROOT = Path(__file__).resolve().parent
sys.path.insert(0, str(ROOT))

METRIC = "int8 conv TOPS + % of MI355X int8 MFMA peak, ResNet-50 3x3 layer N=32"
PEAK_INT8_TOPS = 5000.0   # dense int8 MFMA, MI355X
PEAK_HBM_GBS = 8000.0
MALL_BYTES = 256 << 20
FLUSH_BYTES = 2 * MALL_BYTES   # read before each timed region (cold)
POOL_BYTES = 4 << 30           # cold buffer pool per config: one input/output set per timed step up to this


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=400)
    ap.add_argument("--warmup", type=int, default=40)
    ap.add_argument("--config", default=None)
    ap.add_argument("--cache", choices=["cold", "warm"], default="cold")
    ap.add_argument("--eager", action="store_true")
    ap.add_argument("--algo", default="auto")
    ap.add_argument("--all", action="store_true", help="(kept for old command lines: every config is timed by default)")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--bmm", action="store_true",
                    help="measure the int32 batched matrix product (bmm_matmul_i32) instead of the convolution")
    ap.add_argument("--fp32", action="store_true",
                    help="measure the fp32 convolution (launch_fprop_nhwc) on the reference's conv_bench suite")
    ap.add_argument("--qi32", action="store_true",
                    help="measure the reference's float-code API (launch_fprop_nhwc_qi32, LinQuantU8) on the workloads")
    ap.add_argument("--fallback", action="store_true",
                    help="time the vector-ALU dot4 kernel against the MFMA kernels on thin-channel and few-output-"
                         "channel layers (every kernel family that accepts each shape)")
    ap.add_argument("--blocked", action="store_true",
                    help="with --fp32: the blocked convolution (launch_block_*_nhwc) on the reference's blocked suite")
    ap.add_argument("--op", choices=["fprop", "bprop", "grad"], default="fprop",
                    help="with --fp32: the pass to time (launch_fprop_nhwc / launch_bprop_nhwc / launch_grad_nhwc)")
    ap.add_argument("--copy-mb", type=int, default=0,
                    help="only run a plain device-to-device copy of this many MiB (counter calibration)")
    return ap.parse_args()


_SLEEP_CYCLES_PER_US = None


def gpu_hold(us: float) -> None:
    """Queue a spin kernel of about `us` microseconds on the current stream (torch's bounded
    clock loop).  Queued just before a timed region's start event, it keeps the GPU busy
    while the host submits the region's launches (a graph replay, or eager launches), so the
    start event is reached with those launches already queued: the region then measures the
    GPU's back-to-back execution of the K steps, not the host's submission latency."""
    import torch

    global _SLEEP_CYCLES_PER_US
    if _SLEEP_CYCLES_PER_US is None:
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        torch.cuda._sleep(1 << 16)  # first call loads the kernel
        a.record()
        torch.cuda._sleep(1 << 22)
        b.record()
        torch.cuda.synchronize()
        _SLEEP_CYCLES_PER_US = (1 << 22) / max(a.elapsed_time(b) * 1e3, 1.0)
    torch.cuda._sleep(int(us * _SLEEP_CYCLES_PER_US))


def hold_us(steps: int, per_step_us: float) -> float:
    """Hold long enough for the host to submit `steps` launches, at most 50 ms."""
    return min(100.0 + per_step_us * steps, 50_000.0)


def copy_calibration(mib: int) -> None:
    """A plain copy kernel of known size: the reference point that scales the FETCH_SIZE /
    WRITE_SIZE counters of rocprofv3 into bytes."""
    import torch

    n = mib << 20
    src = torch.ones(n, dtype=torch.uint8, device="cuda")
    dst = torch.empty_like(src)
    flush = torch.empty(512 << 20, dtype=torch.uint8, device="cuda")
    for _ in range(3):
        flush.fill_(1)  # evicts src/dst from L2 and MALL between copies
        dst.copy_(src)
    torch.cuda.synchronize()
    print(json.dumps({"copy_bytes": n, "launches": 3}), flush=True)


# int32 products: (name, batch, M, N, K, trans_a, trans_b).  The first is the reference's own
# call site on the headline layer (cuda_kernels.cu:1381: im2col columns of ResNet-50 conv2_x,
# N=32, times the packed 64 x 576 filter, trans_b); the rest are plain square and batched
# products.
BMM_SHAPES = [
    ("r50_3x3_im2col", 1, 32 * 56 * 56, 64, 576, False, True),
    ("square_4096", 1, 4096, 4096, 4096, False, False),
    ("batched_512", 32, 512, 512, 512, False, False),
    ("square_4096_tt", 1, 4096, 4096, 4096, True, True),
]
BMM_BYTE_PRODUCTS = 16  # int8 MFMA products per int32 multiply-add (4 shift groups x 4 digit bytes)


def bmm_traffic(name: str):
    """HBM bytes per launch of a --bmm shape from its committed rocprofv3 counter summary, or None."""
    f = ROOT / "profiles" / f"traffic_bmm_{name}.json"
    try:
        return json.loads(f.read_text()).get("bytes_per_launch") if f.exists() else None
    except (ValueError, OSError):
        return None


def bench_bmm(args) -> None:
    """Times bmm_matmul_i32 per shape (HIP events over back-to-back launches on one stream),
    checks sampled rows against the oracle, prints a table on stderr and one JSON line."""
    import numpy as np
    import torch

    import my_own_cnn_amd as M
    import oracle  # checker of sampled output rows and the cpu_baseline leg only

    dev = torch.device("cuda:0")
    peak = PEAK_INT8_TOPS / BMM_BYTE_PRODUCTS  # int32 ops/s the int8 matrix cores can deliver
    rows = []
    shapes = [sh for sh in BMM_SHAPES if args.config in (None, sh[0])]
    if not shapes:
        print(f"bench.py: unknown --bmm shape {args.config}; known: {[sh[0] for sh in BMM_SHAPES]}", file=sys.stderr)
        sys.exit(2)
    for name, batch, m, n, k, ta, tb in shapes:
        gen = torch.Generator(device=dev)
        gen.manual_seed(1234)
        a = torch.randint(-2 ** 31, 2 ** 31 - 1, (batch, k, m) if ta else (batch, m, k), dtype=torch.int32,
                          device=dev, generator=gen)
        b = torch.randint(-2 ** 31, 2 ** 31 - 1, (batch, n, k) if tb else (batch, k, n), dtype=torch.int32,
                          device=dev, generator=gen)
        c = torch.empty((batch, m, n), dtype=torch.int32, device=dev)
        stream = torch.cuda.current_stream()

        def step():
            M.bmm_matmul_i32(a, b, c, batch, m, n, k, ta, tb, stream=stream)

        step()
        torch.cuda.synchronize()
        # exact check of 64 sampled output rows of the first and last batch entries
        rng = np.random.default_rng(7)
        pick = np.sort(rng.choice(m, size=min(m, 64), replace=False))
        an, bn, cn = a.cpu().numpy(), b.cpu().numpy(), c.cpu().numpy()
        ok = True
        for bi in {0, batch - 1}:
            asub = an[bi][:, pick] if ta else an[bi][pick]
            want = oracle.bmm_i32(asub[None], bn[bi][None], ta, tb)[0]
            ok &= bool(np.array_equal(cn[bi][pick], want))
        for _ in range(args.warmup):
            step()
        t0, t1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        torch.cuda.synchronize()
        gpu_hold(hold_us(args.steps, 25.0))
        t0.record(stream)
        for _ in range(args.steps):
            step()
        t1.record(stream)
        torch.cuda.synchronize()
        ms = t0.elapsed_time(t1) / args.steps
        ops = 2.0 * batch * m * n * k
        tops = ops / (ms * 1e-3) / 1e12
        rows.append(dict(name=name, batch=batch, M=m, N=n, K=k, trans_a=ta, trans_b=tb, us=round(ms * 1e3, 3),
                         tops=round(tops, 3), frac=round(tops / peak, 4), exact_sampled=ok))
        del a, b, c
        torch.cuda.empty_cache()
    print(f"{'shape':16s} {'batch':>5s} {'M':>7s} {'N':>5s} {'K':>5s} {'tt':2s} {'us':>10s} {'TOPS':>8s} {'frac':>6s} exact",
          file=sys.stderr)
    for r in rows:
        print(f"{r['name']:16s} {r['batch']:5d} {r['M']:7d} {r['N']:5d} {r['K']:5d} {int(r['trans_a'])}{int(r['trans_b'])} "
              f"{r['us']:10.2f} {r['tops']:8.2f} {r['frac']:6.3f} {r['exact_sampled']}", file=sys.stderr)
    head = rows[0]
    line = {
        "metric": "int32 bmm TOPS (wrap-around int32, 2 ops per multiply-add), reference call site on the "
                  "ResNet-50 3x3 layer N=32",
        "value": head["tops"], "unit": "TOPS", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": round(head["us"] / 1e3, 6), "higher_is_better": True, "scaling": "weak",
        "vs_baseline": None, "dtype": "int32", "data": "synthetic",
        "config": {"workload": head["name"], "batch": head["batch"], "M": head["M"], "N": head["N"], "K": head["K"],
                   "trans_a": head["trans_a"], "trans_b": head["trans_b"], "timing": "eager back-to-back"},
        "roofline": {"bound": "mfma", "achieved": head["tops"], "peak": peak, "unit": "TOPS",
                     "frac": head["frac"], "traffic": bmm_traffic(head["name"]),
                     "peak_note": f"int8 MFMA {PEAK_INT8_TOPS:.0f} TOPS / {BMM_BYTE_PRODUCTS} byte products per "
                                  "int32 multiply-add"},
        "shapes": rows,
    }
    if not args.no_cpu_baseline and head["name"] == BMM_SHAPES[0][0]:
        _, batch, m, n, k, ta, tb = BMM_SHAPES[0]
        rng = np.random.default_rng(3)
        msub = 2048
        a = rng.integers(-2 ** 31, 2 ** 31, size=(1, msub, k), dtype=np.int64).astype(np.int32)
        b = rng.integers(-2 ** 31, 2 ** 31, size=(1, n, k), dtype=np.int64).astype(np.int32)
        t0 = time.perf_counter()
        oracle.bmm_i32(a, b, False, True, nthreads=1)
        secs = time.perf_counter() - t0
        line["cpu_baseline"] = {
            "value": round(2.0 * msub * n * k / secs / 1e12, 6), "unit": "TOPS", "cores": 1, "kind": "port",
            "sample": f"{msub} of the {m} rows of {BMM_SHAPES[0][0]} ({2.0 * msub * n * k / 1e9:.2f} Gop) in "
                      f"{secs:.2f} s; oracle/qconv_oracle.c orc_bmm_i32 (gcc -O3), 1 thread on {cpu_model()}",
        }
    print(json.dumps(line), flush=True)


# The reference's conv_bench default suite (src/main.cpp:163-174):
# (name, n, h, w, c, k, r, s, (pad_h, pad_w, stride_h, stride_w, dil_h, dil_w, groups))
FP32_SUITE = [
    ("resnet_like_56x56", 32, 56, 56, 64, 64, 3, 3, (1, 1, 1, 1, 1, 1, 1)),
    ("resnet_like_28x28", 32, 28, 28, 128, 256, 3, 3, (1, 1, 1, 1, 1, 1, 1)),
    ("downsample_stride2", 32, 112, 112, 32, 32, 3, 3, (1, 1, 2, 2, 1, 1, 1)),
    ("depthwise_3x3", 32, 56, 56, 128, 128, 3, 3, (1, 1, 1, 1, 1, 1, 128)),
    ("grouped_g4", 32, 56, 56, 128, 128, 3, 3, (1, 1, 1, 1, 1, 1, 4)),
    ("pointwise_1x1", 32, 56, 56, 128, 256, 1, 1, (0, 0, 1, 1, 1, 1, 1)),
    ("dilated_3x3", 16, 64, 64, 64, 64, 3, 3, (2, 2, 1, 1, 2, 2, 1)),
    ("small_batch", 1, 56, 56, 64, 64, 3, 3, (1, 1, 1, 1, 1, 1, 1)),
]
# The reference's blocked bench suite (src/main.cpp:176-186): the same fields, then the block grid.
BLOCKED_SUITE = [
    ("blocked_resnet_56x56_b2x2", 32, 56, 56, 64, 64, 3, 3, (1, 1, 1, 1, 1, 1, 1), 2, 2),
    ("blocked_resnet_56x56_b4x4", 32, 56, 56, 64, 64, 3, 3, (1, 1, 1, 1, 1, 1, 1), 4, 4),
    ("blocked_resnet_28x28_b2x4", 32, 28, 28, 128, 256, 3, 3, (1, 1, 1, 1, 1, 1, 1), 2, 4),
    ("blocked_grouped_g4_b2x2", 32, 56, 56, 128, 128, 3, 3, (1, 1, 1, 1, 1, 1, 4), 2, 2),
    ("blocked_pointwise_1x1_b4x4", 32, 56, 56, 128, 256, 1, 1, (0, 0, 1, 1, 1, 1, 1), 4, 4),
    ("blocked_dilated_3x3_b2x2", 16, 64, 64, 64, 64, 3, 3, (2, 2, 1, 1, 2, 2, 1), 2, 2),
    ("blocked_small_batch_b4x4", 1, 56, 56, 64, 64, 3, 3, (1, 1, 1, 1, 1, 1, 1), 4, 4),
]
PEAK_FP32_TFLOPS = 157.3  # dense fp32 MFMA, MI355X
PEAK_SPLIT_TFLOPS = 2500.0 / 6  # dense bf16 MFMA, six products per fp32 one (split operands)


def bench_fp32(args) -> None:
    """Times launch_fprop_nhwc / launch_bprop_nhwc / launch_grad_nhwc on the conv_bench suite, or
    with --blocked launch_block_{fprop,bprop,grad}_nhwc on the blocked suite (HIP events over
    back-to-back launches); checks image 0 of every shape against the oracle (fprop, bprop) or
    all images against the bit-exact direct kernel (grad) with the reference's verify rule,
    prints a table on stderr and one JSON line for the first shape."""
    import numpy as np
    import torch

    import my_own_cnn_amd as M
    import oracle  # checker of the sampled image and the cpu_baseline leg only

    dev = torch.device("cuda:0")
    suite = BLOCKED_SUITE if args.blocked else FP32_SUITE
    rows = []
    for case in suite:
        name, n, h, w, c, k, r, s_, conv = case[:9]
        by, bx = case[9:] if args.blocked else (1, 1)
        if args.config not in (None, name):
            continue
        ph, pw, sh, sw, dh, dw, g = conv
        bp = M.BlockConv2DParams(M.Conv2DParams(*conv), by, bx)
        ho, wo = M.infer_conv_shape(n, h, w, c, r, s_, k, M.Conv2DParams(*conv))
        gen = torch.Generator(device=dev)
        gen.manual_seed(42)
        x = torch.rand((n, h, w, c), device=dev, generator=gen) * 2 - 1
        wshape = (k, by, bx, r, s_, c // g) if args.blocked else (k, r, s_, c // g)
        wt = torch.rand(wshape, device=dev, generator=gen) * 2 - 1
        y = torch.empty((n, ho, wo, k), device=dev)
        stream = torch.cuda.current_stream()

        def fprop(out, algo="auto"):
            if args.blocked:
                M.launch_block_fprop_nhwc(x, wt, out, n, h, w, c, r, s_, k, bp, algo=algo, stream=stream)
            else:
                M.launch_fprop_nhwc(x, wt, out, n, h, w, c, r, s_, k, conv, algo=algo, stream=stream)

        def bprop(dy, out, algo="auto"):
            if args.blocked:
                M.launch_block_bprop_nhwc(dy, wt, out, n, h, w, c, r, s_, k, bp, algo=algo, stream=stream)
            else:
                M.launch_bprop_nhwc(dy, wt, out, n, h, w, c, r, s_, k, conv, algo=algo, stream=stream)

        def grad(dy, out, algo="auto", xin=None):
            xin = x if xin is None else xin
            if args.blocked:
                M.launch_block_grad_nhwc(xin, dy, out, n, h, w, c, r, s_, k, bp, algo=algo, stream=stream)
            else:
                M.launch_grad_nhwc(xin, dy, out, n, h, w, c, r, s_, k, conv, algo=algo, stream=stream)

        if args.op == "fprop":
            fprop(y)
            torch.cuda.synchronize()
            x1, w1 = x[:1].cpu().numpy(), wt.cpu().numpy()
            want = oracle.block_conv_f32(x1, w1, conv) if args.blocked else oracle.conv_f32(x1, w1, conv)
            ok = oracle.verify_tensors(want, y[:1].cpu().numpy(), 1e-4, 1e-3)

            def step():
                fprop(y)
        elif args.op == "bprop":
            dy = torch.rand(y.shape, device=dev, generator=gen) * 2 - 1
            dx = torch.empty_like(x)
            bprop(dy, dx)
            torch.cuda.synchronize()
            dy1, w1 = dy[:1].cpu().numpy(), wt.cpu().numpy()
            want = (oracle.block_bprop_f32(dy1, w1, (1, h, w, c), conv) if args.blocked
                    else oracle.bprop_f32(dy1, w1, (1, h, w, c), conv))
            ok = oracle.verify_tensors(want, dx[:1].cpu().numpy(), 1e-4, 1e-3)

            def step():
                bprop(dy, dx)
        else:
            dy = torch.rand(y.shape, device=dev, generator=gen) * 2 - 1
            dw = torch.empty_like(wt)
            # checked on the image-0 problem against the oracle (the reference loop's order) under
            # the reference's verify rule; at the full batch the reference's own sequential fp32
            # sum over N*Ho*Wo terms drifts past that rule, so it cannot be the yardstick there
            x0, dy0, dw0 = x[:1].contiguous(), dy[:1].contiguous(), torch.empty_like(wt)
            if args.blocked:
                M.launch_block_grad_nhwc(x0, dy0, dw0, 1, h, w, c, r, s_, k, bp, stream=stream)
            else:
                M.launch_grad_nhwc(x0, dy0, dw0, 1, h, w, c, r, s_, k, conv, stream=stream)
            grad(dy, dw)
            torch.cuda.synchronize()
            x1, dy1 = x0.cpu().numpy(), dy0.cpu().numpy()
            want = (oracle.block_grad_f32(x1, dy1, wshape, conv) if args.blocked
                    else oracle.grad_f32(x1, dy1, wshape, conv))
            ok = oracle.verify_tensors(want, dw0.cpu().numpy(), 1e-4, 1e-3)
            # and at the full timed size on small-integer inputs, where every partial sum is an
            # exact fp32 integer in any order: AUTO must equal the direct kernel bit for bit
            xi = torch.randint(-3, 4, x.shape, device=dev, generator=gen).float()
            dyi = torch.randint(-3, 4, dy.shape, device=dev, generator=gen).float()
            grad(dyi, dw, xin=xi)
            dw_ref = torch.empty_like(wt)
            grad(dyi, dw_ref, "direct", xin=xi)
            torch.cuda.synchronize()
            ok = ok and torch.equal(dw, dw_ref)
            del xi, dyi, dw_ref

            def step():
                grad(dy, dw)
        for _ in range(args.warmup):
            step()
        t0, t1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        torch.cuda.synchronize()
        gpu_hold(hold_us(args.steps, 25.0))
        t0.record(stream)
        for _ in range(args.steps):
            step()
        t1.record(stream)
        torch.cuda.synchronize()
        ms = t0.elapsed_time(t1) / args.steps
        flops = 2.0 * n * ho * wo * k * r * s_ * (c // g)  # conv_flops, src/main.cpp:143-145
        nbytes = 4.0 * (x.numel() + wt.numel() + y.numel())
        # what the library dispatches, and the matrix rate of that
        algo = (M.plan_block_f32(args.op, n, h, w, c, r, s_, k, bp) if args.blocked
                else M.plan_f32(args.op, n, h, w, c, r, s_, k, M.Conv2DParams(*conv)))
        split = M.plan_f32_split(args.op, n, h, w, c, r, s_, k, bp if args.blocked else M.Conv2DParams(*conv))
        if split:
            algo = "split " + algo
        peak = PEAK_SPLIT_TFLOPS if split else PEAK_FP32_TFLOPS
        t_mfma = flops / (peak * 1e12)
        t_hbm = nbytes / (PEAK_HBM_GBS * 1e9)
        bound = "mfma" if t_mfma >= t_hbm else "hbm"
        tf = flops / (ms * 1e-3) / 1e12
        gbs = nbytes / (ms * 1e-3) / 1e9
        frac = tf / peak if bound == "mfma" else gbs / PEAK_HBM_GBS
        rows.append(dict(name=name, n=n, h=h, w=w, c=c, k=k, r=r, s=s_, groups=g, stride=sh, by=by, bx=bx, kernel=algo,
                         us=round(ms * 1e3, 2), tflops=round(tf, 3), gbs=round(gbs, 1), bound=bound,
                         peak=round(peak, 1), frac=round(frac, 4), verified=ok,
                         verified_on=("the image-0 problem vs the oracle; the full problem on small integers, AUTO "
                                      "== direct bit for bit" if args.op == "grad" else "image 0 vs the oracle")))
        del x, wt, y
        torch.cuda.empty_cache()
    if not rows:
        print(f"bench.py: unknown --fp32 shape {args.config}; known: {[c[0] for c in suite]}", file=sys.stderr)
        sys.exit(2)
    print(f"{'shape':28s} {'kernel':17s} {'us':>10s} {'TFLOP/s':>8s} {'GB/s':>8s} {'bound':5s} {'frac':>6s} verified",
          file=sys.stderr)
    for r in rows:
        print(f"{r['name']:28s} {r['kernel']:17s} {r['us']:10.2f} {r['tflops']:8.2f} {r['gbs']:8.1f} {r['bound']:5s} "
              f"{r['frac']:6.3f} {r['verified']}", file=sys.stderr)
    head = rows[0]
    suite_name = ("blocked bench suite (src/main.cpp:176-186)" if args.blocked
                  else "conv_bench default suite (src/main.cpp:163-174)")
    line = {
        "metric": f"fp32 {'blocked ' if args.blocked else ''}conv {args.op} TFLOP/s, {suite_name}",
        "value": head["tflops"], "unit": "TFLOP/s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": round(head["us"] / 1e3, 6), "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
        "dtype": "f32", "data": "synthetic",
        "config": {"workload": head["name"], "N": head["n"], "H": head["h"], "W": head["w"], "C": head["c"],
                   "K": head["k"], "R": head["r"], "S": head["s"], "groups": head["groups"], "by": head["by"],
                   "bx": head["bx"], "kernel": head["kernel"], "timing": "eager back-to-back", "cache": "warm"},
        "roofline": {"bound": head["bound"], "achieved": head["tflops"] if head["bound"] == "mfma" else head["gbs"],
                     "peak": head["peak"] if head["bound"] == "mfma" else PEAK_HBM_GBS,
                     "unit": "TFLOP/s" if head["bound"] == "mfma" else "GB/s", "frac": head["frac"], "traffic": None},
        "shapes": rows,
    }
    if not args.no_cpu_baseline and head["name"] == suite[0][0] and args.op == "fprop":
        _, n, h, w, c, k, r, s_, conv = suite[0][:9]
        by, bx = suite[0][9:] if args.blocked else (1, 1)
        rng = np.random.default_rng(3)
        x1 = rng.uniform(-1, 1, size=(1, h, w, c)).astype(np.float32)
        if args.blocked:
            w1 = rng.uniform(-1, 1, size=(k, by, bx, r, s_, c // conv[6])).astype(np.float32)
        else:
            w1 = rng.uniform(-1, 1, size=(k, r, s_, c // conv[6])).astype(np.float32)
        fn = "cpu_block_fprop_nhwc" if args.blocked else "cpu_fprop_nhwc"
        if oracle.ref() is not None:
            if args.blocked:
                y1, secs, _ = oracle.ref_block_f32("fprop", x1, w1, x1.shape, w1.shape, conv)
            else:
                y1, secs = oracle.ref_conv_f32(x1, w1, conv)
            kind, what = "reference", f"{fn} of /root/reference/src/cpu_ref.cpp (g++ -O3)"
        else:
            t0 = time.perf_counter()
            y1 = (oracle.block_conv_f32(x1, w1, conv, nthreads=1) if args.blocked
                  else oracle.conv_f32(x1, w1, conv, nthreads=1))
            secs = time.perf_counter() - t0
            kind, what = "port", "oracle/qconv_oracle.c " + ("orc_block_conv_f32" if args.blocked else "orc_conv_f32")
        flops1 = 2.0 * y1.shape[1] * y1.shape[2] * k * r * s_ * (c // conv[6])
        line["cpu_baseline"] = {"value": round(flops1 / secs / 1e12, 6), "unit": "TFLOP/s", "cores": 1, "kind": kind,
                                "sample": f"1 of the {n} images of {suite[0][0]} ({flops1 / 1e9:.2f} GFLOP) in "
                                          f"{secs:.2f} s; {what}, 1 thread on {cpu_model()}"}
    print(json.dumps(line), flush=True)


# Thin layers for the non-MFMA fallback: the C = 3 stem (C5) and layers with few output channels
# (name, n, h, w, c, k, r, s, (pad_h, pad_w, stride_h, stride_w, dil_h, dil_w, groups), relu)
FALLBACK_SHAPES = [
    ("stem_c3_k64", 32, 224, 224, 3, 64, 7, 7, (3, 3, 2, 2, 1, 1, 1), True),
    ("stem_c3_k16", 32, 224, 224, 3, 16, 7, 7, (3, 3, 2, 2, 1, 1, 1), True),
    ("1x1_64to1", 32, 56, 56, 64, 1, 1, 1, (0, 0, 1, 1, 1, 1, 1), False),
    ("1x1_64to8", 32, 56, 56, 64, 8, 1, 1, (0, 0, 1, 1, 1, 1, 1), False),
    ("1x1_512to4", 32, 14, 14, 512, 4, 1, 1, (0, 0, 1, 1, 1, 1, 1), False),
    ("1x1_16to8", 32, 112, 112, 16, 8, 1, 1, (0, 0, 1, 1, 1, 1, 1), False),
    ("1x1_64to8_n1", 1, 56, 56, 64, 8, 1, 1, (0, 0, 1, 1, 1, 1, 1), False),
    ("3x3_16to8", 32, 112, 112, 16, 8, 3, 3, (1, 1, 1, 1, 1, 1, 1), True),
    ("3x3_64to8", 32, 56, 56, 64, 8, 3, 3, (1, 1, 1, 1, 1, 1, 1), True),
    ("1x1_64to12", 32, 56, 56, 64, 12, 1, 1, (0, 0, 1, 1, 1, 1, 1), False),
    ("1x1_64to16", 32, 56, 56, 64, 16, 1, 1, (0, 0, 1, 1, 1, 1, 1), False),
]


def bench_fallback(args) -> None:
    """Times every int8 kernel family that accepts each FALLBACK_SHAPES layer (graph replay of
    `steps` launches over rotating input/output sets), checks each family's output on image 0
    against the oracle bit for bit, prints a table on stderr and one JSON line; the rows show
    which family AUTO takes and what the others measured."""
    import numpy as np
    import torch

    import my_own_cnn_amd as M
    import oracle  # checker of image 0 only
    from my_own_cnn_amd import workloads as W

    dev = torch.device("cuda:0")
    families = ["dot4", "igemm", "stem", "band", "flat", "stream"]
    rows = []
    for name, n, h, w, c, k, r, s_, conv, relu in FALLBACK_SHAPES:
        if args.config not in (None, name):
            continue
        g = conv[6]
        kw = dict(padding=conv[:2], stride=conv[2:4], dilation=conv[4:6], groups=g)
        ho, wo = M.infer_conv_shape(n, h, w, c, r, s_, k, M.Conv2DParams(*conv))
        x0 = W.fill_i8_uniform(n * h * w * c, 31, -128, 127).reshape(n, h, w, c)
        wt = W.fill_i8_uniform(k * r * s_ * (c // g), 32, -127, 127).reshape(k, r, s_, c // g)
        bias = W.fill_i32_uniform(k, 33, -1024, 1024)
        wsc = W.fill_f32_uniform(k, 34, 1e-3, 1e-2)
        want = oracle.requant_i8(oracle.conv_i8_acc(x0[:1], wt, conv), bias, wsc, 0.02, 1.0, relu)
        set_bytes = x0.nbytes + n * ho * wo * k
        nsets = max(1, min(args.steps, POOL_BYTES // set_bytes))
        xpool = torch.empty((nsets,) + x0.shape, dtype=torch.int8, device=dev)
        xpool.copy_(torch.from_numpy(x0).to(dev).unsqueeze(0).expand_as(xpool))
        ypool = torch.empty((nsets, n, ho, wo, k), dtype=torch.int8, device=dev)
        wd, bd, sd = (torch.from_numpy(a).to(dev) for a in (wt, bias, wsc))
        auto = M.plan(M.make_desc(x0.shape, wt.shape, **kw))
        row = {"name": name, "n": n, "h": h, "w": w, "c": c, "k": k, "r": r, "s": s_, "stride": conv[2], "groups": g,
               "auto": auto, "us": {}, "verified": {}}
        for fam in families:
            try:
                M.plan(M.make_desc(x0.shape, wt.shape, algo=fam, **kw))
            except M.MiqError:
                continue  # this family does not take the shape

            def step(i, fam=fam):
                M.qconv2d_nhwc_i8(xpool[i % nsets], wd, bd, sd, relu=relu, in_scale=0.02, algo=fam,
                                  out=ypool[i % nsets], **kw)

            step(0)
            torch.cuda.synchronize()
            row["verified"][fam] = bool(np.array_equal(ypool[0, :1].cpu().numpy(), want))
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=side):
                for i in range(args.steps):
                    step(i)
            graph.replay()
            torch.cuda.synchronize()
            t0, t1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            gpu_hold(hold_us(args.steps, 3.0))
            t0.record()
            graph.replay()
            t1.record()
            torch.cuda.synchronize()
            row["us"][fam] = round(t0.elapsed_time(t1) * 1e3 / args.steps, 2)
            del graph
        rows.append(row)
        del xpool, ypool
        torch.cuda.empty_cache()
    if not rows:
        print(f"bench.py: unknown --fallback shape {args.config}; known: {[f[0] for f in FALLBACK_SHAPES]}",
              file=sys.stderr)
        sys.exit(2)
    print(f"{'shape':14s} {'auto':6s} " + " ".join(f"{f:>8s}" for f in families) + "  verified", file=sys.stderr)
    for r_ in rows:
        cells = " ".join(f"{r_['us'][f]:8.2f}" if f in r_["us"] else f"{'-':>8s}" for f in families)
        print(f"{r_['name']:14s} {r_['auto']:6s} {cells}  {all(r_['verified'].values())}", file=sys.stderr)
    head = rows[0]
    line = {
        "metric": "int8 us per launch by kernel family on thin layers (the vector-ALU fallback against the MFMA "
                  "kernels)",
        "value": head["us"][head["auto"]], "unit": "us", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": round(head["us"][head["auto"]] / 1e3, 6), "higher_is_better": False, "scaling": "weak",
        "vs_baseline": None, "dtype": "int8", "data": "synthetic",
        "config": {"workload": head["name"], "kernel": head["auto"], "timing": "hipgraph back-to-back",
                   "cache": "rotating sets"},
        "shapes": rows,
    }
    print(json.dumps(line), flush=True)


def bench_qi32(args) -> None:
    """Times the reference's own entry point, launch_fprop_nhwc_qi32<LinQuantU8>, on the workloads'
    shapes with uint8 float codes and per-sample zero points (int32 accumulators out); checks
    image 0 of each against the oracle bit for bit; prints a table on stderr and one JSON line.
    The API's floor is HBM: 4-byte codes in and int32 sums out (x + w + y bytes at 8 TB/s)."""
    import numpy as np
    import torch

    import my_own_cnn_amd as M
    import oracle  # checker of the sampled image only
    from my_own_cnn_amd import workloads as W

    dev = torch.device("cuda:0")
    rows = []
    # the workloads, then C2 with the reference's blocked-suite filter grids (main.cpp:177-178)
    cases = [(name, wl, (1, 1)) for name, wl in W.WORKLOADS.items()]
    cases += [("r50_3x3_b2x2", W.WORKLOADS["r50_3x3"], (2, 2)), ("r50_3x3_b4x4", W.WORKLOADS["r50_3x3"], (4, 4))]
    for name, wl, (by, bx) in cases:
        if args.config not in (None, name):
            continue
        gen = torch.Generator(device=dev)
        gen.manual_seed(7)
        x = torch.randint(0, 256, (wl.n, wl.h, wl.w, wl.c), device=dev, generator=gen).float()
        wshape = (wl.k, wl.r, wl.s, wl.c // wl.groups) if (by, bx) == (1, 1) else \
            (wl.k, by, bx, wl.r, wl.s, wl.c // wl.groups)
        w = torch.randint(0, 256, wshape, device=dev, generator=gen).float()
        zp = [int(v) for v in np.random.default_rng(5).integers(0, 256, size=wl.n)]
        arr = M.qparams_array(M.DataType.LinQuantU8, zp)
        in_qp = torch.from_numpy(np.frombuffer(arr.tobytes(), np.uint8).copy()).to(dev)
        farr = M.qparams_array(M.DataType.LinQuantU8, [131])
        f_qp = torch.from_numpy(np.frombuffer(farr.tobytes(), np.uint8).copy()).to(dev)
        y = torch.empty((wl.n, wl.ho, wl.wo, wl.k), dtype=torch.int32, device=dev)
        p = M.Conv2DParams(*wl.conv7)
        stream = torch.cuda.current_stream()

        bp = M.BlockConv2DParams(p, by, bx)

        def step():
            if (by, bx) == (1, 1):
                M.launch_fprop_nhwc_qi32(M.DataType.LinQuantU8, x, w, y, wl.n, wl.h, wl.w, wl.c, wl.r, wl.s, wl.k, p,
                                         in_qp, f_qp, stream=stream)
            else:
                M.launch_block_fprop_nhwc_qi32(M.DataType.LinQuantU8, x, w, y, wl.n, wl.h, wl.w, wl.c, wl.r, wl.s,
                                               wl.k, bp, in_qp, f_qp, stream=stream)

        step()
        torch.cuda.synchronize()
        want = oracle.conv_qi32(x[:1].cpu().numpy(), w.cpu().numpy(), wl.conv7, zp[:1], 131,
                                (0, 0) if (by, bx) == (1, 1) else (by, bx))
        ok = bool(np.array_equal(y[:1].cpu().numpy(), want))
        for _ in range(args.warmup):
            step()
        t0, t1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        torch.cuda.synchronize()
        gpu_hold(hold_us(args.steps, 25.0))
        t0.record(stream)
        for _ in range(args.steps):
            step()
        t1.record(stream)
        torch.cuda.synchronize()
        ms = t0.elapsed_time(t1) / args.steps
        tops = wl.ops / (ms * 1e-3) / 1e12
        nbytes = 4.0 * (x.numel() + w.numel() + y.numel())
        if (by, bx) == (1, 1):
            kern = M.plan_qi32(wl.n, wl.h, wl.w, wl.c, wl.r, wl.s, wl.k, p)
        else:
            kern = M.plan_block_qi32(wl.n, wl.h, wl.w, wl.c, wl.r, wl.s, wl.k, bp)
        if kern == "igemm" and (wl.c // wl.groups) % 4 != 0:
            kern = "igemm-scalar"
        gbs = nbytes / (ms * 1e-3) / 1e9
        rows.append(dict(name=name, kernel=kern, us=round(ms * 1e3, 2), int32_tops=round(tops, 2),
                         gbs=round(gbs, 1), frac_hbm=round(gbs / PEAK_HBM_GBS, 4),
                         hbm_floor_us=round(nbytes / (PEAK_HBM_GBS * 1e9) * 1e6, 2), verified_image0=ok))
        del x, w, y
        torch.cuda.empty_cache()
    print(f"{'config':13s} {'kernel':12s} {'us':>9s} {'floor us':>9s} {'TOPS':>8s} {'GB/s':>8s} {'hbm':>6s} exact",
          file=sys.stderr)
    for r in rows:
        print(f"{r['name']:13s} {r['kernel']:12s} {r['us']:9.2f} {r['hbm_floor_us']:9.2f} {r['int32_tops']:8.2f} "
              f"{r['gbs']:8.1f} {r['frac_hbm']:6.3f} {r['verified_image0']}", file=sys.stderr)
    head = next((r for r in rows if r["name"] == "r50_3x3"), rows[0])
    print(json.dumps({
        "metric": "float-code qi32 conv TOPS (launch_fprop_nhwc_qi32<LinQuantU8>, int32 accumulators)",
        "value": head["int32_tops"], "unit": "TOPS", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": round(head["us"] / 1e3, 6), "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
        "dtype": "int32", "data": "synthetic",
        "config": {"workload": head["name"], "kernel": head["kernel"], "timing": "eager back-to-back", "cache": "warm"},
        "roofline": {"bound": "hbm", "achieved": head["gbs"], "peak": PEAK_HBM_GBS, "unit": "GB/s",
                     "frac": head["frac_hbm"], "traffic": None},
        "shapes": rows}), flush=True)


def cpu_model() -> str:
    try:
        for ln in open("/proc/cpuinfo"):
            if ln.startswith("model name"):
                return ln.split(":", 1)[1].strip()
    except OSError:
        pass
    return platform.processor() or "unknown"


def cpu_baseline(wl):
    """The reference CPU path on the full workload, one thread."""
    import numpy as np
    import oracle  # cpu_baseline leg: the oracle is the checker / baseline, never the measured path

    inp = wl.inputs()
    x = inp["x"].astype(np.float32)
    w = inp["w"].astype(np.float32)
    zp = np.zeros(wl.n, np.int32)
    if oracle.ref() is not None:
        _, secs = oracle.ref_conv_qi32("s5", x, w, wl.conv7, zp, 0)
        kind, what = "reference", "cpu_fprop_nhwc_qi32 of /root/reference/src/cpu_ref.cpp (g++ -O3), float codes"
    else:
        t0 = time.perf_counter()
        oracle.conv_i8_acc(inp["x"], inp["w"], wl.conv7, nthreads=1)
        secs = time.perf_counter() - t0
        kind, what = "port", "oracle/qconv_oracle.c restatement of cpu_ref.cpp (gcc -O3), int8 codes"
    return {
        "value": round(wl.ops / secs / 1e12, 6),
        "unit": "TOPS",
        "cores": 1,
        "kind": kind,
        "sample": f"full {wl.name} batch (N={wl.n}, {wl.ops / 1e9:.2f} Gop int32 accumulation) in {secs:.2f} s; "
                  f"{what}; 1 thread on {cpu_model()}",
        "workload": wl.name,
    }


def main():
    args = parse()
    if args.copy_mb:
        copy_calibration(args.copy_mb)
        return
    if args.gpus != 1:
        print(f"bench.py: this build measures one GPU only (asked for --gpus {args.gpus}); "
              "the convolution shards on the batch dimension with no exchange; that split is designed, not benchmarked", file=sys.stderr)
        sys.exit(2)

    import numpy as np
    import torch

    import my_own_cnn_amd as M
    from my_own_cnn_amd import workloads as W

    if not torch.cuda.is_available():
        print("bench.py: no GPU visible", file=sys.stderr)
        sys.exit(1)
    if args.bmm:
        bench_bmm(args)
        return
    if args.fp32:
        bench_fp32(args)
        return
    if args.qi32:
        bench_qi32(args)
        return
    if args.fallback:
        bench_fallback(args)
        return
    dev = torch.device("cuda:0")
    # every BASELINE config by default (the headline first: its line is `value`); --config
    # times one
    names = [args.config] if args.config else [W.HEADLINE] + [n for n in W.WORKLOADS if n != W.HEADLINE]
    flush = torch.empty((FLUSH_BYTES // 4,), dtype=torch.float32, device=dev).fill_(1.0)

    def flush_caches():
        # a read of 2x the Infinity Cache (MALL) and every L2: evicts earlier steps' data and
        # leaves no dirty lines behind, so nothing is written back during the timed region
        torch.sum(flush)
        torch.cuda.synchronize()

    results = {}
    for name in names:
        wl = W.WORKLOADS[name]
        inp = wl.inputs()
        w = torch.from_numpy(inp["w"]).to(dev)
        bias = torch.from_numpy(inp["bias"]).to(dev)
        ws = torch.from_numpy(inp["w_scale"]).to(dev)
        set_bytes = wl.x_bytes + wl.y_bytes
        # cold: one pooled buffer of input/output sets, one per timed step up to POOL_BYTES
        # (then reused in rotation, POOL_BYTES >> MALL apart), filled by one copy kernel; every
        # timed step reads a set that nothing has touched since the flush before the timed region
        nsets = 1 if args.cache == "warm" else max(1, min(args.steps, POOL_BYTES // set_bytes))
        x0 = torch.from_numpy(inp["x"]).to(dev)
        xpool = torch.empty((nsets,) + tuple(x0.shape), dtype=torch.int8, device=dev)
        xpool.copy_(x0.unsqueeze(0).expand_as(xpool))
        ypool = torch.empty((nsets, wl.n, wl.ho, wl.wo, wl.k), dtype=torch.int8, device=dev)
        kw = dict(stride=wl.stride, padding=wl.pad, relu=wl.relu, in_scale=wl.in_scale, out_scale=wl.out_scale,
                  algo=args.algo)
        algo = M.plan(M.make_desc(x0.shape, w.shape, stride=wl.stride, padding=wl.pad, algo=args.algo))

        def step(i, stream=None):
            M.qconv2d_nhwc_i8(xpool[i % nsets], w, bias, ws, out=ypool[i % nsets], stream=stream, **kw)

        # correctness gate before timing: the int8 output of set 0 against the oracle's epilogue
        import oracle
        step(0)
        torch.cuda.synchronize()
        acc = oracle.conv_i8_acc(inp["x"], inp["w"], wl.conv7)
        want = oracle.requant_i8(acc, inp["bias"], inp["w_scale"], wl.in_scale, wl.out_scale, wl.relu)
        verified = bool(np.array_equal(ypool[0].cpu().numpy(), want))

        for i in range(args.warmup):
            step(i)
        torch.cuda.synchronize()

        mode = "eager"
        stream = torch.cuda.current_stream()
        graph = None
        if not args.eager:
            try:
                side = torch.cuda.Stream()
                side.wait_stream(stream)
                graph = torch.cuda.CUDAGraph()
                with torch.cuda.graph(graph, stream=side):
                    for i in range(args.steps):
                        step(i)
                torch.cuda.synchronize()
                graph.replay()  # untimed replay: first-replay setup cost stays out of the timed region
                torch.cuda.synchronize()
                mode = "hipgraph"
            except Exception as exc:  # noqa: BLE001 - fall back to eager timing, say so
                print(f"bench.py: graph capture unavailable ({exc}); timing eager launches", file=sys.stderr)
                graph = None

        t0, t1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        if args.cache == "cold":
            flush_caches()
        torch.cuda.synchronize()
        wall0 = time.perf_counter()
        gpu_hold(hold_us(args.steps, 3.0 if graph is not None else 25.0))
        t0.record(stream)
        if graph is not None:
            graph.replay()
        else:
            for i in range(args.steps):
                step(i)
        t1.record(stream)
        torch.cuda.synchronize()
        wall = time.perf_counter() - wall0
        ms = t0.elapsed_time(t1) / args.steps
        tops = wl.ops / (ms * 1e-3) / 1e12
        gbs = wl.bytes / (ms * 1e-3) / 1e9
        # reference-style per-launch timing (src/bench.cpp:27-43): one event pair around each of
        # up to 200 eager launches, median and the floor(0.9 * (n - 1))-th sample; reported
        # beside the back-to-back figure, never as `value`
        nper = min(args.steps, 200)
        evs = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)) for _ in range(nper)]
        if args.cache == "cold":
            flush_caches()
        for i, (ea, eb) in enumerate(evs):
            ea.record(stream)
            step(i)
            eb.record(stream)
        torch.cuda.synchronize()
        per = sorted(ea.elapsed_time(eb) for ea, eb in evs)
        per_launch = {"median_us": round(per[len(per) // 2] * 1e3, 3),
                      "p90_us": round(per[int(0.9 * (len(per) - 1))] * 1e3, 3), "launches": nper,
                      "timing": "eager, one event pair per launch"}
        t_mfma = wl.ops / (PEAK_INT8_TOPS * 1e12)
        t_hbm = wl.bytes / (PEAK_HBM_GBS * 1e9)
        bound = "mfma" if t_mfma >= t_hbm else "hbm"
        touched = min(args.steps, nsets) * set_bytes
        cache = "warm" if args.cache == "warm" else "cold"
        results[name] = dict(ms=ms, tops=tops, gbs=gbs, bound=bound, verified=verified, algo=algo, mode=mode,
                             nsets=nsets, touched=touched, cache=cache, wall=wall, wl=wl, per_launch=per_launch)
        del xpool, ypool, graph
        torch.cuda.empty_cache()

    head = results[names[0]]
    wl = head["wl"]
    if head["bound"] == "hbm":
        roof = {"bound": "hbm", "achieved": round(head["gbs"], 2), "peak": PEAK_HBM_GBS, "unit": "GB/s",
                "frac": round(head["gbs"] / PEAK_HBM_GBS, 4)}
    else:
        roof = {"bound": "mfma", "achieved": round(head["tops"], 2), "peak": PEAK_INT8_TOPS, "unit": "TFLOP/s",
                "frac": round(head["tops"] / PEAK_INT8_TOPS, 4)}
    roof["traffic"] = None
    traffic_file = ROOT / "profiles" / f"traffic_{wl.name}.json"
    if traffic_file.exists():
        try:
            roof["traffic"] = json.loads(traffic_file.read_text()).get("bytes_per_launch")
        except (ValueError, OSError):
            pass

    line = {
        "metric": METRIC,
        "value": round(head["tops"], 3),
        "unit": "TOPS",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(head["ms"], 6),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "int8",
        "data": "synthetic",
        "config": {
            "workload": wl.name, "N": wl.n, "H": wl.h, "W": wl.w, "C": wl.c, "K": wl.k, "R": wl.r, "S": wl.s,
            "stride": wl.stride, "pad": wl.pad, "relu": wl.relu, "epilogue": "bias+requant+int8 saturate",
            "kernel": head["algo"], "cache": head["cache"], "buffer_sets": head["nsets"],
            "bytes_touched": head["touched"], "timing": head["mode"],
        },
        "mfma_peak_frac": round(head["tops"] / PEAK_INT8_TOPS, 4),
        "gbs": round(head["gbs"], 2),
        "verified_bit_exact": head["verified"],
        "roofline": roof,
        "per_launch": head["per_launch"],
    }
    # every config measured in this run (BASELINE.json configs[0..4]), same timing and cache
    # rules as the headline; `value` stays the headline's
    per_cfg = {}
    for name, r in results.items():
        frac = r["tops"] / PEAK_INT8_TOPS if r["bound"] == "mfma" else r["gbs"] / PEAK_HBM_GBS
        traffic = None
        tf = ROOT / "profiles" / f"traffic_{name}.json"
        if tf.exists():
            try:
                traffic = json.loads(tf.read_text()).get("bytes_per_launch")
            except (ValueError, OSError):
                traffic = None
        per_cfg[name] = {"us": round(r["ms"] * 1e3, 3), "tops": round(r["tops"], 2), "gbs": round(r["gbs"], 1),
                         "bound": r["bound"], "frac": round(frac, 4), "mfma_peak_frac": round(r["tops"] / PEAK_INT8_TOPS, 4),
                         "kernel": r["algo"], "verified_bit_exact": r["verified"], "cache": r["cache"],
                         "bytes_touched": r["touched"], "traffic": traffic,
                         "median_us": r["per_launch"]["median_us"], "p90_us": r["per_launch"]["p90_us"]}
    line["configs"] = per_cfg
    if not args.no_cpu_baseline:
        line["cpu_baseline"] = cpu_baseline(wl)
    print(f"{'config':10s} {'kernel':7s} {'us':>9s} {'TOPS':>8s} {'GB/s':>8s} {'bound':5s} {'frac':>6s} exact"
          f" {'med us':>7s} {'p90 us':>7s}", file=sys.stderr)
    for name, r in per_cfg.items():
        print(f"{name:10s} {r['kernel']:7s} {r['us']:9.2f} {r['tops']:8.1f} {r['gbs']:8.1f} {r['bound']:5s} "
              f"{r['frac']:6.3f} {str(r['verified_bit_exact']):5s} {r['median_us']:7.2f} {r['p90_us']:7.2f}",
              file=sys.stderr)
    print(json.dumps(line), flush=True)
    os.sys.stdout.flush()


if __name__ == "__main__":
    main()
