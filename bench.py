#!/usr/bin/env python3
"""Benchmark of the QloraLinear hot path on one MI355X.

Metric: "QloraLinear fwd+bwd TFLOP/s (prefill) & weight GB/s
(decode), % of roofline".  The headline line is configuration 2 (decode):
one step is the fused dequant-GEMV forward of the two Llama-7B MLP shapes
(NF4 11008x4096 then 4096x11008, LoRA r=16 alpha=32) at batch 1; ``value``
is packed-weight bytes per second.  The same line carries decode at batch 4
and 16 and configuration 3 (prefill: fused forward+backward of a 4096x4096
NF4 layer at 4096 tokens, r=64 alpha=16, fp32 and bf16 activations) in
TFLOP/s.

Inputs are synthetic (torch's seeded generator on the GPU: W ~ 0.02 N(0,1)
quantized on the GPU, A ~ U(+-1/sqrt(K)), B ~ 0.01 N(0,1), X, dY ~ N(0,1))
and resident in HBM before timing.  Decode steps rotate over enough weight
copies (>= 512 MB) that every step reads HBM rather than the 256 MB
Infinity Cache, and run as a replayed HIP graph so that host launch cost is
not measured.  ``cpu_baseline`` times the oracle (the C restatement of
qlora-core's single-threaded CPU path) on a bounded sample on this host.
"""
from __future__ import annotations

import argparse
import json
import math
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(ROOT, "vkqlora.rs_amd"))

HBM_PEAK_GBS = 8000.0
FP32_MFMA_PEAK_TFLOPS = 157.3
BF16_MFMA_PEAK_TFLOPS = 2500.0
METRIC = ("QloraLinear fwd+bwd TFLOP/s (prefill) & weight GB/s (decode), "
          "% of roofline")


def parse():
    ap = argparse.ArgumentParser(description=__doc__.split("\n")[0])
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=200,
                    help="timed decode steps (prefill uses steps/20, >= 5)")
    ap.add_argument("--warmup", type=int, default=20)
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--skip-prefill", action="store_true")
    ap.add_argument("--skip-extra", action="store_true",
                    help="skip configurations 1, 4, 5 and C3's 14336x4096 layer")
    ap.add_argument("--skip-glue", action="store_true",
                    help="skip the RMSNorm / SwiGLU / cross-entropy measurements")
    ap.add_argument("--cpu-seconds", type=float, default=10.0,
                    help="CPU-baseline budget per workload")
    ap.add_argument("--probe", choices=("decode", "prefill", "hbm"), default=None,
                    help="counter probe for rocprofv3 --pmc (prints no JSON line): a few "
                         "eager launches of one workload's kernels (decode: the C2 two-layer "
                         "step at batch 1, 4 and 16; prefill: C3 fwd+bwd, fp32 and bf16; hbm: the "
                         "C5 Adam step, quantize and the 70B-class cross-entropy), then a "
                         "256 MiB device copy (the HBM-traffic calibration)")
    ap.add_argument("--phases", default="decode,prefill,extra,glue,load,mlp",
                    help="comma list of the measurements to run (for per-phase profiles); "
                         "the JSON line always needs decode")
    return ap.parse_args()


def probe(kind, ctx, torch, dev, QD):
    """Kernels for the counter runs, then a plain 256 MiB copy."""
    g = torch.Generator(device="cuda").manual_seed(0x1234)
    if kind == "decode":
        # the C2 step at batch 1, 4 and 16: both layers in one call (one
        # launch at batch 1; a T1 launch and one split launch at 4 and 16),
        # five weight copies
        r, alpha = 16, 32.0
        layers = []
        for N, K in [(11008, 4096), (4096, 11008)]:
            w = torch.randn(N, K, device=dev, generator=g) * 0.02
            base = QD.DeviceWeight.quantize(w, 64, True, ctx=ctx)
            del w
            a = (torch.rand(r, K, device=dev, generator=g) * 2 - 1) / math.sqrt(K)
            b = torch.randn(N, r, device=dev, generator=g) * 0.01
            layers.append(dict(copies=[base.clone() for _ in range(5)], a=a, b=b,
                               lora=QD.lora_struct(a, b, r, alpha), N=N, K=K))
        for batch in (1, 4, 16):
            for L in layers:
                L["x"] = torch.randn(batch, L["K"], device=dev, generator=g)
                L["y"] = torch.empty(batch, L["N"], device=dev)
            for i in range(5):
                QD.forward_group([(L["copies"][i], L["lora"], L["x"], L["y"], None)
                                  for L in layers], batch, ctx=ctx)
            torch.cuda.synchronize()
        del layers
    elif kind == "prefill":
        for act in (torch.float32, torch.bfloat16):
            L = _layer(torch, dev, QD, ctx, g, 4096, 4096, 4096, 64, 16.0, act=act)
            for _ in range(2):
                _fwd_bwd(QD, ctx, L)
            torch.cuda.synchronize()
            del L
    else:
        # C5 Adam step (four r=64 adapter tensors), C5 quantize, 70B-class CE
        import ctypes as C
        import qlora_hip as QH
        r = 64
        tens = []
        for N, K in ((28672, 8192), (8192, 28672)):
            tens += [(torch.randn(r * K, device=dev, generator=g),
                      torch.randn(r * K, device=dev, generator=g) * 0.01),
                     (torch.randn(N * r, device=dev, generator=g),
                      torch.randn(N * r, device=dev, generator=g) * 0.01)]
        opt = QH.Adam8bit(lr=1e-3, ctx=ctx)
        cnt = len(tens)
        pp = (C.c_void_p * cnt)(*[p.data_ptr() for p, _ in tens])
        gp = (C.c_void_p * cnt)(*[g_.data_ptr() for _, g_ in tens])
        ll = (C.c_size_t * cnt)(*[p.numel() for p, _ in tens])
        st = QH._lib.AdamStats()
        for _ in range(3):
            QH._lib.check(ctx.lib.qh_adam8bit_step_dev(opt.h, pp, gp, ll, cnt, C.byref(st),
                                                       None))
        w = torch.randn(28672, 8192, device=dev, generator=g) * 0.02
        for _ in range(2):
            QD.DeviceWeight.quantize(w, 64, True, ctx=ctx)
        del w
        logits = torch.randn(2048, 128256, device=dev, generator=g)
        targets = torch.randint(0, 128256, (2048,), device=dev, dtype=torch.int32,
                                generator=g)
        for _ in range(2):
            QD.softmax_cross_entropy(logits, targets, ctx=ctx)
        torch.cuda.synchronize()
        del logits
    torch.cuda.empty_cache()
    src = torch.empty(64 << 20, device=dev)  # 256 MiB of fp32
    dst = torch.empty_like(src)
    for _ in range(3):
        dst.copy_(src)
    torch.cuda.synchronize()
    print("# probe done", file=sys.stderr, flush=True)


def profile_value(name, key):
    """A figure from a committed counter summary under profiles/ (a line
    `key: value`, e.g. the HBM bytes per launch from FETCH_SIZE + WRITE_SIZE
    scaled by the same counters on a copy of known size), or None when the
    summary or the line is absent."""
    try:
        with open(os.path.join(ROOT, "profiles", name)) as f:
            for line in f:
                if line.startswith(key + ":"):
                    return float(line.split(":", 1)[1])
    except OSError:
        pass
    return None


def measured_traffic():
    """HBM bytes per batch-1 decode launch (profiles/decode_c2_traffic.md)."""
    return profile_value("decode_c2_traffic.md", "traffic_bytes_per_launch")


# ---------------------------------------------------------------------------
def hbm_copy_peak(torch, dev, nbytes=1 << 30, reps=10):
    """Measured HBM peak: a device-to-device copy of 1 GiB (read + written
    bytes per second), the STREAM-like reference the decode fraction is also
    quoted against."""
    a = torch.empty(nbytes // 4, dtype=torch.float32, device=dev).fill_(1.0)
    b = torch.empty_like(a)
    b.copy_(a)
    torch.cuda.synchronize()
    e0 = torch.cuda.Event(enable_timing=True)
    e1 = torch.cuda.Event(enable_timing=True)
    e0.record()
    for _ in range(reps):
        b.copy_(a)
    e1.record()
    torch.cuda.synchronize()
    ms = e0.elapsed_time(e1) / reps
    del a, b
    return dict(gbs=2 * nbytes / (ms * 1e6), bytes=2 * nbytes, ms=ms,
                kernel="torch copy_ of 1 GiB (read + write)")


def read_ceiling(torch, dev, sizes=(24 << 20, 48 << 20, 1 << 30)):
    """What ONE launch of a plain streaming read reaches at a given size:
    libqh_probe.so's qh_probe_read (16-byte loads, a contiguous slice per
    workgroup), best over a small sweep of grid, block, unroll and
    non-temporal loads, timed as graph replays over enough distinct buffers
    (>= 600 MiB) that no launch finds its bytes in the 256 MiB MALL. Returns
    {MiB: {gbs, us, groups, threads, unroll, nt}}, or None when the probe
    library is not built."""
    import ctypes as C
    path = os.path.join(ROOT, "vkqlora.rs_amd", "qlora_hip", "libqh_probe.so")
    if not os.path.exists(path):
        return None
    P = C.CDLL(path)
    P.qh_probe_read.argtypes = [C.c_void_p, C.c_size_t, C.c_void_p, C.c_int, C.c_int,
                                C.c_int, C.c_int, C.c_void_p]
    P.qh_probe_read.restype = C.c_int
    sink = torch.empty(1 << 13, dtype=torch.int32, device=dev)
    out = {}
    for nbytes in sizes:
        copies = max(1, -(-(600 << 20) // nbytes))
        bufs = [torch.full((nbytes // 4,), i + 1, dtype=torch.int32, device=dev)
                for i in range(copies)]
        best = None
        for groups in (512, 1024, 2048):
            for threads in (512, 1024):
                for unroll in (4, 8):
                    for nt in (0, 1):
                        def launch(b, groups=groups, threads=threads, unroll=unroll, nt=nt):
                            rc = P.qh_probe_read(
                                b.data_ptr(), nbytes, sink.data_ptr(), groups, threads,
                                unroll, nt, torch.cuda.current_stream().cuda_stream)
                            if rc != 0:
                                raise RuntimeError(f"qh_probe_read: HIP error {rc}")
                        s = torch.cuda.Stream()
                        s.wait_stream(torch.cuda.current_stream())
                        with torch.cuda.stream(s):
                            for b in bufs:
                                launch(b)
                        torch.cuda.current_stream().wait_stream(s)
                        torch.cuda.synchronize()
                        gr = torch.cuda.CUDAGraph()
                        with torch.cuda.graph(gr):
                            for b in bufs:
                                launch(b)
                        gr.replay()
                        torch.cuda.synchronize()
                        reps = max(3, 48 // copies)
                        e0 = torch.cuda.Event(enable_timing=True)
                        e1 = torch.cuda.Event(enable_timing=True)
                        e0.record()
                        for _ in range(reps):
                            gr.replay()
                        e1.record()
                        torch.cuda.synchronize()
                        ms = e0.elapsed_time(e1) / (reps * copies)
                        del gr
                        gbs = nbytes / (ms * 1e6)
                        if best is None or gbs > best["gbs"]:
                            best = dict(gbs=gbs, us=ms * 1e3, groups=groups,
                                        threads=threads, unroll=unroll, nt=nt)
        out[str(nbytes >> 20)] = best
        del bufs
        torch.cuda.empty_cache()
    return out


# ---------------------------------------------------------------------------
def decode_bench(args, ctx, torch, dev, QD):
    """Config 2: decode-shaped fused dequant-GEMV forward."""
    r, alpha = 16, 32.0
    shapes = [(11008, 4096), (4096, 11008)]  # (out_dim N, in_dim K)
    g = torch.Generator(device="cuda").manual_seed(0x1234)
    layers = []
    for N, K in shapes:
        w = torch.randn(N, K, device=dev, generator=g) * 0.02
        base = QD.DeviceWeight.quantize(w, 64, True, ctx=ctx)
        del w
        bound = 1.0 / math.sqrt(K)
        a = (torch.rand(r, K, device=dev, generator=g) * 2 - 1) * bound
        b = torch.randn(N, r, device=dev, generator=g) * 0.01
        layers.append(dict(N=N, K=K, base=base, a=a, b=b,
                           lora=QD.lora_struct(a, b, r, alpha)))
    wbytes = sum(L["base"].nbytes for L in layers)
    copies = max(2, math.ceil(512e6 / wbytes))
    for L in layers:
        L["copies"] = [L["base"]] + [L["base"].clone() for _ in range(copies - 1)]
        L["structs"] = [c.struct() for c in L["copies"]]
    torch.cuda.synchronize()

    results = {}
    for batch in (1, 4, 16):
        xs = [torch.randn(batch, L["K"], device=dev, generator=g) for L in layers]
        ys = [torch.empty(batch, L["N"], device=dev) for L in layers]

        def step(i):
            # both layers in one call: at batch 1 they share one launch
            QD.forward_group([(L["structs"][(i * len(layers) + li) % copies], L["lora"],
                               xs[li], ys[li], None) for li, L in enumerate(layers)],
                             batch, ctx=ctx)

        n_graph = copies  # one graph covers every weight copy once

        def capture(nsteps):
            gr = torch.cuda.CUDAGraph()
            s = torch.cuda.Stream()
            s.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(s):
                step(0)  # warm-up on the capture stream
            torch.cuda.current_stream().wait_stream(s)
            torch.cuda.synchronize()
            with torch.cuda.graph(gr):
                for i in range(nsteps):
                    step(i)
            return gr

        # eager reference result (also sizes the library's scratch)
        step(0)
        torch.cuda.synchronize()
        ref = [y.clone() for y in ys]
        graph = capture(n_graph)
        # the graph must reproduce the eager result on every replay
        for _ in range(2):
            graph.replay()
            torch.cuda.synchronize()
            for y, rr in zip(ys, ref):
                assert torch.equal(y, rr), "graph replay differs from eager run"
        # exactly args.steps timed steps: whole passes over the weight
        # copies, then a graph of the remaining steps
        reps, rem = divmod(max(args.steps, 1), n_graph)
        tail = capture(rem) if rem else None
        nsteps = reps * n_graph + rem
        for _ in range(max(1, -(-args.warmup // n_graph))):
            graph.replay()
        torch.cuda.synchronize()
        e0 = torch.cuda.Event(enable_timing=True)
        e1 = torch.cuda.Event(enable_timing=True)
        t0 = time.perf_counter()
        e0.record()
        for _ in range(reps):
            graph.replay()
        if tail is not None:
            tail.replay()
        e1.record()
        torch.cuda.synchronize()
        wall_step = (time.perf_counter() - t0) / nsteps * 1e3
        ms_step = e0.elapsed_time(e1) / nsteps

        # Per-kernel durations: with timing on, the library launches each
        # hot-path kernel with start/stop events that the GPU stamps at that
        # kernel's own start and end (hipExtLaunchKernelGGL), so the eager
        # launches here time the kernels alone, without host gaps.
        ctx.set_timing(True)
        for i in range(n_graph):  # warm-up pass, not kept
            step(i)
        torch.cuda.synchronize()
        ctx.timing_report(reset=True)
        for _ in range(4):  # kept: 4 passes over every weight copy
            for i in range(n_graph):
                step(i)
        torch.cuda.synchronize()
        rep = ctx.timing_report(reset=True)
        ctx.set_timing(False)
        kern = {k: dict(launches=v[0], avg_ms=v[1] / max(v[0], 1))
                for k, v in rep.items()}
        gemv_bytes = sum(L["base"].nbytes + 4 * batch * (L["K"] + L["N"])
                         + 4 * L["b"].numel() for L in layers)
        full_bytes = gemv_bytes + sum(4 * L["a"].numel() for L in layers)
        flops = sum(2 * batch * L["N"] * L["K"] + 2 * batch * r * (L["N"] + L["K"])
                    for L in layers)
        main_name = next((k for k in ("decode_stream2", "decode_stream", "decode_split",
                                      "gemv", "forward_gemm") if k in kern), None)
        main = kern.get(main_name) if main_name else None
        res = dict(
            ms_per_step=ms_step, wall_ms_per_step=wall_step,
            weight_gbs=wbytes / (ms_step * 1e6),
            total_gbs=full_bytes / (ms_step * 1e6),
            tflops=flops / (ms_step * 1e9),
            kernels=kern, steps=nsteps)
        if main:
            # the one-launch kernels also read LoRA A (their T1 producers);
            # the two-kernel paths read it in their T1 kernel
            per_step = main["launches"] / (4 * n_graph)
            # bytes one launch reads: both layers for a two-layer launch
            # (batch 1-2 side by side, or a pair on the split kernel), one
            # layer otherwise
            per_launch_layers = (len(layers) / per_step
                                 if main_name in ("decode_stream2", "decode_split") else 1)
            kb = ((full_bytes if main_name.startswith("decode_stream") else gemv_bytes)
                  * per_launch_layers / len(layers))
            kms = main["avg_ms"]
            if set(kern) == {main_name}:
                # the step is nothing but these launches: their duration in
                # the replayed graph (back to back, as the step runs; the
                # gap to the next launch included) is the step time over
                # the launches.  The eager launches above start on an idle
                # GPU between host calls and vary by +-5 % run to run.
                kms = ms_step / per_step
            res.update(main_kernel=main_name, main_kernel_ms=kms,
                       main_kernel_eager_ms=main["avg_ms"], main_kernel_bytes=kb,
                       main_kernel_gbs=kb / (kms * 1e6))
        # each layer alone (one call per layer: its own launch), beside the
        # two-layer step above; kernel durations from the timing events
        per_layer = {}
        for li, L in enumerate(layers):
            def one(i, li=li, L=L):
                QD.forward_group([(L["structs"][i % copies], L["lora"], xs[li], ys[li], None)],
                                 batch, ctx=ctx)
            ctx.set_timing(True)
            for i in range(copies):
                one(i)
            torch.cuda.synchronize()
            ctx.timing_report(reset=True)
            for _ in range(4):
                for i in range(copies):
                    one(i)
            torch.cuda.synchronize()
            rl = ctx.timing_report(reset=True)
            ctx.set_timing(False)
            lk = {k: dict(launches=v[0], avg_us=1e3 * v[1] / max(v[0], 1)) for k, v in rl.items()}
            lbytes = (L["base"].nbytes + 4 * batch * (L["K"] + L["N"]) + 4 * L["b"].numel()
                      + 4 * L["a"].numel())
            lus = sum(v["avg_us"] for v in lk.values())
            per_layer[f'{L["N"]}x{L["K"]}'] = dict(
                kernels=lk, kernel_us=lus, bytes=lbytes, gbs=lbytes / (lus * 1e3),
                frac_hbm=lbytes / (lus * 1e3) / 8000.0)
        res["per_layer"] = per_layer
        results[batch] = res
    return results, dict(copies=copies, packed_weight_bytes=wbytes, r=r,
                         alpha=alpha, host_path=host_path_bench(ctx, torch, layers, r, alpha))


def host_path_bench(ctx, torch, layers, r, alpha, reps=5):
    """The host-slice entry point (qh_qlora_forward, the reference's
    gpu_qlora_forward signature): host buffers in and out, so every call
    moves W, X, the adapters and Y over PCIe.  Reported beside the
    device-resident figure, never as it."""
    import numpy as np
    from qlora_hip import api
    rng = np.random.default_rng(0x5EED)
    host = []
    for L in layers:
        b0 = L["base"]
        q = dict(rows=b0.rows, cols=b0.cols, block_size=b0.block_size, n=b0.n,
                 codes=b0.codes.cpu().numpy(), scale_codes=b0.scale_codes.cpu().numpy(),
                 absmax=b0.absmax.cpu().numpy())
        host.append((q, L["a"].cpu().numpy().ravel(), L["b"].cpu().numpy().ravel(),
                     rng.standard_normal(L["K"]).astype(np.float32)))
    for q, a, b, x in host:  # warm-up (staging buffers)
        api.forward(q, a, b, r, alpha, x, 1, ctx=ctx)
    t0 = time.perf_counter()
    for _ in range(reps):
        for q, a, b, x in host:
            api.forward(q, a, b, r, alpha, x, 1, ctx=ctx)
    ms = (time.perf_counter() - t0) / reps * 1e3
    wbytes = sum(L["base"].nbytes for L in layers)
    return dict(ms_per_step=ms, weight_gbs=wbytes / (ms * 1e6), reps=reps,
                note="batch 1, both C2 layers through qh_qlora_forward with host "
                     "buffers: PCIe transfers included")


# ---------------------------------------------------------------------------
def prefill_bench(args, ctx, torch, dev, QD, act_dtype):
    """Config 3: fused forward + backward, 4096x4096 NF4, 4096 tokens."""
    N = K = 4096
    M, r, alpha = 4096, 64, 16.0
    g = torch.Generator(device="cuda").manual_seed(0x5678)
    w = torch.randn(N, K, device=dev, generator=g) * 0.02
    W = QD.DeviceWeight.quantize(w, 64, True, ctx=ctx)
    del w
    bound = 1.0 / math.sqrt(K)
    a = (torch.rand(r, K, device=dev, generator=g) * 2 - 1) * bound
    b = torch.randn(N, r, device=dev, generator=g) * 0.01
    lora = QD.lora_struct(a, b, r, alpha)
    x = torch.randn(M, K, device=dev, generator=g).to(act_dtype)
    dy = torch.randn(M, N, device=dev, generator=g).to(act_dtype)
    y = torch.empty(M, N, device=dev)
    t1 = torch.empty(M, r, device=dev)
    gx = torch.empty(M, K, device=dev)
    ga = torch.empty(r, K, device=dev)
    gb = torch.empty(N, r, device=dev)
    qw = W.struct()

    def step():
        QD.forward(None, lora, x, M, y, t1=t1, ctx=ctx, qw=qw)
        QD.backward(None, lora, x, dy, M, gx, ga, gb, t1=t1, ctx=ctx, qw=qw)

    steps = max(5, args.steps // 20)
    for _ in range(max(2, args.warmup // 10)):
        step()
    torch.cuda.synchronize()
    ctx.set_timing(True)
    ctx.timing_report(reset=True)
    e0 = torch.cuda.Event(enable_timing=True)
    e1 = torch.cuda.Event(enable_timing=True)
    e0.record()
    for _ in range(steps):
        step()
    e1.record()
    torch.cuda.synchronize()
    ms = e0.elapsed_time(e1) / steps
    rep = ctx.timing_report(reset=True)
    ctx.set_timing(False)
    flops = 4 * M * N * K + 6 * M * r * (K + N)  # fwd 2MNK + 2Mr(K+N), bwd 2MNK + 4Mr(K+N)
    kern = {k: dict(launches=v[0], avg_ms=v[1] / max(v[0], 1)) for k, v in rep.items()}
    fwd_flops = 2 * M * N * K + 2 * M * r * N
    peak = FP32_MFMA_PEAK_TFLOPS
    # The large GEMMs run on bf16 MFMA: two MFMAs per product for bf16
    # activations (x.wh + x.wl), three for fp32 ones (xh.wh + xh.wl + xl.wh).
    mfma_per_product = 2 if act_dtype == torch.bfloat16 else 3
    act_name = "bfloat16" if act_dtype == torch.bfloat16 else "float32"
    roof = None
    fk = kern.get("forward_gemm_bf16") or kern.get("forward_gemm")
    if fk:
        bf = "forward_gemm_bf16" in kern
        # the pass that writes the operands as bf16 planes belongs to the GEMM
        # (the mean of the forward's and the input gradient's, alike in size)
        gemm_ms = fk["avg_ms"] + kern.get("planes", dict(avg_ms=0.0))["avg_ms"]
        ach = fwd_flops / (gemm_ms * 1e9)
        roof = dict(bound="mfma",
                    kernel=("planes + forward_gemm_bf16 (k_planes: NF4 and activations to bf16 "
                            f"planes; k_plane_gemm: {mfma_per_product} bf16 MFMAs per product)"
                            if bf and "planes" in kern else
                            "forward_gemm_bf16 (k_nf4_bf16 forward: NF4 dequant in the K loop, "
                            f"{mfma_per_product} bf16 MFMAs per product)" if bf
                            else "forward_gemm (k_gemm NF4 fwd, fp32 MFMA)"),
                    achieved=ach, unit="TFLOP/s", flops_per_launch=fwd_flops,
                    peak=BF16_MFMA_PEAK_TFLOPS / mfma_per_product if bf else peak,
                    peak_note=(f"bf16 dense MFMA peak / {mfma_per_product} MFMAs per product"
                               if bf else "fp32 MFMA peak"),
                    frac=ach / (BF16_MFMA_PEAK_TFLOPS / mfma_per_product if bf else peak),
                    mfma_busy_frac=(ach * mfma_per_product / BF16_MFMA_PEAK_TFLOPS if bf
                                    else ach / peak),
                    mfma_busy_counter=(profile_value(
                        "prefill_c3_counters.md",
                        f"mfma_busy_counter[forward_gemm_bf16,{act_name}]")
                        if bf else None),
                    ratio_to_fp32_mfma_peak=ach / peak,
                    traffic=(profile_value(
                        "prefill_c3_counters.md",
                        f"traffic_bytes_per_launch[forward_gemm_bf16,{act_name}]")
                        if bf else None))
    return dict(ms_per_step=ms, tflops=flops / (ms * 1e9),
                ratio_to_fp32_mfma_peak=flops / (ms * 1e9) / peak,
                step_roofline=mfma_roof(flops, ms, "whole fwd+bwd step", mfma_per_product),
                frac_bf16_peak=flops / (ms * 1e9) / BF16_MFMA_PEAK_TFLOPS,
                mfma_per_product=mfma_per_product, flops_per_step=flops,
                steps=steps, kernels=kern, roofline=roof,
                act_dtype=str(act_dtype).replace("torch.", ""))


# ---------------------------------------------------------------------------
def mfma_roof(flops, ms, scope, per_product=3):
    """Roofline of a step whose large products run on bf16 MFMA: an fp32
    product is three MFMAs (xh.wh + xh.wl + xl.wh), so its peak is the bf16
    dense peak / 3 (bf16 activations: / 2)."""
    ach = flops / (ms * 1e9)
    peak = BF16_MFMA_PEAK_TFLOPS / per_product
    return dict(bound="mfma", achieved=ach, peak=peak, unit="TFLOP/s", frac=ach / peak,
                peak_note=(f"bf16 dense MFMA peak / {per_product} MFMAs per product "
                           "(activations and weight as bf16 hi + lo parts)"),
                scope=scope)


def _timed_ms(torch, fn, reps):
    """Mean wall time of fn() on the current stream, between GPU events."""
    fn()
    torch.cuda.synchronize()
    e0 = torch.cuda.Event(enable_timing=True)
    e1 = torch.cuda.Event(enable_timing=True)
    e0.record()
    for _ in range(reps):
        fn()
    e1.record()
    torch.cuda.synchronize()
    return e0.elapsed_time(e1) / reps


def _graph_ms(torch, fn, outs, reps):
    """fn() captured once as a HIP graph and replayed: mean time per replay
    between GPU events (the kernels' own time, host launch cost excluded).
    The replays must reproduce the eager result of fn() bit for bit (every
    tensor of outs()), checked before timing."""
    fn()
    torch.cuda.synchronize()
    ref = [t.clone() for t in outs()]
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        fn()  # warm-up on the capture stream
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    gr = torch.cuda.CUDAGraph()
    with torch.cuda.graph(gr):
        fn()
    for _ in range(3):
        gr.replay()
        torch.cuda.synchronize()
        for t, r in zip(outs(), ref):
            assert torch.equal(t, r), "graph replay differs from the eager run"
    e0 = torch.cuda.Event(enable_timing=True)
    e1 = torch.cuda.Event(enable_timing=True)
    e0.record()
    for _ in range(reps):
        gr.replay()
    e1.record()
    torch.cuda.synchronize()
    del gr
    return e0.elapsed_time(e1) / reps


def _layer(torch, dev, QD, ctx, g, N, K, M, r, alpha, act=None):
    act = act or torch.float32
    w = torch.randn(N, K, device=dev, generator=g) * 0.02
    W = QD.DeviceWeight.quantize(w, 64, True, ctx=ctx)
    del w
    a = (torch.rand(r, K, device=dev, generator=g) * 2 - 1) / math.sqrt(K)
    b = torch.randn(N, r, device=dev, generator=g) * 0.01
    t = dict(N=N, K=K, M=M, r=r, W=W, qw=W.struct(), a=a, b=b,
             lora=QD.lora_struct(a, b, r, alpha),
             x=torch.randn(M, K, device=dev, generator=g).to(act),
             dy=torch.randn(M, N, device=dev, generator=g).to(act),
             y=torch.empty(M, N, device=dev), t1=torch.empty(M, r, device=dev),
             gx=torch.empty(M, K, device=dev), ga=torch.empty(r, K, device=dev),
             gb=torch.empty(N, r, device=dev))
    return t


def _fwd_bwd(QD, ctx, L):
    QD.forward(None, L["lora"], L["x"], L["M"], L["y"], t1=L["t1"], ctx=ctx, qw=L["qw"])
    QD.backward(None, L["lora"], L["x"], L["dy"], L["M"], L["gx"], L["ga"], L["gb"],
                t1=L["t1"], ctx=ctx, qw=L["qw"])


def _fwd_bwd_flops(L):
    M, N, K, r = L["M"], L["N"], L["K"], L["r"]
    return 4 * M * N * K + 6 * M * r * (K + N)


def _adam_step_ms(torch, ctx, tensors, reps=24, max_resident_pages=None):
    """Device 8-bit Adam step over `tensors` (list of (param, grad) CUDA
    tensors).  The step's working set (params, grads, int8 state) is copied
    until the copies pass 512 MB (at most 512 copies), each copy with its own
    optimizer, and the timed steps cycle through them, so that each step's
    data has left the 256 MB MALL.  `kernel_ms` is the Adam kernel's own
    duration (GPU-stamped events around each launch) averaged over `reps`
    steps (the events add their own time); `step_ms` is the eager step
    between events (host launch cost included), from a second pass with the
    per-launch event timing off; `ms` (and the rates) the lower of the two.
    The first step of each copy creates its state, untimed."""
    import ctypes as C
    import qlora_hip as QH
    n = sum(p.numel() for p, _ in tensors)
    blocks = sum(-(-p.numel() // 256) for p, _ in tensors)
    nbytes = 16 * n + 16 * blocks
    copies = max(1, min(512, math.ceil(512e6 / nbytes)))
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    sets = []
    for i in range(copies):
        ts = tensors if i == 0 else [(p.clone(), g_.clone()) for p, g_ in tensors]
        opt = QH.Adam8bit(lr=1e-3, max_resident_pages=max_resident_pages, ctx=ctx)
        cnt = len(ts)
        sets.append(dict(
            ts=ts, opt=opt, cnt=cnt,
            pp=(C.c_void_p * cnt)(*[p.data_ptr() for p, _ in ts]),
            gp=(C.c_void_p * cnt)(*[g_.data_ptr() for _, g_ in ts]),
            ll=(C.c_size_t * cnt)(*[p.numel() for p, _ in ts])))
    st = QH._lib.AdamStats()

    def step(k):
        S = sets[k % copies]
        QH._lib.check(ctx.lib.qh_adam8bit_step_dev(S["opt"].h, S["pp"], S["gp"], S["ll"],
                                                   S["cnt"], C.byref(st), stream))
    for k in range(copies):  # state creation
        step(k)
    torch.cuda.synchronize()
    reps = max(reps, copies)
    ctx.set_timing(True)
    ctx.timing_report(reset=True)
    for k in range(reps):
        step(k)
    torch.cuda.synchronize()
    rep = ctx.timing_report(reset=True)
    ctx.set_timing(False)
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record()
    for k in range(reps):
        step(k)
    e1.record()
    torch.cuda.synchronize()
    step_ms = e0.elapsed_time(e1) / reps
    launches, total = rep.get("adam", (reps, step_ms * reps))
    kms = total / max(launches, 1)
    # the per-launch events add their own time to each bracketed launch, so
    # the step rate of the uninstrumented pass (launches included; the
    # kernel's upper bound when the GPU is the bottleneck) is the figure
    ms = min(kms, step_ms)
    return dict(kernel_ms=kms, step_ms=step_ms, ms=ms, elements=n, tensors=len(tensors),
                bytes=nbytes, gbs=nbytes / (ms * 1e6), frac_hbm=nbytes / (ms * 1e6) / HBM_PEAK_GBS,
                copies=copies, rotated_bytes=copies * nbytes, reps=reps)


def extra_bench(args, ctx, torch, dev, QD):
    """Configurations 1, 4 and 5 and C3's second layer, each at its own
    shapes (3, 4 and 2): GPU time per call, rate,
    fraction of the matching peak."""
    out = {}
    g = torch.Generator(device="cuda").manual_seed(0x9ABC)
    # C1: one 576x576 layer, 64 tokens, r=8 (launch-bound)
    L = _layer(torch, dev, QD, ctx, g, 576, 576, 64, 8, 16.0)
    ms = _timed_ms(torch, lambda: _fwd_bwd(QD, ctx, L), 20)
    f = _fwd_bwd_flops(L)
    gms = _graph_ms(torch, lambda: _fwd_bwd(QD, ctx, L),
                    lambda: [L["y"], L["gx"], L["ga"], L["gb"]], 50)
    out["C1"] = dict(workload="fwd+bwd 576x576 NF4, 64 tokens, r=8", ms=ms, flops=f,
                     tflops=f / (ms * 1e9),
                     ratio_to_fp32_mfma_peak=f / (ms * 1e9) / FP32_MFMA_PEAK_TFLOPS,
                     roofline=mfma_roof(f, ms, "whole fwd+bwd call (latency-bound: 10+ "
                                                "dependent launches of small tiles)"),
                     bound="launch", graph_ms=gms, graph_tflops=f / (gms * 1e9),
                     timing=("ms: eager calls between GPU events (host launch cost "
                             "included); graph_ms: the same calls replayed as one HIP "
                             "graph, checked bit-equal to the eager result"))
    if not args.no_cpu_baseline:
        out["C1"]["cpu_baseline"] = cpu_baseline_c1()
    del L
    # C3, second layer: 14336x4096, 4096 tokens, r=64, fp32 X
    L = _layer(torch, dev, QD, ctx, g, 14336, 4096, 4096, 64, 16.0)
    ms = _timed_ms(torch, lambda: _fwd_bwd(QD, ctx, L), 3)
    f = _fwd_bwd_flops(L)
    out["C3_14336x4096"] = dict(workload="fwd+bwd 14336x4096 NF4, 4096 tokens, r=64, fp32 X",
                                ms=ms, flops=f, tflops=f / (ms * 1e9),
                                ratio_to_fp32_mfma_peak=f / (ms * 1e9) / FP32_MFMA_PEAK_TFLOPS,
                                roofline=mfma_roof(f, ms, "whole fwd+bwd step"))
    del L
    torch.cuda.empty_cache()
    # C4: a SmolLM-135M block's seven projections, 2048 tokens, r=8, then
    # one Adam step over the 14 adapter tensors (max_resident_pages=4)
    projs = [(576, 576), (192, 576), (192, 576), (576, 576), (1536, 576), (1536, 576),
             (576, 1536)]
    Ls = [_layer(torch, dev, QD, ctx, g, N, K, 2048, 8, 16.0) for N, K in projs]
    # q / k / v read one normed input, gate / up another: each group runs
    # through the grouped entry points (one launch per stage); o and down
    # alone
    groups = [[0, 1, 2], [3], [4, 5], [6]]

    def c4_per_layer():
        for L in Ls:
            _fwd_bwd(QD, ctx, L)

    def c4_fb():
        for grp in groups:
            if len(grp) == 1:
                _fwd_bwd(QD, ctx, Ls[grp[0]])
                continue
            G = [Ls[i] for i in grp]
            lay = [(L["qw"], L["lora"]) for L in G]
            QD.forward_shared(lay, G[0]["x"], 2048, [L["y"] for L in G], [L["t1"] for L in G],
                              ctx=ctx)
            QD.backward_shared(lay, G[0]["x"], [L["dy"] for L in G], 2048, G[0]["gx"],
                               [L["ga"] for L in G], [L["gb"] for L in G],
                               [L["t1"] for L in G], ctx=ctx)
    ms = _timed_ms(torch, c4_fb, 5)
    ms_pl = _timed_ms(torch, c4_per_layer, 5)
    f = sum(_fwd_bwd_flops(L) for L in Ls)
    gms = _graph_ms(torch, c4_fb, lambda: [t for L in Ls for t in (L["y"], L["gx"], L["ga"],
                                                                    L["gb"])], 20)
    tens = []
    for L in Ls:
        tens += [(L["a"].clone(), L["ga"]), (L["b"].clone(), L["gb"])]
    ad = _adam_step_ms(torch, ctx, tens, max_resident_pages=4)
    out["C4"] = dict(workload=("fwd+bwd of q/k/v/o/gate/up/down (SmolLM-135M shapes, "
                               "2048 tokens, r=8; q/k/v and gate/up as groups sharing "
                               "their input), then one 8-bit Adam step over the 14 "
                               "adapter tensors"),
                     fwd_bwd_ms=ms, per_layer_ms=ms_pl, flops=f, tflops=f / (ms * 1e9),
                     ratio_to_fp32_mfma_peak=f / (ms * 1e9) / FP32_MFMA_PEAK_TFLOPS,
                     roofline=mfma_roof(f, gms, "the seven projections' fwd+bwd as a "
                                                "replayed HIP graph"),
                     adam=ad, step_ms=ms + ad["ms"], graph_fwd_bwd_ms=gms,
                     graph_tflops=f / (gms * 1e9),
                     graph_ratio_to_fp32_mfma_peak=f / (gms * 1e9) / FP32_MFMA_PEAK_TFLOPS,
                     timing=("fwd_bwd_ms: eager calls between GPU events (host launch "
                             "cost included); graph_fwd_bwd_ms: the same calls replayed "
                             "as one HIP graph, checked bit-equal to the eager result"))
    del Ls, tens
    torch.cuda.empty_cache()
    # C5: 70B-class layers: quantize throughput (bit-exact path), fwd+bwd
    # at 2048 tokens, r=64, then Adam over all four adapter tensors
    c5 = dict(workload=("28672x8192 and 8192x28672: quantize_nf4 from fp32, fwd+bwd at "
                        "2048 tokens r=64, 8-bit Adam over the 4 adapter tensors"))
    qs, fbs, tens = [], [], []
    for N, K in ((28672, 8192), (8192, 28672)):
        w = torch.randn(N, K, device=dev, generator=g) * 0.02
        n = N * K
        qms = _timed_ms(torch, lambda: QD.DeviceWeight.quantize(w, 64, True, ctx=ctx), 3)
        qb = n * (4 + 0.5 + 1 / 64) + 4 * -(-n // 16384)
        qs.append(dict(shape=f"{N}x{K}", ms=qms, bytes=qb, gbs=qb / (qms * 1e6),
                       frac_hbm=qb / (qms * 1e6) / HBM_PEAK_GBS))
        del w
        torch.cuda.empty_cache()
        L = _layer(torch, dev, QD, ctx, g, N, K, 2048, 64, 16.0)
        ms = _timed_ms(torch, lambda: _fwd_bwd(QD, ctx, L), 3)
        f = _fwd_bwd_flops(L)
        fbs.append(dict(shape=f"{N}x{K}", ms=ms, flops=f, tflops=f / (ms * 1e9),
                        ratio_to_fp32_mfma_peak=f / (ms * 1e9) / FP32_MFMA_PEAK_TFLOPS,
                        roofline=mfma_roof(f, ms, "whole fwd+bwd step")))
        tens += [(L["a"].clone(), L["ga"].clone()), (L["b"].clone(), L["gb"].clone())]
        del L
        torch.cuda.empty_cache()
    c5.update(quantize=qs, fwd_bwd=fbs, adam=_adam_step_ms(torch, ctx, tens))
    out["C5"] = c5
    del tens
    torch.cuda.empty_cache()
    out["decode_70b"] = decode_large_bench(torch, dev, QD, ctx, g)
    return out


def decode_large_bench(torch, dev, QD, ctx, g):
    """Decode (forward only) of C5's layers (28672x8192 and 8192x28672),
    r=16, at batches 1, 4 and 16: not a BASELINE configuration, the
    70B-class case of the decode GEMV (several rounds of workgroups; T1 from
    its own launch).  Three weight copies (363 MB) rotate past the MALL; the
    time per call is the sum of the call's kernels' GPU-stamped durations
    (host gaps excluded)."""
    out = {}
    for N, K in ((28672, 8192), (8192, 28672)):
        out[f"{N}x{K}"] = _decode_large(torch, dev, QD, ctx, g, N, K)
    return dict(workload=("decode forward of C5's NF4 layers (block 64, double quant), r=16, "
                          "fp32 X, batches 1/4/16; 3 weight copies rotated"), layers=out)


def _decode_large(torch, dev, QD, ctx, g, N, K):
    r = 16
    copies = []
    for _ in range(3):
        w = torch.randn(N, K, device=dev, generator=g) * 0.02
        W = QD.DeviceWeight.quantize(w, 64, True, ctx=ctx)
        del w
        a = (torch.rand(r, K, device=dev, generator=g) * 2 - 1) / math.sqrt(K)
        b = torch.randn(N, r, device=dev, generator=g) * 0.01
        copies.append((W, QD.lora_struct(a, b, r, 2.0 * r), a, b))
    torch.cuda.empty_cache()
    wbytes = N * K // 2 + N * K // 64 + N * K // 16384 * 4
    res = {}
    for M in (1, 4, 16):
        x = torch.randn(M, K, device=dev, generator=g)
        y = torch.empty(M, N, device=dev)
        for W, lora, _, _ in copies:
            QD.forward(W, lora, x, M, y, ctx=ctx)
        torch.cuda.synchronize()
        reps = 12
        ctx.set_timing(True)
        ctx.timing_report(reset=True)
        for i in range(reps):
            W, lora, _, _ = copies[i % len(copies)]
            QD.forward(W, lora, x, M, y, ctx=ctx)
        torch.cuda.synchronize()
        rep = ctx.timing_report(reset=True)
        ctx.set_timing(False)
        ms = sum(t for _, t in rep.values()) / reps
        algo = wbytes + (r * K + N * r + M * K + M * N) * 4
        res[str(M)] = dict(ms=ms, weight_gbs=wbytes / (ms * 1e6), total_gbs=algo / (ms * 1e6),
                           frac_hbm=algo / (ms * 1e6) / HBM_PEAK_GBS,
                           kernels={k: dict(launches=n, avg_ms=t / n) for k, (n, t) in rep.items()})
    print(f"# decode 70b-class {N}x{K}: " + ", ".join(
        f"batch {m} {v['ms'] * 1e3:.1f} us ({v['total_gbs']:.0f} GB/s)" for m, v in res.items()),
        file=sys.stderr, flush=True)
    del copies
    torch.cuda.empty_cache()
    return res


def glue_bench(args, ctx, torch, dev, QD):
    """The block glue around the projections (llama.rs: RMSNorm, SwiGLU,
    softmax cross-entropy) at two model scales, 2048 tokens: SmolLM-135M
    (hidden 576, MLP 1536, vocab 49152; C4's block) and a 70B-class block
    (hidden 8192, MLP 28672, vocab 128256; C5's layers).  Inputs rotate over
    enough copies that each call misses the 256 MB MALL; the calls over all
    copies are captured once as a HIP graph and replayed, so host launch
    cost stays out (each replay is checked against the eager outputs first).
    Time per call is between GPU events around the replays; bytes are
    algorithmic (each input read once, each output written once)."""
    import ctypes as C
    g = torch.Generator(device="cuda").manual_seed(0x5151)
    out = {}
    T = 2048
    st = lambda: C.c_void_p(torch.cuda.current_stream().cuda_stream)  # noqa: E731
    L = ctx.lib
    for name, H, I, V in (("smollm135m", 576, 1536, 49152), ("70b", 8192, 28672, 128256)):
        res = {}

        def run(op, ws_bytes, make, call, n_out, nbytes, calls=20):
            copies = max(1, -(-512_000_000 // ws_bytes))
            sets = [make() for _ in range(copies)]

            def all_calls():
                for t in sets:
                    call(*t)
            all_calls()
            torch.cuda.synchronize()
            ref = [[x.clone() for x in t[-n_out:]] for t in sets]
            gr = torch.cuda.CUDAGraph()
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                call(*sets[0])
            torch.cuda.current_stream().wait_stream(side)
            torch.cuda.synchronize()
            with torch.cuda.graph(gr):
                all_calls()
            for _ in range(2):
                gr.replay()
                torch.cuda.synchronize()
                for t, rr in zip(sets, ref):
                    for x, y in zip(t[-n_out:], rr):
                        assert torch.equal(x, y), f"{op}: graph replay differs from eager run"
            reps = max(2, -(-calls // copies))
            gr.replay()
            torch.cuda.synchronize()
            e0 = torch.cuda.Event(enable_timing=True)
            e1 = torch.cuda.Event(enable_timing=True)
            e0.record()
            for _ in range(reps):
                gr.replay()
            e1.record()
            torch.cuda.synchronize()
            ms = e0.elapsed_time(e1) / (reps * copies)
            res[op] = dict(ms=ms, bytes=nbytes, gbs=nbytes / (ms * 1e6),
                           frac_hbm=nbytes / (ms * 1e6) / HBM_PEAK_GBS, copies=copies)
            del sets, ref, gr
            torch.cuda.empty_cache()

        w = torch.rand(H, device=dev, generator=g) + 0.5
        rn = lambda *s: torch.randn(*s, device=dev, generator=g)  # noqa: E731
        em = lambda *s: torch.empty(*s, device=dev)  # noqa: E731
        run("rmsnorm", T * H * 8, lambda: (rn(T, H), em(T, H)),
            lambda x, y: QD.rmsnorm(x, w, 1e-5, out=y, ctx=ctx), 1, T * H * 8 + H * 4)
        run("rmsnorm_backward_dx", T * H * 12, lambda: (rn(T, H), rn(T, H), em(T, H)),
            lambda x, dy, dx: QD.check(L.qh_rmsnorm_backward_dev(
                ctx.h, QD._p(x), QD._p(w), QD._p(dy), T, H, 1e-5, QD._p(dx), None, st())),
            1, T * H * 12 + H * 4)
        run("swiglu", T * I * 12, lambda: (rn(T, I), rn(T, I), em(T, I)),
            lambda a, b, o: QD.swiglu(a, b, out=o, ctx=ctx), 1, T * I * 12)
        run("swiglu_backward", T * I * 20,
            lambda: (rn(T, I), rn(T, I), rn(T, I), em(T, I), em(T, I)),
            lambda a, b, d, dg, du: QD.check(L.qh_swiglu_backward_dev(
                ctx.h, QD._p(a), QD._p(b), QD._p(d), T * I, QD._p(dg), QD._p(du), st())),
            2, T * I * 20)
        tg = torch.randint(0, V, (T,), device=dev, generator=g, dtype=torch.int32)
        run("softmax_cross_entropy", T * V * 8,
            lambda: (rn(T, V) * 3, em(1), em(T, V)),
            lambda lg, loss, d: QD.check(L.qh_softmax_cross_entropy_dev(
                ctx.h, QD._p(lg), QD._p(tg), T, V, QD._p(loss), QD._p(d), st())),
            2, T * V * 8 + T * 4 + 4, calls=5)
        out[name] = dict(tokens=T, hidden=H, mlp=I, vocab=V, ops=res)
        print(f"# glue {name}: " + ", ".join(f"{k} {v['gbs']:.0f} GB/s" for k, v in res.items()),
              file=sys.stderr, flush=True)
    return out


def mlp_block_bench(args, ctx, torch, dev, QD):
    """The device-resident MLP block (qh_mlp_forward_dev + _backward_dev:
    RMSNorm, gate/up/down QLoRA projections, SwiGLU, residual add) fwd+bwd
    at 2048 tokens, SmolLM-135M shapes (r=8) and 70B-class shapes (r=64).
    Flops are the three projections' fwd+bwd (4MNK + 6Mr(K+N) each); the
    glue's bytes are left out of the rate."""
    g = torch.Generator(device="cuda").manual_seed(0x3141)
    out = {}
    T = 2048
    for name, H, F, r, reps in (("smollm135m", 576, 1536, 8, 10), ("70b", 8192, 28672, 64, 3)):
        Ws, loras, flops = [], [], 0
        for N, K in ((F, H), (F, H), (H, F)):
            w = torch.randn(N, K, device=dev, generator=g) * 0.02
            Ws.append(QD.DeviceWeight.quantize(w, 64, True, ctx=ctx))
            del w
            a = (torch.rand(r, K, device=dev, generator=g) * 2 - 1) / math.sqrt(K)
            b = torch.randn(N, r, device=dev, generator=g) * 0.01
            loras.append((a, b, r, 16.0))
            flops += 4 * T * N * K + 6 * T * r * (K + N)
        norm = torch.rand(H, device=dev, generator=g) + 0.5
        blk = QD.MLPBlock(norm, *Ws, loras=loras, eps=1e-5, ctx=ctx)
        x = torch.randn(T, H, device=dev, generator=g)
        dy = torch.randn(T, H, device=dev, generator=g)
        c = blk.new_cache(T)

        def step():
            blk.forward(x.clone(), c)
            blk.backward(c, dy)
        ms = _timed_ms(torch, step, reps)
        out[name] = dict(workload=f"MLP block fwd+bwd, hidden {H}, mlp {F}, r={r}, {T} tokens",
                         ms=ms, flops=flops, tflops=flops / (ms * 1e9),
                         ratio_to_fp32_mfma_peak=flops / (ms * 1e9) / FP32_MFMA_PEAK_TFLOPS,
                         roofline=mfma_roof(flops, ms, "the block's fwd+bwd (projection "
                                                       "flops; the glue's time included)"))
        print(f"# mlp block {name}: {ms:.2f} ms, {flops / (ms * 1e9):.1f} TFLOP/s",
              file=sys.stderr, flush=True)
        del blk, Ws, loras, c, x, dy
        torch.cuda.empty_cache()
    return out


def load_bench(args, ctx, torch, dev, QD):
    """Weights into HBM from the host, C5's 28672x8192 layer: the packed
    NF4 file image (pinned host memory, parsed and copied part by part into
    HBM) against the fp32 path (pinned fp32 weights copied to HBM, then
    quantized there).  Host-to-device copies bound both; the packed path
    moves 0.5157 B per weight instead of 4."""
    import numpy as np
    import qlora_hip as QH
    N, K = 28672, 8192
    g = torch.Generator(device="cuda").manual_seed(0x10AD)
    w = torch.randn(N, K, device=dev, generator=g) * 0.02
    W = QD.DeviceWeight.quantize(w, 64, True, ctx=ctx)
    host = dict(rows=N, cols=K, block_size=64, n=N * K, codes=W.codes.cpu().numpy(),
                scale_codes=W.scale_codes.cpu().numpy(), absmax=W.absmax.cpu().numpy())
    img = QH.nf4_file_bytes({"w": host})
    pinned = torch.empty(len(img), dtype=torch.uint8, pin_memory=True)
    pinned.numpy()[:] = np.frombuffer(img, np.uint8)
    w_host = torch.empty(N, K, dtype=torch.float32, pin_memory=True)
    w_host.copy_(w)
    del w
    torch.cuda.empty_cache()

    def packed():
        return QD.load_nf4(pinned, device=dev, ctx=ctx)["w"]

    def fp32():
        wd = w_host.to(dev, non_blocking=True)
        q = QD.DeviceWeight.quantize(wd, 64, True, ctx=ctx)
        torch.cuda.current_stream().synchronize()
        return q

    out = {}
    for name, fn, nbytes in (("packed_file", packed, len(img)), ("fp32_then_quantize", fp32,
                                                                  N * K * 4)):
        fn()
        torch.cuda.synchronize()
        reps = 5
        t0 = time.perf_counter()
        for _ in range(reps):
            q = fn()
        torch.cuda.synchronize()
        ms = (time.perf_counter() - t0) / reps * 1e3
        out[name] = dict(ms=ms, host_bytes=nbytes, gbs=nbytes / (ms * 1e6))
        assert torch.equal(q.codes, W.codes) and torch.equal(q.scale_codes, W.scale_codes)
        del q
    out["speedup"] = out["fp32_then_quantize"]["ms"] / out["packed_file"]["ms"]
    out["workload"] = f"{N}x{K} NF4 (block 64, double quant) from host memory into HBM"
    print(f"# load {N}x{K}: packed {out['packed_file']['ms']:.2f} ms, fp32+quantize "
          f"{out['fp32_then_quantize']['ms']:.2f} ms", file=sys.stderr, flush=True)
    del pinned, w_host, W
    torch.cuda.empty_cache()
    return out


def cpu_baseline_c1():
    sys.path.insert(0, os.path.join(ROOT, "oracle"))
    import oracle as O
    N = K = 576
    r, alpha, M = 8, 16.0, 64
    rng = O.Rng(0x1234_5678_9ABC_DEF0 ^ 0)
    q = O.quantize(rng.normal(N * K, 0.02))
    a = rng.uniform(r * K, -1 / 24, 1 / 24)
    b = rng.normal(N * r, 0.01)
    x = rng.normal(M * K)
    dy = rng.normal(M * N)
    t0, steps = time.perf_counter(), 0
    while True:
        wd = O.dequantize(q)
        O.qlora_forward(wd, N, K, a, b, r, alpha, x, M)
        wd = O.dequantize(q)  # qlora.rs:133: the backward dequantizes again
        O.qlora_backward(wd, N, K, a, b, r, alpha, x, dy, M)
        steps += 1
        if time.perf_counter() - t0 > 2.0 or steps >= 20:
            break
    dt = (time.perf_counter() - t0) / steps
    flops = 4 * M * N * K + 6 * M * r * (K + N)
    return dict(value=flops / (dt * 1e12), unit="TFLOP/s", ms=dt * 1e3, cores=1, kind="port",
                sample=f"{steps} full fwd+bwd calls (single thread), {dt * 1e3:.1f} ms each",
                nproc=os.cpu_count())


def cpu_baseline_decode(seconds):
    sys.path.insert(0, os.path.join(ROOT, "oracle"))
    import numpy as np
    import oracle as O
    r, alpha = 16, 32.0
    rng = O.Rng(0x1234_5678_9ABC_DEF0 ^ 2)
    layers = []
    for N, K in ((11008, 4096), (4096, 11008)):
        w = rng.normal(N * K, 0.02)
        q = O.quantize(w)
        bound = 1.0 / math.sqrt(K)
        layers.append((N, K, q, rng.uniform(r * K, -bound, bound),
                       rng.normal(N * r, 0.01), rng.normal(K)))
    wbytes = sum(O.storage_bytes(L[2]) for L in layers)
    t0, steps = time.perf_counter(), 0
    while True:
        for N, K, q, a, b, x in layers:
            wd = O.dequantize(q)  # qlora.rs:97 dequantizes on every forward
            O.qlora_forward(wd, N, K, a, b, r, alpha, x, 1)
        steps += 1
        if time.perf_counter() - t0 > seconds or steps >= 50:
            break
    dt = (time.perf_counter() - t0) / steps
    return dict(value=wbytes / (dt * 1e9), unit="GB/s", cores=1, kind="port",
                sample=(f"{steps} full decode steps (both layers, batch 1, "
                        f"dequantize + forward, single thread), {dt * 1e3:.1f} ms/step"),
                nproc=os.cpu_count())


def cpu_baseline_prefill(seconds):
    sys.path.insert(0, os.path.join(ROOT, "oracle"))
    import oracle as O
    N = K = 4096
    r, alpha, M = 64, 16.0, 4096
    rows = 64
    rng = O.Rng(0x1234_5678_9ABC_DEF0 ^ 3)
    w = rng.normal(N * K, 0.02)
    q = O.quantize(w)
    a = rng.uniform(r * K, -1 / 64, 1 / 64)
    b = rng.normal(N * r, 0.01)
    x = rng.normal(rows * K)
    dy = rng.normal(rows * N)
    # the two dequantizations of a step (qlora.rs:97 and :133), timed once
    t0 = time.perf_counter()
    wd = O.dequantize(q)
    wd = O.dequantize(q)
    t_deq = time.perf_counter() - t0
    t0, steps = time.perf_counter(), 0
    while True:
        O.qlora_forward(wd, N, K, a, b, r, alpha, x, rows)
        O.qlora_backward(wd, N, K, a, b, r, alpha, x, dy, rows)
        steps += 1
        if time.perf_counter() - t0 > seconds or steps >= 20:
            break
    t_slice = (time.perf_counter() - t0) / steps
    full = t_deq + (M // rows) * t_slice
    flops = 4 * M * N * K + 6 * M * r * (K + N)
    return dict(value=flops / (full * 1e12), unit="TFLOP/s", cores=1, kind="port",
                step_s=full,
                sample=(f"fwd+bwd on a {rows}-row slice of the {M}-token batch ({steps} reps, "
                        f"{t_slice:.2f} s each) scaled by {M // rows} (every GEMM term is "
                        f"linear in tokens), plus the step's two dequantizations timed once "
                        f"({t_deq:.2f} s): {full:.1f} s per full step"),
                nproc=os.cpu_count())


def _cpu_threads():
    """Host threads for the all-core figures: the cores this process may
    run on, at most 16 (the GPU box's share)."""
    try:
        n = len(os.sched_getaffinity(0))
    except AttributeError:
        n = os.cpu_count() or 1
    return max(1, min(16, n))


def _parallel(fns):
    """Runs the callables on host threads (the oracle's ctypes calls release
    the GIL) and returns their results in order."""
    import concurrent.futures as cf
    with cf.ThreadPoolExecutor(max_workers=len(fns)) as ex:
        return list(ex.map(lambda f: f(), fns))


def cpu_baseline_c4(seconds):
    """Configuration 4 on the host: the seven SmolLM-135M projections'
    dequantize + fwd + dequantize + bwd at 2048 tokens (r=8, alpha=16; own X
    and dY each), then one 8-bit Adam step over the 14 adapter tensors with
    max_resident_pages=4 (qlora.rs:86-165, optim.rs:206-248), single thread,
    in full."""
    sys.path.insert(0, os.path.join(ROOT, "oracle"))
    import numpy as np
    import oracle as O
    T, r, alpha = 2048, 8, 16.0
    rng = O.Rng(0x1234_5678_9ABC_DEF0 ^ 4)
    projs = [(576, 576), (192, 576), (192, 576), (576, 576), (1536, 576), (1536, 576),
             (576, 1536)]
    layers = []
    for N, K in projs:
        q = O.quantize(rng.normal(N * K, 0.02))
        bound = 1.0 / math.sqrt(K)
        layers.append((N, K, q, rng.uniform(r * K, -bound, bound), rng.normal(N * r, 0.01),
                       rng.normal(T * K), rng.normal(T * N)))
    t0 = time.perf_counter()
    grads, params = [], []
    for N, K, q, a, b, x, dy in layers:
        wd = O.dequantize(q)
        O.qlora_forward(wd, N, K, a, b, r, alpha, x, T)
        wd = O.dequantize(q)
        _, ga, gb = O.qlora_backward(wd, N, K, a, b, r, alpha, x, dy, T)
        params += [a.copy(), b.copy()]
        grads += [ga, gb]
    t_fb = time.perf_counter() - t0
    opt = O.Adam8bit(lr=1e-3, max_resident_pages=4)
    t0 = time.perf_counter()
    opt.step(params, grads)
    t_adam = time.perf_counter() - t0
    flops = sum(4 * T * N * K + 6 * T * r * (K + N) for N, K, *_ in layers)
    return dict(value=flops / (t_fb * 1e12), unit="TFLOP/s", cores=1, kind="port",
                fwd_bwd_s=t_fb, adam_ms=t_adam * 1e3,
                sample=(f"the full step once, single thread: seven projections' fwd+bwd "
                        f"{t_fb:.2f} s, the 14-tensor Adam step {t_adam * 1e3:.1f} ms"),
                nproc=os.cpu_count())


def cpu_baseline_c5(seconds):
    """Configuration 5 on the host, single thread: quantize_nf4 of the
    28672x8192 layer in full (quant.rs:104-154), that layer's fwd+bwd on a
    64-row slice of the 2048 tokens scaled by 32 (every GEMM term is linear
    in tokens) plus the step's two dequantizations (qlora.rs:86-165), and
    the 8-bit Adam step over all four adapter tensors in full
    (optim.rs:206-248; the 8192x28672 layer's gradients drawn at random,
    its cost does not depend on their values)."""
    sys.path.insert(0, os.path.join(ROOT, "oracle"))
    import numpy as np
    import oracle as O
    rng = np.random.default_rng(0x5C5)
    r, alpha, T, rows = 64, 16.0, 2048, 64
    N, K = 28672, 8192
    w = rng.standard_normal(N * K, dtype=np.float32) * np.float32(0.02)
    t0 = time.perf_counter()
    q = O.quantize(w)
    tq = time.perf_counter() - t0
    del w
    qbytes = N * K * (4 + 0.5 + 1 / 64) + 4 * -(-(N * K) // 16384)
    bound = 1.0 / math.sqrt(K)
    a = rng.uniform(-bound, bound, r * K).astype(np.float32)
    b = rng.standard_normal(N * r, dtype=np.float32) * np.float32(0.01)
    x = rng.standard_normal(rows * K, dtype=np.float32)
    dy = rng.standard_normal(rows * N, dtype=np.float32)
    t0 = time.perf_counter()
    wd = O.dequantize(q)
    wd = O.dequantize(q)
    t_deq = time.perf_counter() - t0
    t0 = time.perf_counter()
    O.qlora_forward(wd, N, K, a, b, r, alpha, x, rows)
    _, ga, gb = O.qlora_backward(wd, N, K, a, b, r, alpha, x, dy, rows)
    t_slice = time.perf_counter() - t0
    del wd, q
    full = t_deq + (T // rows) * t_slice
    flops = 4 * T * N * K + 6 * T * r * (K + N)
    tens = [(a.copy(), ga), (b.copy(), gb)]
    for n in (r * 28672, 8192 * r):  # the 8192x28672 layer's A and B
        tens.append((rng.standard_normal(n, dtype=np.float32),
                     rng.standard_normal(n, dtype=np.float32) * np.float32(0.01)))
    opt = O.Adam8bit(lr=1e-3)
    t0 = time.perf_counter()
    opt.step([p for p, _ in tens], [g_ for _, g_ in tens])
    ta = time.perf_counter() - t0
    n = sum(p.size for p, _ in tens)
    return dict(value=flops / (full * 1e12), unit="TFLOP/s", cores=1, kind="port",
                quantize=dict(shape=f"{N}x{K}", s=tq, gbs=qbytes / (tq * 1e9)),
                fwd_bwd=dict(shape=f"{N}x{K}", step_s=full, slice_s=t_slice,
                             dequantize_s=t_deq),
                adam=dict(s=ta, elements=n, gbs=(16 * n) / (ta * 1e9)),
                sample=(f"single thread: quantize of 28672x8192 in full ({tq:.2f} s); its "
                        f"fwd+bwd on a {rows}-row slice ({t_slice:.1f} s) scaled by "
                        f"{T // rows} plus two dequantizations ({t_deq:.1f} s): "
                        f"{full:.0f} s per full step; the 4-tensor Adam step in full "
                        f"({ta * 1e3:.1f} ms)"),
                nproc=os.cpu_count())


def cpu_all_cores_decode(seconds):
    """The C2 decode step on every host thread: each thread holds its own
    row block of both layers (quantized on its own) and runs dequantize +
    forward on it, the work of qlora.rs:86-107 split by output rows."""
    sys.path.insert(0, os.path.join(ROOT, "oracle"))
    import oracle as O
    nt = _cpu_threads()
    r, alpha = 16, 32.0
    rng = O.Rng(0x1234_5678_9ABC_DEF0 ^ 2)
    work, wbytes = [], 0
    for N, K in ((11008, 4096), (4096, 11008)):
        bound = 1.0 / math.sqrt(K)
        a, x = rng.uniform(r * K, -bound, bound), rng.normal(K)
        for t in range(nt):
            n0, n1 = N * t // nt, N * (t + 1) // nt
            q = O.quantize(rng.normal((n1 - n0) * K, 0.02))
            wbytes += O.storage_bytes(q)
            work.append((t, n1 - n0, K, q, a, rng.normal((n1 - n0) * r, 0.01), x))

    def run(t):
        for tt, n, K, q, a, b, x in work:
            if tt == t:
                O.qlora_forward(O.dequantize(q), n, K, a, b, r, alpha, x, 1)
    t0, steps = time.perf_counter(), 0
    while True:
        _parallel([lambda t=t: run(t) for t in range(nt)])
        steps += 1
        if time.perf_counter() - t0 > seconds / 2 or steps >= 50:
            break
    dt = (time.perf_counter() - t0) / steps
    return dict(value=wbytes / (dt * 1e9), unit="GB/s", cores=nt, kind="port",
                sample=(f"{steps} decode steps on {nt} threads (each its row block of both "
                        f"layers: dequantize + forward), {dt * 1e3:.1f} ms/step"))


def cpu_all_cores_prefill(seconds):
    """The C3 fwd+bwd on every host thread: each thread runs a 64-row token
    slice (its own X and dY) against the shared dequantized weight; the full
    step is the threads' time scaled to 4096 tokens plus the two
    dequantizations (one thread)."""
    sys.path.insert(0, os.path.join(ROOT, "oracle"))
    import oracle as O
    nt = _cpu_threads()
    N = K = 4096
    r, alpha, M, rows = 64, 16.0, 4096, 64
    rng = O.Rng(0x1234_5678_9ABC_DEF0 ^ 3)
    q = O.quantize(rng.normal(N * K, 0.02))
    a = rng.uniform(r * K, -1 / 64, 1 / 64)
    b = rng.normal(N * r, 0.01)
    xs = [(rng.normal(rows * K), rng.normal(rows * N)) for _ in range(nt)]
    t0 = time.perf_counter()
    wd = O.dequantize(q)
    wd = O.dequantize(q)
    t_deq = time.perf_counter() - t0

    def run(t):
        x, dy = xs[t]
        O.qlora_forward(wd, N, K, a, b, r, alpha, x, rows)
        O.qlora_backward(wd, N, K, a, b, r, alpha, x, dy, rows)
    t0 = time.perf_counter()
    _parallel([lambda t=t: run(t) for t in range(nt)])
    t_par = time.perf_counter() - t0
    full = t_deq + (M / (rows * nt)) * t_par
    flops = 4 * M * N * K + 6 * M * r * (K + N)
    return dict(value=flops / (full * 1e12), unit="TFLOP/s", cores=nt, kind="port",
                step_s=full,
                sample=(f"{nt} threads, each fwd+bwd on its own {rows}-row token slice "
                        f"({t_par:.2f} s for all), scaled to {M} tokens, plus the two "
                        f"dequantizations ({t_deq:.2f} s): {full:.1f} s per full step"))


# ---------------------------------------------------------------------------
def main():
    args = parse()
    world = int(os.environ.get("WORLD_SIZE", "1"))
    if args.gpus != 1 or world != 1:
        print("bench.py measures one GPU: this build has no multi-GPU path "
              "(the hot path would shard by tokens, one process per GPU); run with --gpus 1",
              file=sys.stderr)
        sys.exit(2)
    import torch
    import qlora_hip
    from qlora_hip import device as QD
    if not torch.cuda.is_available():
        print("no GPU visible", file=sys.stderr)
        sys.exit(1)
    dev = torch.device("cuda:0")
    ctx = qlora_hip.default_context()
    print(f"# device: {ctx.device_name()}", file=sys.stderr, flush=True)
    if args.probe:
        probe(args.probe, ctx, torch, dev, QD)
        return
    phases = set(args.phases.split(","))
    if args.skip_prefill:
        phases.discard("prefill")
    if args.skip_extra:
        phases -= {"extra", "load", "mlp"}
    if args.skip_glue:
        phases.discard("glue")
    if "decode" not in phases:
        # a profiling run of other phases: no JSON line
        run_phases(args, phases, ctx, torch, dev, QD)
        return

    copy_peak = hbm_copy_peak(torch, dev)
    print(f"# HBM copy: {copy_peak['gbs']:.0f} GB/s", file=sys.stderr, flush=True)
    read_ceil = read_ceiling(torch, dev)
    if read_ceil:
        print("# one-launch read ceiling: " + ", ".join(
            f"{k} MiB {v['gbs']:.0f} GB/s" for k, v in read_ceil.items()),
            file=sys.stderr, flush=True)
    dec, dec_cfg = decode_bench(args, ctx, torch, dev, QD)
    print(f"# decode done: {json.dumps({b: round(v['weight_gbs'], 1) for b, v in dec.items()})}",
          file=sys.stderr, flush=True)
    prefill, extra, glue, load, mlp = run_phases(args, phases, ctx, torch, dev, QD)
    cpu_dec = cpu_pre = cpu_all = None
    if not args.no_cpu_baseline:
        cpu_dec = cpu_baseline_decode(args.cpu_seconds)
        cpu_all = cpu_all_cores_decode(args.cpu_seconds)
        print(f"# cpu decode: 1 thread {cpu_dec['value']:.2f} GB/s, {cpu_all['cores']} threads "
              f"{cpu_all['value']:.2f} GB/s", file=sys.stderr, flush=True)
        if "prefill" in phases:
            cpu_pre = cpu_baseline_prefill(args.cpu_seconds)
            prefill["cpu_baseline"] = cpu_pre
            prefill["cpu_baseline_all_cores"] = cpu_all_cores_prefill(args.cpu_seconds)
        if "extra" in phases and extra:
            extra["C4"]["cpu_baseline"] = cpu_baseline_c4(args.cpu_seconds)
            extra["C5"]["cpu_baseline"] = cpu_baseline_c5(args.cpu_seconds)
            print(f"# cpu C4 {extra['C4']['cpu_baseline']['sample']}; C5 "
                  f"{extra['C5']['cpu_baseline']['sample']}", file=sys.stderr, flush=True)
    emit(args, copy_peak, read_ceil, dec, dec_cfg, cpu_dec, prefill, extra, glue, load, mlp,
         cpu_all)


def vendor_gemm_ref(torch, dev, reps=20):
    """A plain bf16 GEMM of C3's shape (4096 x 4096 x 4096, C = A B^T) through
    torch.matmul (the vendor library), on this box: the MFMA rate a tuned
    library GEMM reaches with no dequantization in its K loop.  A reference
    for the forward kernel's rate only (the product never calls it)."""
    M = N = K = 4096
    g = torch.Generator(device="cuda").manual_seed(0x9e)
    a = torch.randn(M, K, device=dev, generator=g).to(torch.bfloat16)
    b = torch.randn(N, K, device=dev, generator=g).to(torch.bfloat16)
    ms = _timed_ms(torch, lambda: a @ b.t(), reps)
    tf = 2 * M * N * K / (ms * 1e9)
    return dict(shape=[M, N, K], ms=ms, tflops=tf, frac_bf16_peak=tf / BF16_MFMA_PEAK_TFLOPS,
                how="torch.matmul, bf16 in, fp32 accumulate, mean of %d launches" % reps)


def run_phases(args, phases, ctx, torch, dev, QD):
    prefill = {}
    if "prefill" in phases:
        vendor = vendor_gemm_ref(torch, dev)
        for dt_ in (torch.float32, torch.bfloat16):
            p = prefill_bench(args, ctx, torch, dev, QD, dt_)
            # the forward kernel's MFMA rate (its flops times the MFMAs per
            # product) against the vendor GEMM's on the same box
            p["roofline"]["mfma_rate_vs_vendor_gemm"] = (
                p["roofline"]["achieved"] * p["mfma_per_product"] / vendor["tflops"])
            prefill[p["act_dtype"]] = p
            print(f"# prefill {p['act_dtype']}: {p['tflops']:.1f} TFLOP/s",
                  file=sys.stderr, flush=True)
        prefill["vendor_bf16_gemm"] = vendor
        print(f"# vendor bf16 GEMM 4096^3: {vendor['tflops']:.0f} TFLOP/s",
              file=sys.stderr, flush=True)
    extra = {}
    if "extra" in phases:
        extra = extra_bench(args, ctx, torch, dev, QD)
        print(f"# extra configs done: {sorted(extra)}", file=sys.stderr, flush=True)
    glue = glue_bench(args, ctx, torch, dev, QD) if "glue" in phases else None
    load = load_bench(args, ctx, torch, dev, QD) if "load" in phases else None
    mlp = mlp_block_bench(args, ctx, torch, dev, QD) if "mlp" in phases else None
    return prefill, extra, glue, load, mlp


def _frac_of_read(d1, read_ceil):
    """The decode launch against one read launch of (about) its own size."""
    if not read_ceil:
        return None
    mib = d1["main_kernel_bytes"] / (1 << 20)
    key = min(read_ceil, key=lambda k: abs(int(k) - mib))
    return dict(size_mib=int(key), frac=d1["main_kernel_gbs"] / read_ceil[key]["gbs"])


def emit(args, copy_peak, read_ceil, dec, dec_cfg, cpu_dec, prefill, extra, glue, load, mlp,
         cpu_all=None):
    d1 = dec[1]
    roof = None
    if "main_kernel_gbs" in d1:
        roof = dict(bound="hbm",
                    kernel=(f"{d1['main_kernel']} (fused NF4 dequant-GEMV + LoRA "
                            "epilogue, batch 1"
                            + (", both layers in one launch)" if d1["main_kernel"] == "decode_stream2"
                               else ", mean of the two layers)")),
                    achieved=d1["main_kernel_gbs"], peak=HBM_PEAK_GBS, unit="GB/s",
                    frac=d1["main_kernel_gbs"] / HBM_PEAK_GBS,
                    measured_copy_peak=copy_peak,
                    frac_of_measured=(d1["main_kernel_gbs"] / copy_peak["gbs"]
                                      if copy_peak else None),
                    read_ceiling=read_ceil,
                    frac_of_read_ceiling=_frac_of_read(d1, read_ceil),
                    bytes_per_launch=d1["main_kernel_bytes"],
                    avg_launch_ms=d1["main_kernel_ms"], traffic=measured_traffic())
    line = {
        "metric": METRIC,
        "value": d1["weight_gbs"],
        "unit": "GB/s",
        "n_gpus": 1,
        "steps": d1["steps"],
        "warmup": args.warmup,
        "ms_per_step": d1["ms_per_step"],
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32",
        "data": "synthetic (seeded torch RNG on GPU; NF4 weights quantized on GPU)",
        "config": {
            "workload": ("C2 decode: fused NF4 dequant-GEMV forward of 11008x4096 "
                         "then 4096x11008 (block 64, double quant), LoRA r=16 "
                         "alpha=32, batch 1, fp32 X"),
            "global_batch": 1,
            "weight_copies_rotated": dec_cfg["copies"],
            "packed_weight_bytes_per_step": dec_cfg["packed_weight_bytes"],
            "parallelism": "none (1 GPU)",
        },
        "roofline": roof,
        "cpu_baseline": cpu_dec,
        "cpu_baseline_all_cores": cpu_all,
        "decode_batches": {str(b): {k: v for k, v in r_.items()} for b, r_ in dec.items()},
        "decode_host_path": dec_cfg["host_path"],
        "prefill": prefill,
        "configs": extra,
        "block_glue": glue,
        "weight_load": load,
        "mlp_block": mlp,
    }
    print(json.dumps(line))


if __name__ == "__main__":
    main()
