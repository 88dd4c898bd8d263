#!/usr/bin/env python
"""Benchmark of the MoE expert-layer hot path on one MI355X.

A step is one forward + backward of the layer (router -> permute -> grouped SwiGLU MLP -> unpermute)
on seeded synthetic input already resident in HBM: drawn on the CPU generator in fp32 in a fixed
order and cast, so that the CPU baseline computes on the very same bits.  Prints ONE JSON line:
  value      whole-layer TFLOP/s with the grouped-GEMM numerator 18*N*H*F (N = T*k routed rows)
  roofline   the grouped GEMM launches, timed with HIP events inside the timed steps
  permute    achieved GB/s of the permute / unpermute row kernels (HBM roofline)
  cpu_baseline  the oracle (CPU restatement of the reference's torch-native path) timed on this
             box's host cores on a bounded sample of the same workload
"""
import argparse
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

MFMA_PEAK = {"bf16": 2500.0, "f16": 2500.0, "f32": 157.3}  # dense TFLOP/s, MI355X
HBM_PEAK_GBPS = 8000.0


def parse_args():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=50)
    ap.add_argument("--warmup", type=int, default=10)
    ap.add_argument("--workload", default="mixtral",
                    help="mixtral (default, the configuration the metric is quoted on), tiny, "
                         "finegrained, mixtral_skew, dsv3_shard (the shard's shape with bf16 weights, "
                         "forward + backward), dsv3_shard_fp8 (4096 routed rows on block-scaled fp8 "
                         "weights, forward + input gradient)")
    ap.add_argument("--device-inputs", action="store_true",
                    help="draw the inputs on the device generator (starts faster; the CPU baseline "
                         "then draws its own)")
    ap.add_argument("--dispatcher", default="allgather", choices=["allgather", "alltoall"])
    ap.add_argument("--pre-router-norm", action="store_true",
                    help="put the RMSNorm in front of the router into the step (the layer input is "
                         "then the un-normalised residual stream, which the combine adds back)")
    ap.add_argument("--operands", default="random", choices=["random", "zeros"],
                    help="zeros: activations, gradients and expert weights all zero, routing from random "
                         "logits: the same launches without data-dependent switching power (a "
                         "diagnostic, not the benchmark)")
    ap.add_argument("--graph", action=argparse.BooleanOptionalAction, default=None,
                    help="time replays of the step captured in a HIP graph; the eager figures are "
                         "reported beside it and the per-kernel figures still come from eager steps.  "
                         "Default: on for the workloads whose launch gaps show (`tiny`: 26 launches of a few "
                         "microseconds each; `dsv3_shard_fp8`: eight to ten launches of 10-300 us; "
                         "`finegrained`: 41 launches in 5.7 ms), off elsewhere; --no-graph times eager "
                         "steps")
    ap.add_argument("--fp8-activations", action="store_true",
                    help="dsv3_shard_fp8 only: quantise the rows entering each of the four products to "
                         "fp8 as well (a power-of-two scale per row and 128 elements) and run them on the "
                         "block-scaled fp8 MFMA; not the configuration as stated (bf16 activations), "
                         "reported beside it")
    ap.add_argument("--shared-overlap", action="store_true",
                    help="workloads with shared experts: run them on their own stream beside the "
                         "dispatch and the routed experts (the reference's moe_shared_expert_overlap)")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--blas-reference", action="store_true",
                    help="also time the BLAS library (torch.matmul) on one expert's share of each of "
                         "the six GEMM shapes, after the timed steps; adds 'blas_reference'")
    ap.add_argument("--cpu-tokens", type=int, default=4096,
                    help="tokens of the bounded CPU sample (same H, F, E, top-k)")
    args = ap.parse_args()
    if args.graph is None:
        args.graph = args.workload in ("tiny", "dsv3_shard_fp8", "finegrained")
    return args


class KernelTimer:
    """Wraps the package's tensor-level launch wrappers with HIP event pairs on the launch stream.  The
    layer itself launches from native autograd nodes, so the timed kernels come from a pass that issues
    a step's launches one by one through the wrappers (`launch_by_launch`, `launch_by_launch_fp8`)."""

    def __init__(self, torch, ops):
        self.torch = torch
        self.ops = ops
        self.records = []  # (name, start_event, end_event, work)
        self.enabled = False
        self._orig = {}

    def _wrap(self, name, label_fn):
        orig = getattr(self.ops, name)
        self._orig[name] = orig
        torch = self.torch

        def wrapped(*a, **kw):
            if not self.enabled:
                return orig(*a, **kw)
            s = torch.cuda.Event(enable_timing=True)
            e = torch.cuda.Event(enable_timing=True)
            s.record()
            out = orig(*a, **kw)
            e.record()
            self.records.append((label_fn(*a, **kw), s, e))
            return out

        setattr(self.ops, name, wrapped)

    def install(self):
        def gmm_label(a, b, off, trans_a=False, trans_b=False, out_dtype=None):
            N, K = a.shape
            if trans_a:
                M, mode = b.shape[1], "TN"
            else:
                M, mode = (b.shape[1], "NT") if trans_b else (b.shape[2], "NN")
            return ("gmm_%s" % mode, 2.0 * N * K * M, (N, K, M))

        self._wrap("gmm", gmm_label)

        def glu_fwd_label(a, w1, off, act="silu"):
            N, K = a.shape
            return ("gmm_NN+glu", 2.0 * N * K * w1.shape[2], (N, K, w1.shape[2]))

        def glu_bwd_label(go, w2, fc1, off, act="silu"):
            N, K = go.shape
            return ("gmm_NT+glu_bwd", 2.0 * N * K * w2.shape[1], (N, K, w2.shape[1]))

        self._wrap("gmm_glu", glu_fwd_label)
        self._wrap("gmm_glu_bwd", glu_bwd_label)
        for nm in ("permute_rows", "unpermute_rows", "unpermute_rows_bwd", "glu_fwd", "glu_bwd",
                   "permute_plan", "route_topk", "route_topk_bwd", "rmsnorm_fwd", "rmsnorm_bwd", "gate_fwd",
                   "gate_bwd"):
            self._wrap(nm, (lambda n: (lambda *a, **kw: (n, 0.0, None)))(nm))

    def install_fp8(self):
        def label(a, b_q, b_scale, off, trans_b=False):
            N, K = a.shape
            M = b_q.shape[1] if trans_b else b_q.shape[2]
            return ("gmm_fp8w_%s" % ("NT" if trans_b else "NN"), 2.0 * N * K * M, (N, K, M), float(b_q.numel()))

        self._wrap("gmm_fp8w", label)

        def label_a(a_q, a_scale, b_q, b_scale, off, trans_b=False):
            N, K = a_q.shape
            M = b_q.shape[1] if trans_b else b_q.shape[2]
            return ("gmm_fp8a_%s" % ("NT" if trans_b else "NN"), 2.0 * N * K * M, (N, K, M), float(b_q.numel()))

        self._wrap("gmm_fp8a", label_a)
        for nm in ("glu_fwd", "glu_bwd", "quantize_fp8_rows", "glu_fwd_quantize_fp8_rows",
                   "glu_bwd_quantize_fp8_rows"):
            self._wrap(nm, (lambda n: (lambda *a, **kw: (n, 0.0, None)))(nm))

    def uninstall(self):
        for k, v in self._orig.items():
            setattr(self.ops, k, v)

    def summary(self):
        agg = {}
        for label, s, e in self.records:
            name, work, shape = label[:3]
            key = name if shape is None else "%s %s" % (name, "x".join(map(str, shape)))
            d = agg.setdefault(key, {"name": name, "ms": 0.0, "calls": 0, "work": work,
                                     "bytes": label[3] if len(label) > 3 else 0.0})
            d["ms"] += s.elapsed_time(e)
            d["calls"] += 1
        return agg


def launch_by_launch(torch, ops, w, router_weight, experts, shared, norm, x, dy, route_logits=None, logit_bias=None):
    """One forward + backward of the layer as its sequence of launches, without autograd."""
    T, H, E, F, k = w.tokens, w.hidden, w.experts, w.ffn, w.topk
    x, dy = x.detach().view(T, H), dy.view(T, H)
    w1, w2 = experts.weight1.detach().view(E, H, 2 * F), experts.weight2.detach().view(E, F, H)
    h, residual = x, None
    if norm is not None:
        (h, rstd), residual = ops.rmsnorm_fwd(x, norm.weight.detach(), norm.eps), x
    logits = ops.gate_fwd(h, router_weight) if route_logits is None else route_logits
    if logit_bias is not None:
        logits = logits + logit_bias
    aux_scale = E * 0.01 / (T * T * k)
    probs, rmap, counts, stats, _ = ops.route_topk(logits, k, want_stats=True)
    ops.router_bookkeeping(stats, counts, E, aux_factor=aux_scale, want_aux=True)
    plan = ops.permute_plan(rmap, T * k, want_sorted=False)
    off, dst = plan.expert_offsets, plan.dst_map
    xp, _ = ops.permute_rows(h, dst, T * k)
    fc1, act = ops.gmm_glu(xp, w1, off)
    y = ops.gmm(act, w2, off)
    addend = None
    if shared is not None:
        s1, s2 = shared.linear_fc1.weight.detach().unsqueeze(0), shared.linear_fc2.weight.detach().unsqueeze(0)
        one = ops.one_group(T, x.device)._gmoe_offsets
        sfc1 = ops.gmm(h, s1, one, trans_b=True)
        sact = ops.glu_fwd(sfc1)
        addend = ops.gmm(sact, s2, one, trans_b=True)
    ops.unpermute_rows(y, dst, T, merging_probs=probs, residual=residual, addend=addend)
    dyp, dprobs = ops.unpermute_rows_bwd(dy, y, dst, probs)
    dfc1 = ops.gmm_glu_bwd(dyp, w2, fc1, off)
    ops.gmm(act, dyp, off, trans_a=True)
    dxp = ops.gmm(dfc1, w1, off, trans_b=True)
    ops.gmm(xp, dfc1, off, trans_a=True)
    dh, _ = ops.unpermute_rows(dxp, dst, T)
    if shared is not None:
        dsact = ops.gmm(dy, s2, one)
        ops.gmm(dy, sact, one, trans_a=True)
        dsfc1 = ops.glu_bwd(dsact, sfc1)
        dh = dh + ops.gmm(dsfc1, s1, one)
        ops.gmm(dsfc1, h, one, trans_a=True)
    dlogits = ops.route_topk_bwd(logits, k, "softmax", False, None, rmap, dprobs, counts, aux_scale)
    dg, _ = ops.gate_bwd(dlogits, h, router_weight)
    dh = dh + dg
    if norm is not None:
        ops.rmsnorm_bwd(dh, x, norm.weight.detach(), rstd, dy)


def launch_by_launch_fp8(ops, fp8, x, dy, off):
    """One forward + input gradient of the fp8 shard as its sequence of launches."""
    w1, s1, w2, s2 = fp8.weight1_q, fp8.weight1_scale, fp8.weight2_q, fp8.weight2_scale
    x = x.detach()
    if fp8.fp8_activations:
        fc1 = ops.gmm_fp8a(*ops.quantize_fp8_rows(x), w1, s1, off)
        ops.gmm_fp8a(*ops.glu_fwd_quantize_fp8_rows(fc1), w2, s2, off)
        dact = ops.gmm_fp8a(*ops.quantize_fp8_rows(dy), w2, s2, off, trans_b=True)
        ops.gmm_fp8a(*ops.glu_bwd_quantize_fp8_rows(dact, fc1), w1, s1, off, trans_b=True)
    else:
        fc1 = ops.gmm_fp8w(x, w1, s1, off)
        ops.gmm_fp8w(ops.glu_fwd(fc1), w2, s2, off)
        dact = ops.gmm_fp8w(dy, w2, s2, off, trans_b=True)
        ops.gmm_fp8w(ops.glu_bwd(dact, fc1), w1, s1, off, trans_b=True)


def blas_reference(torch, w, dev, reps=10, zeros=False):
    """The vendor BLAS library on one expert's share (N/E rows) of the layer's six GEMMs, same dtype,
    same kind of data: a yardstick for what this chip sustains on these shapes, not part of `value`."""
    n = w.routed_rows // w.experts
    H, F = w.hidden, w.ffn
    g = torch.Generator(device=dev).manual_seed(7)

    def rnd(*shape, scale=1.0):
        if zeros:
            return torch.zeros(*shape, device=dev, dtype=w.dtype)
        return (scale * torch.randn(*shape, generator=g, device=dev, dtype=torch.float32)).to(w.dtype)

    x, fc1, act, dy = rnd(n, H), rnd(n, 2 * F), rnd(n, F), rnd(n, H)
    w1, w2 = rnd(H, 2 * F, scale=0.02), rnd(F, H, scale=0.02)
    cases = {
        "NN fc1 %dx%dx%d" % (n, H, 2 * F): (lambda: torch.matmul(x, w1), 2.0 * n * H * 2 * F),
        "NN fc2 %dx%dx%d" % (n, F, H): (lambda: torch.matmul(act, w2), 2.0 * n * F * H),
        "NT dx %dx%dx%d" % (n, 2 * F, H): (lambda: torch.matmul(fc1, w1.t()), 2.0 * n * H * 2 * F),
        "NT dact %dx%dx%d" % (n, H, F): (lambda: torch.matmul(dy, w2.t()), 2.0 * n * F * H),
        "TN dW1 %dx%dx%d" % (n, H, 2 * F): (lambda: torch.matmul(x.t(), fc1), 2.0 * n * H * 2 * F),
        "TN dW2 %dx%dx%d" % (n, F, H): (lambda: torch.matmul(act.t(), dy), 2.0 * n * F * H),
    }
    out = {}
    for name, (fn, flops) in cases.items():
        fn()
        torch.cuda.synchronize()
        s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        s.record()
        for _ in range(reps):
            fn()
        e.record()
        torch.cuda.synchronize()
        ms = s.elapsed_time(e) / reps
        out[name] = {"avg_ms": round(ms, 4), "tflops": round(flops / ms / 1e9, 1)}
    return out


def cpu_baseline(w, tokens, dispatcher, inputs=None):
    """Oracle forward+backward of the layer on the host for the first `tokens` tokens of the
    workload: the very tensors the GPU ran on when `inputs` (the CPU-drawn dict) is given."""
    import torch
    from oracle import moe_oracle as orc
    import __graft_entry__ as entry

    pkg = entry.load_package()
    cores = os.cpu_count() or 1
    env = os.environ.get("OMP_NUM_THREADS")
    if env:
        cores = min(cores, int(env))
    torch.set_num_threads(cores)
    ws = pkg.configs.scaled(w, tokens=tokens)
    if inputs is None:
        inp = pkg.configs.make_inputs(ws, seed=1234)
        shared = "its own draw of the inputs"
    else:
        seq = tokens // w.batch  # token index = s * B + b: the first sequence positions
        inp = dict(inputs, x=inputs["x"][:seq], dy=inputs["dy"][:seq])
        shared = "the first %d sequence positions of the GPU run's own tensors" % seq
    x = inp["x"].float().requires_grad_(True)
    w_r = inp["w_r"].float().requires_grad_(True)
    w1 = inp["w1"].detach().clone().requires_grad_(True)  # storage dtype; the oracle computes in fp32
    w2 = inp["w2"].detach().clone().requires_grad_(True)
    dy = inp["dy"].float()
    kw = {}
    if w.shared_ffn:
        kw = dict(shared_w1=inp["shared_w1"], shared_w2=inp["shared_w2"])
    t0 = time.perf_counter()
    out, aux, info = orc.moe_layer(x, w_r, w1, w2, ws.topk, dispatcher=dispatcher, **kw)
    out.backward(dy)
    dt = time.perf_counter() - t0
    flops = ws.gemm_flops()
    return {
        "value": flops / dt / 1e12,
        "unit": "TFLOP/s",
        "cores": cores,
        "kind": "port",
        "seconds": dt,
        "sample": "oracle (torch CPU, fp32 math) layer fwd+bwd on T=%d of %d tokens (%s), same H=%d "
                  "F=%d E=%d top-%d; 1 repetition" % (tokens, w.tokens, shared, w.hidden, w.ffn,
                                                      w.experts, w.topk),
    }


def hbm_entry(agg, name, nbytes, label=None):
    v = agg.get(name)
    if not v:
        return None
    avg = v["ms"] / v["calls"]
    gbps = nbytes / (avg * 1e-3) / 1e9
    return {"bound": "hbm", "kernel": label or name, "achieved": round(gbps, 1), "peak": HBM_PEAK_GBPS,
            "unit": "GB/s", "frac": round(gbps / HBM_PEAK_GBPS, 4), "avg_ms": round(avg, 4),
            "bytes": nbytes}


def run_fp8_shard(args, torch, pkg, dev):
    """The DeepSeek-V3-shape shard as one GPU receives it after dispatch: N = 4096 routed rows spread
    multinomially over 32 local experts (two empty), H 7168, F 2048, block-scaled fp8 (e4m3) expert
    weights, bf16 activations; a step is the gated expert MLP forward plus the gradient of its input
    (four grouped GEMMs on fp8 weights + the activation forward and backward)."""
    w = pkg.configs.WORKLOADS["dsv3_shard"]
    E, H, F = w.experts, w.hidden, w.ffn
    N = w.tokens * w.topk * E // w.global_experts  # 4096
    g = torch.Generator().manual_seed(1234)
    x_cpu = torch.randn(N, H, generator=g)
    w1_cpu = 0.02 * torch.randn(E, H, 2 * F, generator=g)
    w2_cpu = 0.02 * torch.randn(E, F, H, generator=g)
    dy_cpu = torch.randn(N, H, generator=g)
    counts = pkg.configs.multinomial_counts(N, E, seed=1234, empty=2)
    cfg = pkg.MoEConfig(hidden_size=H, num_moe_experts=E, moe_ffn_hidden_size=F, params_dtype=w.dtype)
    mlp = pkg.GroupedMLP(E, cfg, device=dev)
    with torch.no_grad():
        mlp.weight1.view(E, H, 2 * F).copy_(w1_cpu.to(dev))
        mlp.weight2.view(E, F, H).copy_(w2_cpu.to(dev))
    fp8 = pkg.Fp8GroupedMLP(mlp, fp8_activations=args.fp8_activations)
    del mlp
    x = x_cpu.to(dev, w.dtype).requires_grad_(True)
    dy = dy_cpu.to(dev, w.dtype)
    tpe = counts.to(dev)
    tpe._gmoe_offsets = pkg.ops.expert_offsets_from_batch_sizes(counts, dev)

    def step():
        x.grad = None
        out, _ = fp8(x, tpe)
        out.backward(dy)

    if args.graph:
        # every step of this run on one side stream, the capture included (see main())
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        torch.cuda.set_stream(side)
    for _ in range(args.warmup):
        step()
    torch.cuda.synchronize()
    marks = [torch.cuda.Event(enable_timing=True) for _ in range(args.steps + 1)]
    t0 = time.perf_counter()
    for i in range(args.steps):
        marks[i].record()
        step()
    marks[args.steps].record()
    torch.cuda.synchronize()
    dt = time.perf_counter() - t0
    timer = KernelTimer(torch, pkg.ops)
    timer.install_fp8()
    timer.enabled = True
    for _ in range(args.steps):
        launch_by_launch_fp8(pkg.ops, fp8, x, dy, tpe._gmoe_offsets)
    torch.cuda.synchronize()
    timer.uninstall()
    per_step = sorted(marks[i].elapsed_time(marks[i + 1]) for i in range(args.steps))
    median = per_step[len(per_step) // 2]
    eager = None
    if args.graph:
        # the same step recorded once and replayed: its ten launches of 10-300 us without the gaps
        # the host leaves between them
        eager = {"ms_per_step": round(dt * 1e3 / args.steps, 4), "ms_per_step_median": round(median, 4)}
        x.grad = None
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            step()
        for _ in range(args.warmup):
            graph.replay()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for i in range(args.steps):
            marks[i].record()
            graph.replay()
        marks[args.steps].record()
        torch.cuda.synchronize()
        dt = time.perf_counter() - t0
        per_step = sorted(marks[i].elapsed_time(marks[i + 1]) for i in range(args.steps))
        median = per_step[len(per_step) // 2]
        del graph
    flops = 12.0 * N * H * F
    weight_bytes = float(E * H * 2 * F + E * F * H)  # one pass over both fp8 weight tensors
    agg = timer.summary()
    kernels = {}
    for k, v in sorted(agg.items()):
        avg = v["ms"] / v["calls"]
        ent = {"calls_per_step": v["calls"] / args.steps, "avg_ms": round(avg, 4)}
        if v["work"]:
            ent["tflops"] = round(v["work"] / (avg * 1e-3) / 1e12, 1)
        if v.get("bytes"):
            ent["weight_GBps"] = round(v["bytes"] / (avg * 1e-3) / 1e9, 1)
        kernels[k] = ent
    gemm = {k: v for k, v in agg.items() if v["name"].startswith("gmm_fp8")}
    gemm_ms = sum(v["ms"] for v in gemm.values()) / args.steps
    dom_key = max(gemm, key=lambda k: gemm[k]["work"] * (1.0 if "NN" in k else 0.99))
    d = gemm[dom_key]
    d_ms = d["ms"] / d["calls"]
    value = flops / (dt / args.steps) / 1e12
    result = {
        "metric": "MoE layer fwd+bwd TFLOP/s (1 GPU, % MFMA peak); permute GB/s (% HBM)",
        "value": round(value, 2), "unit": "TFLOP/s", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": round(dt * 1e3 / args.steps, 4),
        "ms_per_step_median": round(median, 4), "higher_is_better": True, "scaling": "weak",
        "vs_baseline": None,
        "dtype": ("fp8 (e4m3 rows and weights on the block-scaled fp8 MFMA)" if args.fp8_activations
                  else "bf16 (fp8 e4m3 weights widened exactly to bf16)"),
        "data": "synthetic",
        "config": {"workload": "dsv3_shard_fp8: expert MLP fwd + dX on N=%d routed rows over %d local "
                               "experts (multinomial counts, 2 empty), H=%d F=%d, block-scaled fp8 "
                               "weights" % (N, E, H, F) +
                               (", rows quantised to fp8 as well" if args.fp8_activations else ""),
                   "flops_per_step": flops,
                   "weight_bytes_per_pass": weight_bytes,
                   "launch": "HIP graph replay" if args.graph else "eager"},
        "pct_mfma_peak": round(100 * value / (5000.0 if args.fp8_activations else MFMA_PEAK["bf16"]), 2),
        # weight-streaming regime (128 rows per expert): both rooflines of the largest launch
        "roofline": {"bound": "hbm", "kernel": "gmm_fp8_skinny_kernel " + dom_key,
                     "achieved": round(d["bytes"] / (d_ms * 1e-3) / 1e9, 1), "peak": HBM_PEAK_GBPS,
                     "unit": "GB/s", "frac": round(d["bytes"] / (d_ms * 1e-3) / 1e9 / HBM_PEAK_GBPS, 4),
                     "traffic": None,
                     "mfma": {"achieved": round(d["work"] / (d_ms * 1e-3) / 1e12, 1),
                              "peak": MFMA_PEAK["bf16"], "unit": "TFLOP/s",
                              "frac": round(d["work"] / (d_ms * 1e-3) / 1e12 / MFMA_PEAK["bf16"], 4)},
                     "all_gmm_launches": {"ms_per_step": round(gemm_ms, 4),
                                          "weight_GBps": round(2 * weight_bytes / (gemm_ms * 1e-3) / 1e9, 1),
                                          "frac_hbm": round(2 * weight_bytes / (gemm_ms * 1e-3) / 1e9 / HBM_PEAK_GBPS, 4),
                                          "tflops": round(flops / (gemm_ms * 1e-3) / 1e12, 1)}},
        "kernels": kernels,
    }
    if eager is not None:
        result["eager"] = eager
    if not args.no_cpu_baseline:
        from oracle import moe_oracle as orc

        cores = min(os.cpu_count() or 1, int(os.environ.get("OMP_NUM_THREADS", "1024")))
        torch.set_num_threads(cores)
        q1, s1 = orc.quantize_fp8_block(w1_cpu)
        q2, s2 = orc.quantize_fp8_block(w2_cpu)
        xc = x_cpu.to(w.dtype).requires_grad_(True)
        t0 = time.perf_counter()
        w1d = orc.dequantize_fp8_block(q1, s1)
        w2d = orc.dequantize_fp8_block(q2, s2)
        out = orc.grouped_mlp(xc, w1d, w2d, counts)
        out.backward(dy_cpu.to(w.dtype))
        cdt = time.perf_counter() - t0
        result["cpu_baseline"] = {"value": flops / cdt / 1e12, "unit": "TFLOP/s", "cores": cores,
                                  "kind": "port", "seconds": cdt,
                                  "sample": "oracle (dequantise, fp32 matmul per expert) fwd + dX on the "
                                            "same %d rows and weights; 1 repetition" % N}
    print(json.dumps(result))


def main():
    args = parse_args()
    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) != 1:
        print("bench.py measures one GPU's share of the MoE layer; this build has no multi-GPU path "
              "(run with --gpus 1)", file=sys.stderr)
        sys.exit(2)

    import torch
    import __graft_entry__ as entry

    entry.ensure_built()
    pkg = entry.load_package()
    configs = pkg.configs
    assert torch.cuda.is_available(), "bench.py needs a GPU"
    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)
    if args.workload == "dsv3_shard_fp8":
        return run_fp8_shard(args, torch, pkg, dev)
    w = configs.WORKLOADS[args.workload]

    # ---- inputs resident in HBM before the timed region ------------------------------------------
    S = w.tokens // w.batch
    E, H, F = w.experts, w.hidden, w.ffn
    cfg = pkg.MoEConfig(hidden_size=H, num_moe_experts=E, moe_ffn_hidden_size=F,
                        moe_router_topk=w.topk, moe_router_load_balancing_type="aux_loss",
                        moe_aux_loss_coeff=0.01, moe_token_dispatcher_type=args.dispatcher,
                        params_dtype=w.dtype, moe_shared_expert_intermediate_size=w.shared_ffn,
                        moe_shared_expert_overlap=bool(args.shared_overlap and w.shared_ffn))
    torch.manual_seed(1234)
    router = pkg.GalvatronMoERouter(cfg, device=dev).train()
    mlp = pkg.GalvatronMoEMLP(cfg, device=dev).train()
    cpu_inputs = None
    g = torch.Generator(device=dev).manual_seed(1234)
    if args.device_inputs or args.operands == "zeros":
        x = torch.randn(S, w.batch, H, generator=g, device=dev, dtype=torch.float32).to(w.dtype)
        dy = torch.randn(S, w.batch, H, generator=g, device=dev, dtype=torch.float32).to(w.dtype)
        data = "synthetic (device generator)"
    else:
        # CPU generator, fp32, fixed order (x, w_r, w1, w2, dy, shared), then cast: the CPU baseline
        # below computes on these very tensors
        cpu_inputs = configs.make_inputs(w, seed=1234)
        x, dy = cpu_inputs["x"].to(dev), cpu_inputs["dy"].to(dev)
        with torch.no_grad():
            router.router.weight.copy_(cpu_inputs["w_r"].to(dev))
            mlp.experts.weight1.view(E, H, 2 * F).copy_(cpu_inputs["w1"].to(dev))
            mlp.experts.weight2.view(E, F, H).copy_(cpu_inputs["w2"].to(dev))
            if w.shared_ffn:
                mlp.shared_experts.linear_fc1.weight.copy_(cpu_inputs["shared_w1"].t().to(dev))
                mlp.shared_experts.linear_fc2.weight.copy_(cpu_inputs["shared_w2"].t().to(dev))
        data = "synthetic (CPU generator, seed 1234, shared with the CPU baseline)"
    logit_bias = None
    if w.zipf:
        logit_bias = configs.make_inputs(w, with_weights=False)["logit_bias"].to(dev).to(w.dtype)
    fixed_logits = None
    if args.operands == "zeros":
        fixed_logits = torch.randn(w.tokens, E, generator=g, device=dev, dtype=torch.float32).to(w.dtype)
        with torch.no_grad():
            x.zero_()
            dy.zero_()
            for prm in mlp.parameters():
                prm.zero_()
        data = "synthetic, all-zero operands (diagnostic)"
    params = list(router.parameters()) + list(mlp.parameters())
    pre_norm = None
    if args.pre_router_norm:
        pre_norm = pkg.PreRouterNorm(cfg, device=dev).train()
        params += list(pre_norm.parameters())
    x.requires_grad_(True)

    def route(h):
        if fixed_logits is not None:
            logits = fixed_logits + 0 * router.router.gating(h).view(-1, E)
            return pkg.topk_softmax_with_capacity(logits, w.topk)[:2]
        if logit_bias is None:
            return router(h)
        logits = router.router.gating(h).view(-1, E) + logit_bias
        return pkg.topk_softmax_with_capacity(logits, w.topk)[:2]

    def step():
        for p in params:
            p.grad = None
        x.grad = None
        h, residual = (x, None) if pre_norm is None else pre_norm(x)
        probs, rmap = route(h)
        out = mlp(h, residual, probs, rmap)
        out.backward(dy)
        return out

    if args.graph:
        # Autograd remembers the stream a leaf's gradient accumulation first ran on; if that is the
        # default stream, a later capture on another stream would have to pull the default stream
        # into the capture, which is not allowed.  So every step of this run, the warm-up included,
        # is issued on one side stream, and the capture uses that stream too.
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        torch.cuda.set_stream(side)
    for _ in range(args.warmup):
        step()
    torch.cuda.synchronize()

    # rows whose k-th and (k+1)-th largest logits are equal in the router's dtype: there the choice
    # depends on the tie rule (lowest expert index here; torch.topk leaves it open)
    with torch.no_grad():
        h0 = x if pre_norm is None else pre_norm(x)[0]
        lg = router.router.gating(h0).view(-1, E) if fixed_logits is None else fixed_logits
        if logit_bias is not None:
            lg = lg + logit_bias
        tie_rows = 0
        if w.topk < E:
            top = torch.topk(lg.float(), w.topk + 1, dim=1)[0]
            tie_rows = int((top[:, w.topk - 1] == top[:, w.topk]).sum())
        del h0, lg

    marks = [torch.cuda.Event(enable_timing=True) for _ in range(args.steps + 1)]

    def timed_steps():
        t0 = time.perf_counter()
        for i in range(args.steps):
            marks[i].record()
            step()
        marks[args.steps].record()
        torch.cuda.synchronize()
        return time.perf_counter() - t0

    dt = timed_steps()
    per_step = sorted(marks[i].elapsed_time(marks[i + 1]) for i in range(args.steps))
    median_ms = per_step[len(per_step) // 2]
    # per-kernel times from a second pass outside the timed region
    timer = KernelTimer(torch, pkg.ops)
    timer.install()
    timer.enabled = True
    with torch.no_grad():
        for _ in range(args.steps):
            launch_by_launch(torch, pkg.ops, w, router.router.weight.detach(), mlp.experts, mlp.shared_experts,
                             None if pre_norm is None else pre_norm.pre_router_norm, x, dy, fixed_logits, logit_bias)
    torch.cuda.synchronize()
    timer.uninstall()
    eager = None
    if args.graph:
        # the same step recorded once and replayed: no launch gaps between its kernels
        eager = {"ms_per_step": round(dt * 1e3 / args.steps, 3), "ms_per_step_median": round(median_ms, 3)}
        for p in params:
            p.grad = None
        x.grad = None
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            step()
        for _ in range(args.warmup):
            graph.replay()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for i in range(args.steps):
            marks[i].record()
            graph.replay()
        marks[args.steps].record()
        torch.cuda.synchronize()
        dt = time.perf_counter() - t0
        per_step = sorted(marks[i].elapsed_time(marks[i + 1]) for i in range(args.steps))
        median_ms = per_step[len(per_step) // 2]
        del graph

    # One plain device copy of known size (1 GiB read + 1 GiB written), outside the timed region:
    # the reference point for scaling FETCH_SIZE / WRITE_SIZE counters of a profiled run.
    calib = torch.empty(1 << 28, dtype=torch.float32, device=dev)
    calib_dst = torch.empty_like(calib)
    calib_dst.copy_(calib)
    torch.cuda.synchronize()
    del calib, calib_dst

    # permute_rows once more on inputs that are not in any cache (outside the timed region): in the
    # step its rows come straight from the router's read of x, which leaves part of them in the
    # last-level cache.  A 1 GiB fill between calls evicts them.
    cold_ms = []
    with torch.no_grad():
        x2 = x.detach().view(-1, H)
        rmap0 = route(x.detach() if pre_norm is None else pre_norm(x.detach())[0])[1]
        plan = pkg.ops.permute_plan(rmap0, w.routed_rows, want_sorted=False)
        evict = torch.empty(1 << 28, dtype=torch.float32, device=dev)
        for _ in range(6):
            evict.fill_(1.0)
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            pkg.ops.permute_rows(x2, plan.dst_map, w.routed_rows)
            e1.record()
            torch.cuda.synchronize()
            cold_ms.append(e0.elapsed_time(e1))
        del evict, plan, rmap0, x2
    cold_ms = sorted(cold_ms[1:])   # the first call also pays the allocator

    ms_per_step = dt * 1e3 / args.steps
    flops = w.gemm_flops()
    value = flops / (dt / args.steps) / 1e12
    dkey = {torch.bfloat16: "bf16", torch.float16: "f16", torch.float32: "f32"}[w.dtype]
    peak = MFMA_PEAK[dkey]

    agg = timer.summary()
    gemm = {k: v for k, v in agg.items() if v["name"].startswith("gmm_")}
    gemm_ms = sum(v["ms"] for v in gemm.values()) / args.steps
    gemm_flops = sum(v["work"] * v["calls"] for v in gemm.values()) / args.steps
    kernels = {}
    for k, v in sorted(agg.items()):
        avg = v["ms"] / v["calls"]
        ent = {"calls_per_step": v["calls"] / args.steps, "avg_ms": round(avg, 4)}
        if v["work"]:
            ent["tflops"] = round(v["work"] / (avg * 1e-3) / 1e12, 1)
        kernels[k] = ent
    # dominant kernel: the forward fc1 grouped GEMM (NN), the largest single launch.  Its HBM-side
    # bytes cannot be read inside this process (they come from rocprofv3 counter runs of this very
    # command, FETCH_SIZE and WRITE_SIZE scaled by what the 1 GiB copy above reads back), so
    # `traffic` stays null here and the profiled figure is quoted with its source.
    profiled_traffic = {("mixtral", "gmm_NN+glu 32768x4096x28672"):
                        {"bytes_per_launch": 17.4e9, "source": "profiles/bench_mixtral_hbm_traffic.md"}}
    dom_key = max(gemm, key=lambda k: gemm[k]["work"] * (1 if k.startswith("gmm_NN") else 0.5)) if gemm else None
    roofline = None
    if dom_key:
        d = gemm[dom_key]
        ach = d["work"] / (d["ms"] / d["calls"] * 1e-3) / 1e12
        kernel = "gmm_f32_kernel " if w.dtype == torch.float32 else "gmm_rows_kernel "
        roofline = {"bound": "mfma", "kernel": kernel + dom_key, "achieved": round(ach, 1),
                    "peak": peak, "unit": "TFLOP/s", "frac": round(ach / peak, 4),
                    "traffic": None,
                    "traffic_profiled": profiled_traffic.get((w.name, dom_key)),
                    "all_gmm_launches": {"achieved": round(gemm_flops / (gemm_ms * 1e-3) / 1e12, 1),
                                         "frac": round(gemm_flops / (gemm_ms * 1e-3) / 1e12 / peak, 4),
                                         "ms_per_step": round(gemm_ms, 3)}}

    es = torch.finfo(w.dtype).bits // 8
    row_bytes = w.tokens * H * es
    n_rows_bytes = w.routed_rows * H * es
    permute = {"permute_rows": hbm_entry(agg, "permute_rows", w.permute_bytes()),
               # two launches per step share the label: the combine and the backward of the permute
               "unpermute_rows": hbm_entry(agg, "unpermute_rows", w.unpermute_bytes() +
                                           (row_bytes / 2 if (pre_norm is not None or w.shared_ffn) else 0)),
               # reads the token's gradient row and the k forward-input rows, writes k rows and the
               # gate gradients: (T + 2N) * H * sizeof + T * E * sizeof(probs)
               "unpermute_rows_bwd": hbm_entry(agg, "unpermute_rows_bwd",
                                               row_bytes + 2 * n_rows_bytes + w.tokens * E * es)}
    if permute["permute_rows"] is not None:
        cold = cold_ms[len(cold_ms) // 2]
        permute["permute_rows"]["cold_input"] = {
            "avg_ms": round(cold, 4), "achieved": round(w.permute_bytes() / (cold * 1e-3) / 1e9, 1),
            "frac": round(w.permute_bytes() / (cold * 1e-3) / 1e9 / HBM_PEAK_GBPS, 4),
            "note": "median of 5 calls, a 1 GiB fill before each"}
    if pre_norm is not None:
        permute["rmsnorm_fwd"] = hbm_entry(agg, "rmsnorm_fwd", 2 * row_bytes)   # x read, y written
        # dy, x and the residual branch's gradient read, dx written
        permute["rmsnorm_bwd"] = hbm_entry(agg, "rmsnorm_bwd", 4 * row_bytes)

    result = {
        "metric": "MoE layer fwd+bwd TFLOP/s (1 GPU, % MFMA peak); permute GB/s (% HBM)",
        "value": round(value, 2),
        "unit": "TFLOP/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms_per_step, 3),
        "ms_per_step_median": round(median_ms, 3),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": dkey,
        "data": data,
        "config": {"workload": "%s: MoE layer fwd+bwd, T=%d (batch %d) H=%d F=%d E=%d top-%d, %s "
                               "dispatcher, aux-loss router" % (w.name, w.tokens, w.batch, H, F, E,
                                                                w.topk, args.dispatcher) +
                               (", shared experts %d" % w.shared_ffn if w.shared_ffn else "") +
                               (" on their own stream" if args.shared_overlap and w.shared_ffn else "") +
                               (", pre-router RMSNorm and residual add included" if pre_norm else ""),
                   "flops_per_step": flops,
                   "tie_rows": tie_rows,
                   "launch": "HIP graph replay" if args.graph else "eager",
                   "per_kernel_events": "a second pass of the same number of steps, issued launch by "
                                        "launch outside the timed region"},
        "pct_mfma_peak": round(100 * value / peak, 2),
        "roofline": roofline,
        "permute": permute,
        "kernels": kernels,
    }
    if eager is not None:
        result["eager"] = eager
    if args.blas_reference:
        result["blas_reference"] = blas_reference(torch, w, dev, zeros=args.operands == "zeros")
    if not args.no_cpu_baseline:
        result["cpu_baseline"] = cpu_baseline(w, min(args.cpu_tokens, w.tokens), args.dispatcher,
                                              cpu_inputs)
    print(json.dumps(result))


if __name__ == "__main__":
    main()
