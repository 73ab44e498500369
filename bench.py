#!/usr/bin/env python3
"""Benchmark of the transformer-layer hot path on one MI355X.

Headline workload (`config.workload`): attention core forward + backward, GQA 32 query / 8 KV heads,
head_dim 128, one sequence of 8192 tokens, causal, bf16, fp32 softmax.  One step = one forward and
one backward pass over synthetic N(0,1) inputs already resident in HBM.  `value` is
14 * d * n_q * P / time (P = allowed (query, key) pairs per head), i.e. the algorithmic TFLOP/s.

The JSON line also carries
  roofline      the dominant kernel of the step, timed live with HIP events on the launch stream
  cpu_baseline  the reference's operation order (CPU oracle, plain torch) timed on the host cores
                on a bounded sample of the same workload
  extra         the other quantities of the metric: per-kernel attention times, config-2 / config-3
                attention, RMSNorm / SwiGLU / rotary GB/s at the config-4 sizes, decode-attention GB/s
                at the config-5 per-layer shape.
"""

import argparse
import json
import math
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

PEAK_BF16_TFLOPS = 2500.0   # MI355X dense bf16 MFMA, vendor figure
PEAK_HBM_GBS = 8000.0       # MI355X HBM3E, vendor figure

# HBM bytes per launch of the attention kernels on the headline workload come from rocprofv3 FETCH_SIZE / WRITE_SIZE runs
# whose figures are kept in this file together with a hash of the kernel sources they were measured on; the figure is
# reported only while the sources are unchanged.
TRAFFIC_FILE = os.path.join(ROOT, "profiles", "attention_fwd_bwd_gqa32x8_d128_s8192_hbm_traffic.json")
ATTENTION_SOURCES = ("attn_common.h", "attn_fwd.hip", "attn_bwd.hip", "attn_host.hip", "common.h")


def attention_sources_hash():
    import hashlib
    h = hashlib.sha256()
    for name in ATTENTION_SOURCES:
        with open(os.path.join(ROOT, "scaling_amd", "csrc", name), "rb") as f:
            h.update(f.read())
    return h.hexdigest()


def measured_traffic_bytes(kernel):
    """HBM bytes per launch of `kernel` from the counter runs, or (None, reason) when there is no current measurement."""
    try:
        with open(TRAFFIC_FILE) as f:
            data = json.load(f)
    except (OSError, ValueError):
        return None, "no counter measurement on file"
    if data.get("sources_sha256") != attention_sources_hash():
        return None, "the kernel sources changed after the counters were taken"
    k = data.get("kernels", {}).get(kernel)
    if not k:
        return None, "kernel not in the counter file"
    cal = data["calibration"]
    return 1024.0 * (cal["fetch_scale"] * k["fetch_size_kib"] + cal["write_scale"] * k["write_size_kib"]), None


def causal_pairs(cu):
    return sum((b - a) * (b - a + 1) // 2 for a, b in zip(cu[:-1], cu[1:]))


def time_gpu(fn, steps, warmup, stats=None):
    """Average milliseconds per call over exactly `steps` calls bracketed by events on the current stream (the figure
    `value` / `ms_per_step` are built from).  With a dict in `stats` every call is also bracketed by its own pair of
    events and the median, minimum and maximum of the per-call times are stored there."""
    import torch
    for _ in range(warmup):
        fn()
    start, stop = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    marks = [torch.cuda.Event(enable_timing=True) for _ in range(steps + 1)] if stats is not None else None
    torch.cuda.synchronize()
    start.record()
    for i in range(steps):
        if marks is not None:
            marks[i].record()
        fn()
    if marks is not None:
        marks[steps].record()
    stop.record()
    torch.cuda.synchronize()
    if marks is not None:
        per_call = sorted(marks[i].elapsed_time(marks[i + 1]) for i in range(steps))
        stats.update(median=per_call[len(per_call) // 2], min=per_call[0], max=per_call[-1])
    return start.elapsed_time(stop) / steps


def time_gpu_median(fn, steps, warmup):
    """Median milliseconds per call (each call bracketed by its own events on the current stream)."""
    st = {}
    time_gpu(fn, max(steps, 20), warmup, st)
    return st["median"]


def time_gpu_graph(fn, steps, warmup):
    """Average milliseconds per call with the calls replayed from one HIP graph, so that a launch that takes the
    host longer than the kernel takes the GPU (the 20-30 us bandwidth kernels) is still timed on the GPU side.
    Median of five replays; falls back to eager timing if the calls cannot be captured."""
    import torch
    try:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for _ in range(max(warmup, 2)):
                fn()
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for _ in range(steps):
                fn()
        times = []
        for _ in range(5):
            start, stop = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            torch.cuda.synchronize()
            start.record()
            graph.replay()
            stop.record()
            torch.cuda.synchronize()
            times.append(start.elapsed_time(stop) / steps)
        del graph
        return sorted(times)[len(times) // 2]
    except Exception as exc:  # noqa: BLE001 - any capture problem: measure eagerly instead
        print(f"[bench] graph timing unavailable ({type(exc).__name__}: {exc}); timing eagerly", file=sys.stderr)
        torch.cuda.synchronize()
        return time_gpu(fn, steps, warmup)


def time_rotating(make_call, n_sets, steps, warmup):
    """Average milliseconds per call over a HIP-graph replay that cycles through n_sets distinct sets of input buffers
    (and keeps n_sets results alive, so the outputs land in distinct buffers too): with the sets totalling more than
    twice the 256 MB Infinity Cache every call streams from and to HBM, which replaying one set of 134 - 201 MB does
    not guarantee.  make_call(k) returns the zero-argument call for buffer set k."""
    calls = [make_call(k) for k in range(n_sets)]
    keep = [None] * n_sets
    counter = [0]

    def one():
        k = counter[0] % n_sets
        counter[0] += 1
        keep[k] = calls[k]()

    return time_gpu_graph(one, max(steps, 2 * n_sets), max(warmup, n_sets))


def random_docs_cu(total, lo, hi, seed):
    """Cumulative document lengths: lengths uniform in [lo, hi], the last one truncated so they sum to `total`."""
    import torch
    g = torch.Generator().manual_seed(seed)
    cu = [0]
    while cu[-1] < total:
        cu.append(min(total, cu[-1] + int(torch.randint(lo, hi + 1, (1,), generator=g))))
    return torch.tensor(cu, dtype=torch.int32)


def _rotary_tables(dim, max_seq, base, device):
    """cos / sin tables [max_seq, dim] in bf16 from the product's own RotaryEmbedding module."""
    import torch
    from scaling_amd.config import RotaryConfig
    from scaling_amd.nn import RotaryEmbedding
    return RotaryEmbedding(RotaryConfig(dimensions=dim, max_seq_length=max_seq, base=base), torch.device(device), torch.bfloat16).tables()


def _check_sampled_rows(q, k, v, do, o, lse, dq, dk, dv, cu_list, scale):
    """Finite outputs plus one sampled row per stage against plain fp32 torch arithmetic on that row."""
    import torch
    for name, t in (("o", o), ("lse", lse), ("dq", dq), ("dk", dk), ("dv", dv)):
        assert bool(torch.isfinite(t.float()).all()), f"attention {name} has non-finite values"
    n_rep = q.shape[1] // k.shape[1]
    qf, kf, vf, dof, of = (t.float() for t in (q, k, v, do, o))

    def close(name, got, want):
        err = (got.float() - want).abs().max().item()
        tol = 0.03 * max(1.0, want.abs().max().item())
        assert err <= tol, f"attention {name}: sampled row off by {err:.3e} (tolerance {tol:.3e})"

    # last query of the last document, head 0: attends keys [lo, t]
    t, lo, h = cu_list[-1] - 1, cu_list[-2], 0
    p = torch.softmax((kf[lo:t + 1, 0] @ qf[t, h]) * scale, 0)
    close("o row", o[t, h], p @ vf[lo:t + 1, 0])
    ds = p * (vf[lo:t + 1, 0] @ dof[t, h] - (dof[t, h] * of[t, h]).sum())
    close("dq row", dq[t, h], scale * (ds @ kf[lo:t + 1, 0]))
    # first key of the first document, KV head 0: every query of that document and of the group's heads attends it
    hi = cu_list[1]
    dk_row, dv_row = torch.zeros_like(kf[0, 0]), torch.zeros_like(vf[0, 0])
    for hh in range(n_rep):
        pj = torch.exp((qf[:hi, hh] @ kf[0, 0]) * scale - lse[hh, :hi])              # P[:, key 0] from the saved log-sum-exp
        dsj = pj * (dof[:hi, hh] @ vf[0, 0] - (dof[:hi, hh] * of[:hi, hh]).sum(-1))
        dv_row += pj @ dof[:hi, hh]
        dk_row += scale * (dsj @ qf[:hi, hh])
    close("dv row", dv[0, 0], dv_row)
    close("dk row", dk[0, 0], dk_row)


def attention_case(b, s, nq, nkv, d, cu_list, steps, warmup, seed=0, rotary=False):
    """Times forward, backward stages and the whole step for one attention workload."""
    import torch
    from scaling_amd import ops
    dev = "cuda"
    g = torch.Generator().manual_seed(seed)
    T = b * s
    q = torch.randn(T, nq, d, generator=g).bfloat16().to(dev)
    k = torch.randn(T, nkv, d, generator=g).bfloat16().to(dev)
    v = torch.randn(T, nkv, d, generator=g).bfloat16().to(dev)
    do = torch.randn(T, nq, d, generator=g).bfloat16().to(dev)
    cu = torch.tensor(cu_list, dtype=torch.int32, device=dev)
    scale = 1.0 / math.sqrt(d)
    pairs = causal_pairs(cu_list)
    rot = None
    if rotary:
        cos_tab, sin_tab = _rotary_tables(d, s, 500000, dev)
        pos = torch.zeros(T, dtype=torch.int64)
        for a_, b_ in zip(cu_list[:-1], cu_list[1:]):
            pos[a_:b_] = torch.arange(b_ - a_)
        pos = pos.to(dev)
        rot = (cos_tab, sin_tab, pos, pos)

    o, lse = ops.attention_forward(q, k, v, cu, None, True, scale)
    dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
    from scaling_amd import _lib
    ws = torch.empty(_lib.load().mi_attn_bwd_workspace_bytes_kv(T, T, nq, nkv, d) // 4, dtype=torch.float32, device=dev)
    bufs = (dq, dk, dv, ws)
    # before anything is timed: every output finite, and one row of each (the last query's o and dq, the first key's
    # dk and dv) equal to a plain fp32 evaluation of that row (the full comparison with the oracle is tests/'s job)
    ops.attention_backward(do, q, k, v, o, lse, cu, None, True, scale, buffers=bufs)
    _check_sampled_rows(q, k, v, do, o, lse, dq, dk, dv, cu_list, scale)

    def fwd():
        ops.attention_forward(q, k, v, cu, None, True, scale)

    def fwd_rot():
        ops.attention_forward(q, k, v, cu, None, True, scale, rotary=rot)

    def bwd(flags=0):
        ops.attention_backward(do, q, k, v, o, lse, cu, None, True, scale, flags=flags, buffers=bufs)

    def step():
        fwd()
        bwd()

    def step_precise():
        o2, lse2 = ops.attention_forward(q, k, v, cu, None, True, scale, precise=True)
        ops.attention_backward(do, q, k, v, o2, lse2, cu, None, True, scale, buffers=bufs, precise=True)

    res = {"pairs_per_head": pairs}
    res["ms_step"] = time_gpu(step, steps, warmup)              # mean over exactly `steps` steps: the contract's figure
    st = {}
    time_gpu(step, max(steps, 20), 1, st)                       # the same again with every step bracketed on its own
    res["ms_step_median"], res["ms_step_min"], res["ms_step_max"] = st["median"], st["min"], st["max"]
    res["ms_step_graph"] = time_gpu_graph(step, steps, warmup)
    res["ms_fwd"] = time_gpu_median(fwd, steps, warmup)
    res["ms_bwd_delta"] = time_gpu_median(lambda: bwd(16), steps, 1)
    res["ms_bwd_dkdv"] = time_gpu_median(lambda: bwd(32), steps, 1)
    res["ms_bwd_dq"] = time_gpu_median(lambda: bwd(64), steps, 1)
    res["ms_bwd_dkdv_dq"] = time_gpu_median(lambda: bwd(32 | 64), steps, 1)   # both kinds of blocks in one launch, as a backward pass has them
    # accuracy mode (MI_ATTN_SPLIT_P): the mode whose outputs and gradients meet max-abs 2e-2 / mean-rel 1e-3 literally
    res["ms_step_precise"] = time_gpu(step_precise, steps, warmup)
    step()                                                      # leave the default mode's results in the buffers
    if rot is not None:
        res["ms_fwd_fused_rotary"] = time_gpu(fwd_rot, steps, warmup)
        # training step with the rotary embedding as ops.attention runs it: k rotated by one stand-alone launch, q
        # while the forward kernel loads it (the rotated q is written out for the backward), dq and dk rotated back
        # inside the backward kernels
        cos_t, sin_t, pos_t, _ = rot

        def step_rotary():
            kr = ops._rotary_launch(k, cos_t, sin_t, pos_t, 0, False)
            o2, lse2, qr = ops.attention_forward(q, kr, v, cu, None, True, scale, rotary=(cos_t, sin_t, pos_t, None), return_rotated_q=True)
            ops.attention_backward(do, qr, kr, v, o2, lse2, cu, None, True, scale, buffers=bufs, rotary=rot)

        res["ms_step_with_rotary"] = time_gpu(step_rotary, steps, warmup)
        res["tflops_step_with_rotary"] = 14 * d * nq * pairs / (res["ms_step_with_rotary"] * 1e-3) / 1e12
    flops_unit = d * nq * pairs
    res["tflops_fwd"] = 4 * flops_unit / (res["ms_fwd"] * 1e-3) / 1e12
    res["tflops_step"] = 14 * flops_unit / (res["ms_step"] * 1e-3) / 1e12
    res["tflops_step_graph"] = 14 * flops_unit / (res["ms_step_graph"] * 1e-3) / 1e12
    res["tflops_step_precise"] = 14 * flops_unit / (res["ms_step_precise"] * 1e-3) / 1e12
    res["precise_over_default_time"] = res["ms_step_precise"] / res["ms_step"]
    res["frac_of_bf16_peak_step"] = res["tflops_step"] / PEAK_BF16_TFLOPS
    return res


def attention_float32_case(steps, warmup):
    """The float32 attention core (the reference's default precision; exact-fp32 kernels on the fp32 matrix pipe) at GQA
    32 / 8 heads of 128, one causal sequence of 4096 tokens: forward + backward time and the fraction of the fp32 MFMA peak."""
    import torch
    from scaling_amd import ops
    dev = "cuda"
    g = torch.Generator().manual_seed(5)
    T, nq, nkv, d = 4096, 32, 8, 128
    q = torch.randn(T, nq, d, generator=g).to(dev)
    k = torch.randn(T, nkv, d, generator=g).to(dev)
    v = torch.randn(T, nkv, d, generator=g).to(dev)
    do = torch.randn(T, nq, d, generator=g).to(dev)
    cu = torch.tensor([0, T], dtype=torch.int32, device=dev)
    scale = 1.0 / math.sqrt(d)
    o, lse = ops.attention_forward(q, k, v, cu, None, True, scale)
    bufs = None

    def step():
        o2, lse2 = ops.attention_forward(q, k, v, cu, None, True, scale)
        ops.attention_backward(do, q, k, v, o2, lse2, cu, None, True, scale, buffers=bufs)

    ms = time_gpu(step, max(3, steps // 4), 1)
    ms_fwd = time_gpu(lambda: ops.attention_forward(q, k, v, cu, None, True, scale), max(3, steps // 4), 1)
    flops = 14 * d * nq * (T * (T + 1) // 2)
    return {"ms_step": ms, "ms_fwd": ms_fwd, "tflops_step": flops / (ms * 1e-3) / 1e12,
            "frac_of_fp32_mfma_peak": flops / (ms * 1e-3) / 1e12 / 157.3,
            "note": "float32 q / k / v / o, fp32 probabilities"}


def bandwidth_cases(steps, warmup):
    """RMSNorm / SwiGLU / rotary at the config-4 sizes and decode attention at the config-5 layer shape."""
    import torch
    from scaling_amd import ops
    dev = "cuda"
    out = {}
    g = torch.Generator().manual_seed(1)
    N, H, I = 8192, 4096, 14336
    w = torch.ones(H, dtype=torch.bfloat16, device=dev)
    bias = torch.zeros(H, dtype=torch.bfloat16, device=dev)
    # The norm and rotary working sets (134 - 201 MB) fit the 256 MB Infinity Cache: "GBs" cycles through 8 distinct
    # buffer sets (0.5 - 1.1 GB of inputs), "GBs_same_buffers" replays one set (part of its traffic can be cache hits)
    n_sets = 8
    xs = [torch.randn(N, H, generator=g).bfloat16().to(dev) for _ in range(n_sets)]
    dys = [torch.randn(N, H, generator=g).bfloat16().to(dev) for _ in range(n_sets)]
    x, dy = xs[0], dys[0]
    _, ln_stats = ops.layer_norm_forward(x, w, bias, 1e-5, save_stats=True)   # as the autograd function runs it
    stats = [ops.layer_norm_forward(xi, w, bias, 1e-5, save_stats=True)[1] for xi in xs]

    def both(name, nbytes, rotating, same):
        ms = time_rotating(rotating, n_sets, steps, warmup)
        ms_same = time_gpu_graph(same, steps, warmup)
        out[name] = {"ms": ms, "GBs": nbytes / ms / 1e6, "ms_same_buffers": ms_same, "GBs_same_buffers": nbytes / ms_same / 1e6}

    both("rmsnorm_fwd", 2 * N * H * 2, lambda k: (lambda: ops.rms_norm_forward(xs[k], w, 1e-5)), lambda: ops.rms_norm_forward(x, w, 1e-5))
    both("rmsnorm_bwd", 3 * N * H * 2, lambda k: (lambda: ops.rms_norm_backward(xs[k], w, dys[k], 1e-5)),
         lambda: ops.rms_norm_backward(x, w, dy, 1e-5))
    both("layernorm_fwd", 2 * N * H * 2, lambda k: (lambda: ops.layer_norm_forward(xs[k], w, bias, 1e-5)),
         lambda: ops.layer_norm_forward(x, w, bias, 1e-5))
    both("layernorm_bwd", 3 * N * H * 2, lambda k: (lambda: ops.layer_norm_backward(xs[k], w, dys[k], 1e-5, True, stats[k])),
         lambda: ops.layer_norm_backward(x, w, dy, 1e-5, True, ln_stats))
    del xs, dys, stats
    # the same kernels on 8 x the rows (one launch streams 1.1 - 1.6 GB): the launch's ramp and tail and the dweight
    # reduction launch weigh an eighth as much, so this is the steady-state rate of the same code
    N8 = 8 * N
    x8 = torch.randn(N8, H, generator=g).bfloat16().to(dev)
    dy8 = torch.randn(N8, H, generator=g).bfloat16().to(dev)
    st8 = ops.layer_norm_forward(x8, w, bias, 1e-5, save_stats=True)[1]
    for name, nbytes, call in (
            ("rmsnorm_fwd", 2 * N8 * H * 2, lambda: ops.rms_norm_forward(x8, w, 1e-5)),
            ("rmsnorm_bwd", 3 * N8 * H * 2, lambda: ops.rms_norm_backward(x8, w, dy8, 1e-5)),
            ("layernorm_fwd", 2 * N8 * H * 2, lambda: ops.layer_norm_forward(x8, w, bias, 1e-5)),
            ("layernorm_bwd", 3 * N8 * H * 2, lambda: ops.layer_norm_backward(x8, w, dy8, 1e-5, True, st8))):
        ms8 = time_gpu_graph(call, max(5, steps // 2), 2)
        out[name]["ms_8x_rows"] = ms8
        out[name]["GBs_8x_rows"] = nbytes / ms8 / 1e6
    del x8, dy8, st8
    a = torch.randn(N, I, generator=g).bfloat16().to(dev)
    gate = torch.randn(N, I, generator=g).bfloat16().to(dev)
    dout = torch.randn(N, I, generator=g).bfloat16().to(dev)
    ms = time_gpu_graph(lambda: ops.swiglu_forward(a, gate), steps, warmup)
    out["swiglu_fwd"] = {"ms": ms, "GBs": 3 * N * I * 2 / ms / 1e6}
    ms = time_gpu_graph(lambda: ops.swiglu_backward(a, gate, dout), steps, warmup)
    out["swiglu_bwd"] = {"ms": ms, "GBs": 5 * N * I * 2 / ms / 1e6}
    ms = time_gpu_graph(lambda: ops.gelu_forward(a), steps, warmup)
    out["gelu_fwd"] = {"ms": ms, "GBs": 2 * N * I * 2 / ms / 1e6}
    ms = time_gpu_graph(lambda: ops.gelu_backward(a, dout), steps, warmup)
    out["gelu_bwd"] = {"ms": ms, "GBs": 3 * N * I * 2 / ms / 1e6}
    del a, gate, dout
    rows, vocab = 4096, 128256                      # config-5 vocabulary
    logits = (torch.randn(rows, vocab, generator=torch.Generator(device=dev).manual_seed(2), device=dev) * 2).bfloat16()
    targets = torch.randint(0, vocab, (rows,), device=dev)
    row_scale = torch.full((rows,), 1.0 / rows, device=dev)
    dlogits = torch.empty_like(logits)
    ms = time_gpu_graph(lambda: ops.cross_entropy_forward(logits, targets), steps, warmup)
    out["cross_entropy_fwd"] = {"ms": ms, "GBs": rows * vocab * 2 / ms / 1e6}
    ms = time_gpu_graph(lambda: ops.cross_entropy_forward(logits, targets, row_scale, dlogits), steps, warmup)
    out["cross_entropy_fwd_bwd"] = {"ms": ms, "GBs": 2 * rows * vocab * 2 / ms / 1e6}
    del logits, dlogits
    nq, nkv, d = 32, 8, 128
    qks = [torch.randn(N, nq + nkv, d, generator=g).bfloat16().to(dev) for _ in range(n_sets)]
    cos, sin = _rotary_tables(d, 8192, 500000, dev)
    pos = torch.arange(N, dtype=torch.int64, device=dev) % 4096
    both("rotary", 2 * N * (nq + nkv) * d * 2 + 8 * N, lambda k: (lambda: ops.rotary_embedding(qks[k], cos, sin, pos)),
         lambda: ops.rotary_embedding(qks[0], cos, sin, pos))
    qk8 = torch.randn(8 * N, nq + nkv, d, generator=g).bfloat16().to(dev)
    pos8 = torch.arange(8 * N, dtype=torch.int64, device=dev) % 4096
    ms8 = time_gpu_graph(lambda: ops.rotary_embedding(qk8, cos, sin, pos8), max(5, steps // 2), 2)
    out["rotary"]["ms_8x_rows"] = ms8
    out["rotary"]["GBs_8x_rows"] = (2 * 8 * N * (nq + nkv) * d * 2 + 8 * 8 * N) / ms8 / 1e6
    del qks, qk8, pos8
    B, ctx, max_ctx = 32, 4096, 4352
    # head-major storage viewed as [batch, token, kv head, d]: the layout scaling_amd.nn.KVCache allocates
    kc = torch.randn(B, nkv, max_ctx, d, generator=g).bfloat16().to(dev).transpose(1, 2)
    vc = torch.randn(B, nkv, max_ctx, d, generator=g).bfloat16().to(dev).transpose(1, 2)
    q1 = torch.randn(B, nq, d, generator=g).bfloat16().to(dev)
    ctx_len = torch.full((B,), ctx, dtype=torch.int32, device=dev)
    wsd = ops.decode_workspace(B, nq, d, max_ctx, dev)
    od = torch.empty_like(q1)
    ms = time_gpu_graph(lambda: ops.decode_attention(q1, kc, vc, ctx_len, workspace=wsd, out=od), steps, warmup)
    out["decode_attention"] = {"ms": ms, "GBs": 2 * B * ctx * nkv * d * 2 / ms / 1e6, "batch": B, "ctx": ctx}
    # what a plain device copy of 1 GiB reaches on this box: the practical ceiling of a one-in one-out stream
    src = torch.empty(1 << 30, dtype=torch.uint8, device=dev).fill_(1)
    dst = torch.empty_like(src)
    ms = time_gpu_graph(lambda: dst.copy_(src), max(5, steps // 2), 2)
    out["device_copy_1GiB"] = {"ms": ms, "GBs": 2 * (1 << 30) / ms / 1e6}
    del src, dst
    for v_ in out.values():
        v_["frac_of_hbm_peak"] = v_["GBs"] / PEAK_HBM_GBS
        if "GBs_8x_rows" in v_:
            v_["frac_of_hbm_peak_8x_rows"] = v_["GBs_8x_rows"] / PEAK_HBM_GBS
    return out


def profile_kernels(repeats=3):
    """Each HBM-bound kernel a few times, eagerly, at the sizes bandwidth_cases() times them at, plus a plain 1 GiB device
    copy: the run that rocprofv3 --pmc FETCH_SIZE / WRITE_SIZE passes are taken over (the copy gives the scale of the
    counters).  Returns the algorithmic bytes per launch by kernel family."""
    import torch
    from scaling_amd import ops
    dev = "cuda"
    g = torch.Generator().manual_seed(1)
    N, H, I = 8192, 4096, 14336
    w = torch.ones(H, dtype=torch.bfloat16, device=dev)
    bias = torch.zeros(H, dtype=torch.bfloat16, device=dev)
    x = torch.randn(N, H, generator=g).bfloat16().to(dev)
    dy = torch.randn(N, H, generator=g).bfloat16().to(dev)
    _, stats = ops.layer_norm_forward(x, w, bias, 1e-5, save_stats=True)
    a = torch.randn(N, I, generator=g).bfloat16().to(dev)
    gate = torch.randn(N, I, generator=g).bfloat16().to(dev)
    dout = torch.randn(N, I, generator=g).bfloat16().to(dev)
    rows, vocab = 4096, 128256
    logits = (torch.randn(rows, vocab, generator=torch.Generator(device=dev).manual_seed(2), device=dev) * 2).bfloat16()
    targets = torch.randint(0, vocab, (rows,), device=dev)
    row_scale = torch.full((rows,), 1.0 / rows, device=dev)
    dlogits = torch.empty_like(logits)
    nq, nkv, d = 32, 8, 128
    qk = torch.randn(N, nq + nkv, d, generator=g).bfloat16().to(dev)
    cos, sin = _rotary_tables(d, 8192, 500000, dev)
    pos = torch.arange(N, dtype=torch.int64, device=dev) % 4096
    B, ctx, max_ctx = 32, 4096, 4352
    kc = torch.randn(B, nkv, max_ctx, d, generator=g).bfloat16().to(dev).transpose(1, 2)
    vc = torch.randn(B, nkv, max_ctx, d, generator=g).bfloat16().to(dev).transpose(1, 2)
    q1 = torch.randn(B, nq, d, generator=g).bfloat16().to(dev)
    ctx_len = torch.full((B,), ctx, dtype=torch.int32, device=dev)
    wsd = ops.decode_workspace(B, nq, d, max_ctx, dev)
    od = torch.empty_like(q1)
    src = torch.empty(1 << 30, dtype=torch.uint8, device=dev).fill_(1)
    dst = torch.empty_like(src)
    calls = [
        ("rmsnorm_fwd", 2 * N * H * 2, lambda: ops.rms_norm_forward(x, w, 1e-5)),
        ("rmsnorm_bwd", 3 * N * H * 2, lambda: ops.rms_norm_backward(x, w, dy, 1e-5)),
        ("layernorm_fwd", 2 * N * H * 2, lambda: ops.layer_norm_forward(x, w, bias, 1e-5)),
        ("layernorm_bwd", 3 * N * H * 2, lambda: ops.layer_norm_backward(x, w, dy, 1e-5, True, stats)),
        ("swiglu_fwd", 3 * N * I * 2, lambda: ops.swiglu_forward(a, gate)),
        ("swiglu_bwd", 5 * N * I * 2, lambda: ops.swiglu_backward(a, gate, dout)),
        ("gelu_fwd", 2 * N * I * 2, lambda: ops.gelu_forward(a)),
        ("gelu_bwd", 3 * N * I * 2, lambda: ops.gelu_backward(a, dout)),
        ("cross_entropy_fwd", rows * vocab * 2, lambda: ops.cross_entropy_forward(logits, targets)),
        ("cross_entropy_fwd_bwd", 2 * rows * vocab * 2, lambda: ops.cross_entropy_forward(logits, targets, row_scale, dlogits)),
        ("rotary", 2 * N * (nq + nkv) * d * 2 + 8 * N, lambda: ops.rotary_embedding(qk, cos, sin, pos)),
        ("decode_attention", 2 * B * ctx * nkv * d * 2, lambda: ops.decode_attention(q1, kc, vc, ctx_len, workspace=wsd, out=od)),
        ("device_copy_1GiB", 2 * (1 << 30), lambda: dst.copy_(src)),
    ]
    for _, _, call in calls:
        for _ in range(repeats):
            call()
            torch.cuda.synchronize()
    return {name: nbytes for name, nbytes, _ in calls}


def layer_case(steps, warmup):
    """Config 4: one transformer layer (pre-RMSNorm, GQA 32/8 x 128, rotary, SwiGLU 14336) forward + backward on
    [2, 4096, 4096] bf16.  The projections run on PyTorch matmul; the time of this library's kernels inside the step
    is the step time minus the time of the same projections alone (forward, input gradient, weight gradient)."""
    import torch
    from scaling_amd import config as C
    from scaling_amd.layer import TransformerLayer, TransformerLayerIO
    dev = "cuda"
    bsz, seq, hidden = 2, 4096, 4096
    cfg = C.TransformerArchitectureConfig.from_dict(dict(
        vocab_size=128256, hidden_size=hidden, num_layers=1, num_attention_heads=32, attention_num_kv_heads=8,
        attention_qkv_in_one=False, norm_type="rms", mlp_type="swiglu", mlp_factor=3.5, attention_bias=False, mlp_bias=False,
        precision="bfloat16", sequence_length=seq, rotary_embedding_base=500000,
        masked_softmax={"kernel": "hip", "softmax_in_fp32": True}, weight_tying=False))
    g = torch.Generator().manual_seed(4)

    def init(w):
        w.data.copy_((torch.randn(w.shape, generator=g) * 0.02).to(w.dtype))
        return w

    layer = TransformerLayer(cfg, layer_index=0, init_method=init, device=dev)
    x = torch.randn(bsz, seq, hidden, generator=g).bfloat16().to(dev).requires_grad_()
    dy = torch.randn(bsz, seq, hidden, generator=g).bfloat16().to(dev)
    pos = torch.arange(seq, device=dev).repeat(bsz, 1)
    cu = torch.arange(0, bsz * seq + 1, seq, dtype=torch.int32, device=dev)

    def step():
        for p_ in layer.parameters():
            p_.grad = None
        x.grad = None
        out = layer(TransformerLayerIO(activations=x, position_ids=pos, cumulative_seq_lengths=cu))
        out.activations.backward(dy)

    ms = time_gpu(step, steps, warmup)
    # the projections alone: y = x W^T, dx = dy W, dW = dy^T x for each of the seven weights
    n_tok = bsz * seq
    shapes = [(hidden, hidden), (1024, hidden), (1024, hidden), (hidden, hidden), (14336, hidden), (14336, hidden), (hidden, 14336)]
    mats = [(torch.randn(n_tok, i, device=dev, dtype=torch.bfloat16), torch.randn(o, i, device=dev, dtype=torch.bfloat16),
             torch.randn(n_tok, o, device=dev, dtype=torch.bfloat16)) for o, i in shapes]

    def gemms():
        for xin, w, dout in mats:
            torch.nn.functional.linear(xin, w)
            torch.matmul(dout, w)
            torch.matmul(dout.t(), xin)

    ms_gemm = time_gpu(gemms, steps, warmup)
    gemm_flop = 3 * 2 * n_tok * sum(o * i for o, i in shapes)
    pairs = bsz * seq * (seq + 1) // 2
    attn_flop = 14 * 128 * 32 * pairs
    return {"ms_step": ms, "tokens_per_s": n_tok / (ms * 1e-3), "ms_projection_gemms_alone": ms_gemm,
            "ms_everything_else": ms - ms_gemm, "share_outside_gemms": (ms - ms_gemm) / ms,
            "tflops_model": (gemm_flop + attn_flop) / (ms * 1e-3) / 1e12,
            "note": "everything else = attention core, rotary, RMSNorm, SwiGLU, residual adds and autograd glue"}


def decode_case(steps, layers=32, batch=32, prompt=4096):
    """Config 5: random-init 8B-class decoder, batch of prompts prefilled, then greedy cached decoding.
    Reports decode tokens/s (batch * steps / decode wall time) and the prefill time."""
    import torch
    from scaling_amd.config import TransformerArchitectureConfig
    from scaling_amd.inference import TransformerInferenceModule
    cfg = TransformerArchitectureConfig.from_dict(dict(
        vocab_size=128256, hidden_size=4096, num_layers=layers, num_attention_heads=32, attention_num_kv_heads=8,
        attention_qkv_in_one=False, norm_type="rms", mlp_type="swiglu", mlp_factor=3.5, attention_bias=False, mlp_bias=False,
        precision="bfloat16", sequence_length=prompt + steps + 16, rotary_embedding_base=500000, weight_tying=False,
        masked_softmax={"kernel": "hip", "softmax_in_fp32": True}))
    torch.manual_seed(0)
    model = TransformerInferenceModule(cfg, device="cuda", init_std=0.02)
    g = torch.Generator().manual_seed(0)
    ids = torch.randint(1, cfg.vocab_size, (batch, prompt), generator=g)   # id 0 would split a prompt into documents
    model.generate(2, ids)                       # warm-up: library heuristics, allocator, caches
    torch.cuda.synchronize()
    t0 = time.time()
    model.generate(1, ids)                       # prefill + first token
    torch.cuda.synchronize()
    t_prefill = time.time() - t0
    t0 = time.time()
    model.generate(steps + 1, ids)               # prefill again + steps decode iterations, one launch per kernel
    torch.cuda.synchronize()
    t_eager = max(time.time() - t0 - t_prefill, 1e-9)
    model.generate_graph(4, ids)                 # warm-up of the capture path
    torch.cuda.synchronize()
    t0 = time.time()
    model.generate_graph(steps + 1, ids)         # prefill + steps decode iterations replayed from one HIP graph
    torch.cuda.synchronize()
    t_decode = max(time.time() - t0 - t_prefill, 1e-9)
    out = {"layers": layers, "batch": batch, "prompt": prompt, "decode_steps": steps, "prefill_s": t_prefill,
           "decode_s": t_decode, "decode_tok_per_s": batch * steps / t_decode, "ms_per_decode_step": 1e3 * t_decode / steps,
           "eager_decode_tok_per_s": batch * steps / t_eager, "eager_ms_per_decode_step": 1e3 * t_eager / steps,
           "note": "decode time = (prefill + decode wall time) - prefill wall time; graph capture time is included"}
    del model
    torch.cuda.empty_cache()
    return out


def _cpu_info():
    model, physical = "unknown", set()
    try:
        phys = core = None
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name") and model == "unknown":
                model = line.split(":", 1)[1].strip()
            elif line.startswith("physical id"):
                phys = line.split(":", 1)[1].strip()
            elif line.startswith("core id"):
                core = line.split(":", 1)[1].strip()
                physical.add((phys, core))
    except OSError:
        pass
    return model, os.cpu_count() or 1, len(physical) or None


def cpu_baseline(seconds_budget=25.0):
    """The reference's operation order (CPU oracle, plain torch) on the host cores, two bounded samples:
    the headline workload's attention (same head_dim / GQA ratio / causal mask / bf16 with fp32 softmax, fewer heads and
    a shorter sequence), which gives `value` in the metric's unit, and config 1 (the reference's own CPU-runnable case:
    one transformer layer forward + backward, fp32) at full size."""
    import torch
    import oracle
    model, logical, physical = _cpu_info()
    # the CPU share of a one-GPU box is what OMP_NUM_THREADS announces (16 here), whatever the machine has in total
    cores = int(os.environ.get("OMP_NUM_THREADS", "0")) or logical
    cores = max(1, min(cores, logical))
    torch.set_num_threads(cores)
    s, nq, nkv, d = 2048, 4, 1, 128
    g = torch.Generator().manual_seed(0)
    q = torch.randn(s, 1, nq, d, generator=g).bfloat16().requires_grad_()
    k = torch.randn(s, 1, nkv, d, generator=g).bfloat16().requires_grad_()
    v = torch.randn(s, 1, nkv, d, generator=g).bfloat16().requires_grad_()
    do = torch.randn(nq, s, d, generator=g).bfloat16()
    cu = torch.tensor([0, s], dtype=torch.int32)

    def step():
        out = oracle.multi_head_attention(q, oracle.repeat_kv(k, nq // nkv), oracle.repeat_kv(v, nq // nkv), cu, True,
                                          1 / math.sqrt(d), softmax_in_fp32=True)
        out.backward(do)
        q.grad = k.grad = v.grad = None

    def median_time(fn, budget, min_runs=3, max_runs=10):
        fn()
        times, t_all = [], time.time()
        while len(times) < min_runs or (time.time() - t_all < budget and len(times) < max_runs):
            t0 = time.time()
            fn()
            times.append(time.time() - t0)
        return sorted(times)[len(times) // 2], len(times)

    med, n_runs = median_time(step, seconds_budget / 3)
    flops = 14 * d * nq * (s * (s + 1) // 2)

    # config 1: hidden 256, 4 heads x 64, SwiGLU 688, RMSNorm, rotary base 10000, causal, batch 2 x seq 128, fp32
    spec = oracle.LayerSpec(hidden_size=256, num_attention_heads=4, qkv_in_one=False, norm_type="rms", mlp_type="swiglu",
                            layernorm_epsilon=1e-5, rotary_base=10000, sequence_length=128, causal=True, softmax_in_fp32=True,
                            dtype=torch.float32)
    g1 = torch.Generator().manual_seed(0)
    shapes = {"self_attention.query.weight": (256, 256), "self_attention.key.weight": (256, 256), "self_attention.value.weight": (256, 256),
              "self_attention.dense.weight": (256, 256), "mlp.dense_in.weight": (688, 256), "mlp.siglu_weight.weight": (688, 256),
              "mlp.dense_out.weight": (256, 688)}
    w1 = {name: (torch.randn(shape, generator=g1) * 0.02).requires_grad_() for name, shape in shapes.items()}
    w1["input_layernorm.weight"] = torch.ones(256, requires_grad=True)
    w1["post_attention_layernorm.weight"] = torch.ones(256, requires_grad=True)
    x1 = torch.randn(2, 128, 256, generator=g1).requires_grad_()
    dy1 = torch.randn(2, 128, 256, generator=g1)
    cu1 = torch.tensor([0, 128, 256], dtype=torch.int32)
    pos1 = torch.arange(128).repeat(2, 1)
    tables = spec.tables()

    def step_c1():
        y = oracle.transformer_layer(spec, w1, x1, cu1, pos1, tables=tables)
        y.backward(dy1)
        x1.grad = None
        for t in w1.values():
            t.grad = None

    med1, n1 = median_time(step_c1, seconds_budget / 3, min_runs=5, max_runs=200)

    # config 5 (decode): the oracle's batch-1 cached decode step (the reference's cache is batch-1, attention.py:855-857)
    # at the config-5 layer shape on a reduced layer count, extrapolated linearly in the layers.  The caches are filled
    # with random post-rotary K / V for a context of 4096 tokens instead of running the prefill (a decode step's cost
    # depends on the shapes only); torch.cat grows them by one token per step as the reference does.
    n_layers_cpu, ctx5, hid5, inter5, vocab5 = 2, 4096, 4096, 14336, 128256
    spec5 = oracle.LayerSpec(hidden_size=hid5, num_attention_heads=32, num_kv_heads=8, qkv_in_one=False, norm_type="rms",
                             mlp_type="swiglu", layernorm_epsilon=1e-5, rotary_base=500000, sequence_length=ctx5 + 64,
                             causal=True, softmax_in_fp32=True, dtype=torch.bfloat16)
    g5 = torch.Generator().manual_seed(0)

    def w5(*shape):
        return (torch.randn(shape, generator=g5) * 0.02).bfloat16()

    layers5 = []
    for _ in range(n_layers_cpu):
        layers5.append({"self_attention.query.weight": w5(hid5, hid5), "self_attention.key.weight": w5(1024, hid5),
                        "self_attention.value.weight": w5(1024, hid5), "self_attention.dense.weight": w5(hid5, hid5),
                        "mlp.dense_in.weight": w5(inter5, hid5), "mlp.siglu_weight.weight": w5(inter5, hid5),
                        "mlp.dense_out.weight": w5(hid5, inter5),
                        "input_layernorm.weight": torch.ones(hid5, dtype=torch.bfloat16),
                        "post_attention_layernorm.weight": torch.ones(hid5, dtype=torch.bfloat16)})
    final5 = {"norm.weight": torch.ones(hid5, dtype=torch.bfloat16)}
    head5 = w5(vocab5, hid5)
    tables5 = spec5.tables()
    cu5 = torch.tensor([0, 1], dtype=torch.int32)

    def fresh_caches():
        return [{0: (torch.randn(ctx5, 1, 8, 128, generator=g5).bfloat16(), torch.randn(ctx5, 1, 8, 128, generator=g5).bfloat16())}
                for _ in range(n_layers_cpu)]

    caches5 = fresh_caches()
    x5 = torch.randn(1, 1, hid5, generator=g5).bfloat16()
    step_no = [0]

    @torch.no_grad()
    def decode_layers():
        pos = torch.tensor([[ctx5 + step_no[0] % 32]])
        step_no[0] += 1
        h = x5
        for w, cache in zip(layers5, caches5):
            h = oracle.transformer_layer(spec5, w, h, cu5, pos, tables=tables5, use_cache=True, reset_cache=False, cache=cache)
        return h

    @torch.no_grad()
    def decode_head():
        return torch.nn.functional.linear(oracle.final_norm(spec5, final5, x5), head5).argmax()

    med_layers, n_l = median_time(decode_layers, seconds_budget / 6, min_runs=3, max_runs=30)
    med_head, n_h = median_time(decode_head, seconds_budget / 6, min_runs=3, max_runs=30)
    step32 = 32 * med_layers / n_layers_cpu + med_head
    del layers5, head5, caches5
    return {"value": flops / med / 1e12, "unit": "TFLOP/s", "cores": cores, "kind": "port",
            "cpu_model": model, "logical_cpus": logical, "physical_cores": physical,
            "sample": f"oracle (reference op order, bf16 + fp32 softmax) attention fwd+bwd, b1 s{s} {nq}q/{nkv}kv d{d} causal, "
                      f"median of {n_runs} runs = {med * 1e3:.1f} ms; config 1 (one layer fwd+bwd, fp32, hidden 256, 4 heads x 64, "
                      f"SwiGLU 688, batch 2 x seq 128) at full size: median of {n1} runs = {med1 * 1e3:.2f} ms "
                      f"({256 / med1:.0f} tokens/s)",
            "config1_layer_ms": med1 * 1e3, "config1_tokens_per_s": 256 / med1,
            "config5_decode": {"tok_per_s_extrapolated": 1.0 / step32, "ms_per_step_32_layers_extrapolated": step32 * 1e3,
                               "ms_per_layer_measured": med_layers / n_layers_cpu * 1e3, "ms_final_norm_lm_head_argmax": med_head * 1e3,
                               "how": f"EXTRAPOLATED: oracle cached decode step, batch 1 (the reference's cache takes one sequence), context "
                                      f"{ctx5}, bf16, measured on {n_layers_cpu} layers (median of {n_l} steps) and scaled linearly to 32 "
                                      f"layers, plus final norm + LM head + argmax (median of {n_h}); one token per step, so a batch of "
                                      f"32 prompts would be served one after the other at this rate"}}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    # 20 untimed steps (45 ms of the headline step): with 5 the timed region still began on ramping clocks, which showed
    # as a mean over the bracket 1 - 9 % above the median of the individually timed steps that followed
    ap.add_argument("--warmup", type=int, default=20)
    ap.add_argument("--no-extra", action="store_true", help="skip the secondary workloads")
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline")
    ap.add_argument("--decode-steps", type=int, default=256, help="greedy decode steps of the config-5 workload")
    ap.add_argument("--decode-only", action="store_true",
                    help="only run the config-5 decode workload (for a kernel trace of the decode step)")
    ap.add_argument("--decode-layers", type=int, default=32, help="layers of the config-5 model")
    ap.add_argument("--bandwidth-only", action="store_true",
                    help="only run the HBM-bound kernels (norms, SwiGLU, GELU, cross entropy, rotary, decode attention)")
    ap.add_argument("--profile-kernels", action="store_true",
                    help="only launch every HBM-bound kernel three times (the run the FETCH_SIZE / WRITE_SIZE counter passes are taken over)")
    ap.add_argument("--calibrate-copy", action="store_true",
                    help="only run a plain 1 GiB device copy (reference point for the FETCH_SIZE / WRITE_SIZE counters)")
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py measures one GPU's share of the path; this build uses no collectives, so --gpus must be 1",
              file=sys.stderr)
        sys.exit(2)

    import torch
    from scaling_amd import _lib
    _lib.require_device()
    torch.cuda.set_device(0)

    if args.calibrate_copy:
        src = torch.empty(1 << 30, dtype=torch.uint8, device="cuda").fill_(1)
        dst = torch.empty_like(src)
        ms = time_gpu(lambda: dst.copy_(src), args.steps, args.warmup)
        print(json.dumps({"calibration": "device copy", "bytes_read": 1 << 30, "bytes_written": 1 << 30, "ms": ms,
                          "GBs": 2 * (1 << 30) / ms / 1e6}))
        return

    if args.profile_kernels:
        print(json.dumps({"algorithmic_bytes_per_launch": profile_kernels()}))
        return

    if args.bandwidth_only:
        print(json.dumps({"bandwidth_kernels": bandwidth_cases(args.steps, args.warmup)}))
        return

    if args.decode_only:
        print(json.dumps({"config5_decode": decode_case(args.decode_steps, layers=args.decode_layers)}))
        return

    b, s, nq, nkv, d = 1, 8192, 32, 8, 128
    main_res = attention_case(b, s, nq, nkv, d, [0, s], args.steps, args.warmup)
    flops_unit = d * nq * main_res["pairs_per_head"]
    # dominant kernel of the step and the algorithmic flops it is credited with:
    #   forward 4 (QK^T, PV), backward 10 (dK/dV blocks S, dP, dV, dK; dQ blocks dQ: their S / dP are recomputation)
    kernels = {"attn_fwd_kernel": (main_res["ms_fwd"], 4), "attn_bwd_kernel": (main_res["ms_bwd_dkdv_dq"], 10)}
    dom = max(kernels, key=lambda n: kernels[n][0])
    dom_ms, dom_mult = kernels[dom]
    achieved = dom_mult * flops_unit / (dom_ms * 1e-3) / 1e12
    traffic, traffic_note = measured_traffic_bytes(dom)
    roofline = {"bound": "mfma", "kernel": dom, "achieved": achieved, "peak": PEAK_BF16_TFLOPS, "unit": "TFLOP/s",
                "frac": achieved / PEAK_BF16_TFLOPS, "traffic": traffic, "traffic_unit": "bytes per launch", "traffic_note": traffic_note,
                "avg_launch_ms": dom_ms}

    extra = {"headline": main_res}
    if not args.no_extra:
        extra["config2_mha_b4_s2048"] = attention_case(4, 2048, 32, 32, 128, [i * 2048 for i in range(5)], args.steps, args.warmup, seed=2)
        cu3 = random_docs_cu(8192, 256, 2048, seed=0).tolist()
        extra["config3_gqa_packed_rotary_s8192"] = attention_case(1, 8192, 32, 8, 128, cu3, args.steps, args.warmup, seed=3, rotary=True)
        extra["config3_gqa_packed_rotary_s8192"]["n_docs"] = len(cu3) - 1
        extra["attention_float32_gqa32x8_d128_s4096"] = attention_float32_case(args.steps, args.warmup)
        extra.update(bandwidth_cases(args.steps, args.warmup))
        extra["config4_layer_fwd_bwd_b2_s4096_h4096"] = layer_case(max(5, args.steps // 2), 3)
        extra["config5_decode_8b_b32_ctx4096"] = decode_case(args.decode_steps, layers=args.decode_layers)

    line = {
        "metric": "attn fwd+bwd TFLOP/s (% bf16 MFMA peak); decode tok/s; norm GB/s (% HBM)",
        "value": main_res["tflops_step"], "unit": "TFLOP/s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": main_res["ms_step"], "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
        "dtype": "bf16", "data": "synthetic",
        "config": {"workload": "attention core fwd+bwd, GQA 32q/8kv, head_dim 128, batch 1 x seq 8192, causal, bf16, fp32 softmax; "
                               "default mode: P rounded to bf16 before P V as the reference does (attention.py:211)",
                   "pairs_per_head": main_res["pairs_per_head"], "flop_formula": "14*d*n_q*P",
                   "accuracy_mode": {"what": "MI_ATTN_SPLIT_P (P and dS as two bf16 terms): meets max-abs 2e-2 / mean-rel 1e-3 "
                                             "literally without rotary; the default mode meets them through the documented "
                                             "second clauses of tests/parity.py",
                                     "ms_per_step": main_res["ms_step_precise"], "value": main_res["tflops_step_precise"],
                                     "time_over_default": main_res["precise_over_default_time"]}},
        "frac_of_bf16_peak": main_res["tflops_step"] / PEAK_BF16_TFLOPS,
        "roofline": roofline,
    }
    if not args.no_cpu:
        line["cpu_baseline"] = cpu_baseline()
    line["extra"] = extra
    print(json.dumps(line))


if __name__ == "__main__":
    main()
