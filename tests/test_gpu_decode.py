"""GPU parity of the KV-cache decode kernel against the CPU oracle (per-sequence batch-1 reference
semantics: the step output equals the last row of full causal attention over the cached positions)."""

import math

import pytest
import torch

import oracle
from scaling_amd import _lib, ops
from tests.kernels import launched
from tests.parity import check

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _oracle_decode(q, kc, vc, ctx, scale, dtype):
    """q [B,nq,d], caches [B,max,nkv,d] (already containing the new token); one reference call per sequence."""
    B, nq, d = q.shape
    nkv = kc.shape[2]
    outs = []
    for b in range(B):
        n = int(ctx[b])
        qq = q[b].to(dtype).view(1, 1, nq, d)                                   # [s_q=1, b=1, n, d]
        kk = oracle.repeat_kv(kc[b, :n].to(dtype).unsqueeze(1), nq // nkv)      # [s_k, 1, nq, d]
        vv = oracle.repeat_kv(vc[b, :n].to(dtype).unsqueeze(1), nq // nkv)
        o = oracle.multi_head_attention(qq, kk, vv, torch.tensor([0, 1], dtype=torch.int32), True, scale,
                                        softmax_in_fp32=True)                   # [(1 nq), 1, d]
        outs.append(o.view(nq, d))
    return torch.stack(outs)


@pytest.mark.parametrize("B,nq,nkv,d,max_ctx,lens", [
    (3, 8, 2, 128, 300, [1, 137, 300]),
    (2, 4, 4, 64, 128, [128, 5]),
    (4, 32, 8, 128, 1100, [1024, 1025, 33, 1100]),
    (1, 16, 1, 128, 64, [64]),
    # groups of more than 16 query heads (multi-query attention with 32 heads; 24 = one full and one partial chunk)
    (2, 32, 1, 128, 300, [300, 17]),
    (1, 24, 1, 64, 128, [128]),
    # the other head sizes of the attention kernels
    (2, 4, 2, 96, 200, [200, 33]),
    (3, 8, 8, 32, 100, [100, 1, 64]),
    (40, 12, 6, 96, 70, [70, 69, 1, 35] * 10),
    # batch x KV heads >= 192: the 8-wavefront workgroups (a single split writes the output directly)
    (24, 16, 8, 128, 300, [300, 1, 257, 31] * 6),
    (48, 8, 4, 64, 520, [520, 256, 255, 7, 300, 513] * 8),
])
@pytest.mark.parametrize("n_splits", [0, 1, 3])
def test_decode_parity(B, nq, nkv, d, max_ctx, lens, n_splits):
    print(f"case decode B={B} nq={nq} nkv={nkv} d={d} max_ctx={max_ctx} lens={lens} splits={n_splits}", flush=True)
    g = torch.Generator().manual_seed(B * 31 + d)
    q = torch.randn(B, nq, d, generator=g).bfloat16()
    kc = torch.randn(B, max_ctx, nkv, d, generator=g).bfloat16()
    vc = torch.randn(B, max_ctx, nkv, d, generator=g).bfloat16()
    ctx = torch.tensor(lens, dtype=torch.int32)
    scale = 1 / math.sqrt(d)
    ref = _oracle_decode(q, kc, vc, ctx, scale, torch.float32)
    ref_o = _oracle_decode(q, kc, vc, ctx, scale, torch.bfloat16)
    out = ops.decode_attention(q.to(DEV), kc.to(DEV), vc.to(DEV), ctx.to(DEV), softmax_scale=scale, n_splits=n_splits)
    torch.cuda.synchronize()
    check("decode.o", out, ref, ref_o, kind="decode")


def test_decode_append_and_fused_rotary():
    B, nq, nkv, d, max_ctx = 3, 8, 2, 128, 96
    g = torch.Generator().manual_seed(77)
    lens = [10, 96, 1]                       # lengths INCLUDING the appended token
    q = torch.randn(B, nq, d, generator=g).bfloat16()
    k_new = torch.randn(B, nkv, d, generator=g).bfloat16()
    v_new = torch.randn(B, nkv, d, generator=g).bfloat16()
    kc = torch.randn(B, max_ctx, nkv, d, generator=g).bfloat16()
    vc = torch.randn(B, max_ctx, nkv, d, generator=g).bfloat16()
    ctx = torch.tensor(lens, dtype=torch.int32)
    pos = torch.tensor([n - 1 for n in lens], dtype=torch.int64)
    tabs = oracle.rotary_tables(d, max_ctx, 500000, torch.bfloat16)
    hi = oracle.RotaryTables(tabs.cos.float(), tabs.sin.float(), d)
    # reference: rotate the new q/k at their positions, append, attend
    qr, kr = oracle.apply_rotary(q.float().unsqueeze(0), k_new.float().unsqueeze(0), hi, pos.view(1, B), pos.view(1, B))
    qr, kr = qr[0].bfloat16(), kr[0].bfloat16()     # what is stored / consumed after one rounding
    kc_ref, vc_ref = kc.clone(), vc.clone()
    for b in range(B):
        kc_ref[b, lens[b] - 1] = kr[b]
        vc_ref[b, lens[b] - 1] = v_new[b]
    scale = 1 / math.sqrt(d)
    ref = _oracle_decode(qr, kc_ref, vc_ref, ctx, scale, torch.float32)
    ref_o = _oracle_decode(qr, kc_ref, vc_ref, ctx, scale, torch.bfloat16)
    kcd, vcd = kc.to(DEV), vc.to(DEV)
    out = ops.decode_attention(q.to(DEV), kcd, vcd, ctx.to(DEV), k_new.to(DEV), v_new.to(DEV),
                               rotary=(tabs.cos.to(DEV), tabs.sin.to(DEV), pos.to(DEV)), softmax_scale=scale)
    torch.cuda.synchronize()
    check("decode.o(append+rotary)", out, ref, ref_o, kind="decode")
    # the cache was updated in place: only the appended rows changed, and they hold the rotated key
    for b in range(B):
        kd = (kcd[b, lens[b] - 1].float().cpu() - kr[b].float()).abs()
        assert float(kd.max()) <= 2e-2 and float((kd > 0).float().mean()) < 0.02
        assert torch.equal(vcd[b, lens[b] - 1].cpu(), v_new[b])
    mask = torch.ones(B, max_ctx, dtype=torch.bool)
    for b in range(B):
        mask[b, lens[b] - 1] = False
    assert torch.equal(kcd.cpu()[mask], kc[mask]) and torch.equal(vcd.cpu()[mask], vc[mask])


@pytest.mark.parametrize("B,nq,nkv,d", [(3, 8, 2, 128), (2, 4, 4, 64), (32, 32, 8, 128)])
def test_decode_append_and_fused_interleaved_rotary(B, nq, nkv, d):
    """Interleaved-pair rotary of q and of the appended key inside the decode kernels: same bits as the stand-alone
    kernel followed by a plain append, and within the gates of the oracle."""
    print(f"case decode fused interleaved rotary B={B} nq={nq} nkv={nkv} d={d}", flush=True)
    max_ctx = 96
    g = torch.Generator().manual_seed(B + d)
    lens = [(7 * i) % max_ctx + 1 for i in range(B)]
    lens[0] = max_ctx
    q = torch.randn(B, nq, d, generator=g).bfloat16()
    k_new = torch.randn(B, nkv, d, generator=g).bfloat16()
    v_new = torch.randn(B, nkv, d, generator=g).bfloat16()
    kc = torch.randn(B, max_ctx, nkv, d, generator=g).bfloat16()
    vc = torch.randn(B, max_ctx, nkv, d, generator=g).bfloat16()
    ctx = torch.tensor(lens, dtype=torch.int32)
    pos = torch.tensor([n - 1 for n in lens], dtype=torch.int64)
    scale = 1 / math.sqrt(d)
    qr, kr = oracle.apply_rotary_complex(q.unsqueeze(0), k_new.unsqueeze(0), d, max_ctx, 10000.0, pos.view(1, B), pos.view(1, B))
    qr, kr = qr[0], kr[0]                           # fp32 math, one rounding to bf16 (the reference's order)
    kc_ref, vc_ref = kc.clone(), vc.clone()
    for b in range(B):
        kc_ref[b, lens[b] - 1] = kr[b]
        vc_ref[b, lens[b] - 1] = v_new[b]
    ref = _oracle_decode(qr, kc_ref, vc_ref, ctx, scale, torch.float32)
    ref_o = _oracle_decode(qr, kc_ref, vc_ref, ctx, scale, torch.bfloat16)
    inv_freq = 1.0 / (10000.0 ** (torch.arange(0, d, 2)[: d // 2].float() / d))
    ang = torch.outer(torch.arange(max_ctx).float(), inv_freq).float()
    real, imag = ang.cos().contiguous().to(DEV), ang.sin().contiguous().to(DEV)
    qd, knd, vnd, ctxd, posd = q.to(DEV), k_new.to(DEV), v_new.to(DEV), ctx.to(DEV), pos.to(DEV)
    kc1, vc1 = kc.to(DEV), vc.to(DEV)
    fused = ops.decode_attention(qd, kc1, vc1, ctxd, knd, vnd, rotary=(real, imag, posd), softmax_scale=scale)
    kc2, vc2 = kc.to(DEV), vc.to(DEV)
    q2 = ops.rotary_embedding_complex(qd, real, imag, posd)
    k2 = ops.rotary_embedding_complex(knd, real, imag, posd)
    sep = ops.decode_attention(q2, kc2, vc2, ctxd, k2, vnd, softmax_scale=scale)
    torch.cuda.synchronize()
    check("decode.o(append+interleaved rotary)", fused, ref, ref_o, kind="decode")
    assert torch.equal(fused, sep) and torch.equal(kc1, kc2) and torch.equal(vc1, vc2)
    for b in range(B):
        kd = (kc1[b, lens[b] - 1].float().cpu() - kr[b].float()).abs()
        assert float(kd.max()) <= 2e-2 and float((kd > 0).float().mean()) < 0.02


def test_decode_equals_last_row_of_prefill_kernel():
    """Cached == uncached: the decode kernel agrees with the last query row of the forward kernel."""
    nq, nkv, d, n = 8, 2, 128, 333
    g = torch.Generator().manual_seed(5)
    q = torch.randn(n, nq, d, generator=g).bfloat16().to(DEV)
    k = torch.randn(n, nkv, d, generator=g).bfloat16().to(DEV)
    v = torch.randn(n, nkv, d, generator=g).bfloat16().to(DEV)
    cu = torch.tensor([0, n], dtype=torch.int32, device=DEV)
    full, _ = ops.attention_forward(q, k, v, cu)
    out = ops.decode_attention(q[n - 1:n].contiguous(), k.unsqueeze(0), v.unsqueeze(0),
                               torch.tensor([n], dtype=torch.int32, device=DEV))
    torch.cuda.synchronize()
    diff = (out[0].float() - full[n - 1].float()).abs()
    assert float(diff.max()) <= 1.6e-2


def test_decode_takes_column_slices_of_a_fused_projection():
    """q, k_new and v_new as strided column slices of one [B, (nq + 2 nkv) d] tensor (what a single q/k/v GEMM
    produces) give bit-identical outputs and cache contents to packed copies of the same values."""
    print("case decode strided operands", flush=True)
    B, nq, nkv, d, max_ctx = 5, 8, 2, 128, 200
    g = torch.Generator().manual_seed(5)
    fused = torch.randn(B, (nq + 2 * nkv) * d, generator=g).bfloat16().to(DEV)
    q = fused[:, :nq * d].view(B, nq, d)
    k = fused[:, nq * d:(nq + nkv) * d].view(B, nkv, d)
    v = fused[:, (nq + nkv) * d:].view(B, nkv, d)
    assert not q.is_contiguous() and q.stride(0) == (nq + 2 * nkv) * d
    ctx = torch.tensor([200, 1, 77, 128, 129], dtype=torch.int32, device=DEV)
    outs, caches = [], []
    for packed in (False, True):
        kc = torch.randn(B, max_ctx, nkv, d, generator=torch.Generator().manual_seed(6)).bfloat16().to(DEV)
        vc = torch.randn(B, max_ctx, nkv, d, generator=torch.Generator().manual_seed(7)).bfloat16().to(DEV)
        args = (q.contiguous(), kc, vc, ctx, k.contiguous(), v.contiguous()) if packed else (q, kc, vc, ctx, k, v)
        outs.append(ops.decode_attention(*args))
        caches.append((kc, vc))
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1])
    assert torch.equal(caches[0][0], caches[1][0]) and torch.equal(caches[0][1], caches[1][1])
    for b in range(B):     # the appended rows landed at ctx - 1
        assert torch.equal(caches[0][0][b, int(ctx[b]) - 1], k[b]) and torch.equal(caches[0][1][b, int(ctx[b]) - 1], v[b])
    with pytest.raises(AssertionError):
        ops.decode_attention(fused.view(B, nq + 2 * nkv, d)[:, ::2], caches[0][0], caches[0][1], ctx)   # heads not contiguous


@pytest.mark.parametrize("B,nq,nkv,d,max_ctx,lens", [(3, 8, 2, 128, 300, [1, 137, 300]), (24, 16, 8, 128, 300, [300, 1, 257, 31] * 6),
                                                    (2, 4, 4, 64, 128, [128, 5])])
def test_decode_float16_parity(B, nq, nkv, d, max_ctx, lens):
    """The decode kernels built on the half-precision MFMA (precision: float16), with the in-place append."""
    print(f"case decode f16 B={B} nq={nq} nkv={nkv} d={d} lens={lens}", flush=True)
    g = torch.Generator().manual_seed(B + d)
    q = torch.randn(B, nq, d, generator=g).half()
    kc = torch.randn(B, max_ctx, nkv, d, generator=g).half()
    vc = torch.randn(B, max_ctx, nkv, d, generator=g).half()
    k_new, v_new = torch.randn(B, nkv, d, generator=g).half(), torch.randn(B, nkv, d, generator=g).half()
    ctx = torch.tensor(lens, dtype=torch.int32)
    kc_ref, vc_ref = kc.clone(), vc.clone()
    for b in range(B):
        kc_ref[b, lens[b] - 1] = k_new[b]
        vc_ref[b, lens[b] - 1] = v_new[b]
    scale = 1 / math.sqrt(d)
    ref = _oracle_decode(q, kc_ref, vc_ref, ctx, scale, torch.float32)
    ref_o = _oracle_decode(q, kc_ref, vc_ref, ctx, scale, torch.float16)
    kcd, vcd = kc.to(DEV), vc.to(DEV)
    out = ops.decode_attention(q.to(DEV), kcd, vcd, ctx.to(DEV), k_new.to(DEV), v_new.to(DEV), softmax_scale=scale)
    torch.cuda.synchronize()
    assert out.dtype == torch.float16
    check("decode.f16.o", out, ref, ref_o, kind="decode")
    assert torch.equal(kcd.cpu(), kc_ref) and torch.equal(vcd.cpu(), vc_ref)


@pytest.mark.parametrize("B,nq,nkv,d,max_ctx,n_splits", [
    # one split up to a cache of 256 tokens, then several; the new token first or last of a 32-key chunk, or alone in its split
    (5, 4, 2, 128, 256, 0), (5, 4, 2, 128, 257, 0), (5, 4, 2, 32, 700, 0), (5, 8, 2, 64, 700, 3), (5, 4, 2, 96, 1300, 11),
    (5, 32, 1, 64, 300, 2),         # two workgroups share a KV head and its new row
])
def test_decode_append_at_chunk_and_split_edges(B, nq, nkv, d, max_ctx, n_splits):
    """The wavefront that owns the new key writes it and reads it back: the same as with the row already in the cache."""
    print(f"case decode append edges B={B} nq={nq} nkv={nkv} d={d} max_ctx={max_ctx} splits={n_splits}", flush=True)
    g = torch.Generator().manual_seed(max_ctx + d)
    lens = [1, 32, 129, max_ctx - 1, max_ctx]
    q = torch.randn(B, nq, d, generator=g).bfloat16()
    kc, vc = (torch.randn(B, max_ctx, nkv, d, generator=g).bfloat16() for _ in range(2))
    k_new, v_new = (torch.randn(B, nkv, d, generator=g).bfloat16() for _ in range(2))
    ctx = torch.tensor(lens, dtype=torch.int32)
    kc_ref, vc_ref = kc.clone(), vc.clone()
    for b in range(B):
        kc_ref[b, lens[b] - 1], vc_ref[b, lens[b] - 1] = k_new[b], v_new[b]
    scale = 1 / math.sqrt(d)
    kcd, vcd = kc.to(DEV), vc.to(DEV)
    out = ops.decode_attention(q.to(DEV), kcd, vcd, ctx.to(DEV), k_new.to(DEV), v_new.to(DEV), softmax_scale=scale, n_splits=n_splits)
    present = ops.decode_attention(q.to(DEV), kc_ref.to(DEV), vc_ref.to(DEV), ctx.to(DEV), softmax_scale=scale, n_splits=n_splits)
    torch.cuda.synchronize()
    check("decode.o(append edges)", out, _oracle_decode(q, kc_ref, vc_ref, ctx, scale, torch.float32),
          _oracle_decode(q, kc_ref, vc_ref, ctx, scale, torch.bfloat16), kind="decode")
    assert torch.equal(out, present) and torch.equal(kcd.cpu(), kc_ref) and torch.equal(vcd.cpu(), vc_ref)


# splits that are empty (short contexts, none at all), one and every count of head chunks, the most splits, both sizes of workgroups
@pytest.mark.parametrize("B,nq,nkv,d,max_ctx,lens,n_splits", [
    (1, 32, 8, 128, 1564, [1500], 0), (3, 8, 2, 128, 4000, [4000, 1, 0], 13), (2, 24, 1, 32, 700, [700, 129], 0), (1, 4, 4, 96, 4096, [4096], 16),
    (2, 6, 3, 32, 300, [300, 299], 2), (48, 8, 4, 64, 330, [330, 256, 255, 7, 300, 1] * 8, 3), (1, 16, 4, 128, 2000, [33], 9),
])
def test_decode_merged_by_the_last_workgroup(B, nq, nkv, d, max_ctx, lens, n_splits):
    """With the tickets of a `decode_workspace` the splits of a small call are merged inside the launch: the bits of the two launches, tickets zero
    again after every call; through the C entry in a graph too, where the Python one takes two launches."""
    g = torch.Generator().manual_seed(B + d)
    kc, vc = (torch.randn(B, max_ctx, nkv, d, generator=g).bfloat16().to(DEV) for _ in range(2))
    qs = [torch.randn(B, nq, d, generator=g).bfloat16().to(DEV) for _ in range(3)]
    ctx = torch.tensor(lens, dtype=torch.int32).to(DEV)
    ws = ops.decode_workspace(B, nq, d, max_ctx, DEV)
    plain = torch.empty_like(ws)
    call = lambda q, workspace, out: ops.decode_attention(q, kc, vc, ctx, workspace=workspace, n_splits=n_splits, out=out)
    want = [call(q, plain, torch.empty_like(q)) for q in qs]
    out, q = torch.empty_like(qs[0]), qs[0].clone()
    assert not any("decode_merge" in n for n in launched(lambda: call(q, ws, out)))
    for i in (1, 2, 0):
        out.fill_(float("nan"))
        call(qs[i], ws, out)
        assert torch.equal(out, want[i]) and not ws.tickets.any()
    args = _lib.MiDecodeArgs()
    args.q, args.o, args.k_cache, args.v_cache, args.ctx_len = (t.data_ptr() for t in (q, out, kc, vc, ctx))
    args.batch, args.max_ctx, args.n_q_heads, args.n_kv_heads, args.head_dim, args.n_splits = B, max_ctx, nq, nkv, d, n_splits
    args.softmax_scale = 1.0 / math.sqrt(d)
    args.cache_stride_batch, args.cache_stride_token, args.cache_stride_head = kc.stride()[:3]
    args.workspace, args.workspace_bytes = ws.data_ptr(), ws.numel() * 4

    def entry(n_tickets):
        args.stream = torch.cuda.current_stream().cuda_stream
        _lib.check(_lib.load().mi_attn_decode_with_tickets(args, ws.tickets.data_ptr(), n_tickets), "mi_attn_decode_with_tickets")

    with pytest.raises(RuntimeError, match="ticket"):
        entry(B * nkv - 1)
    for capture in (lambda: entry(B * nq), lambda: call(q, ws, out)):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            capture()
        for i in (0, 1, 2):
            q.copy_(qs[i])
            out.fill_(float("nan"))
            graph.replay()
            assert torch.equal(out, want[i]) and not ws.tickets.any()
    assert getattr(ws[:1], "tickets", None) is None


@pytest.mark.parametrize("nq,nkv,d,max_ctx,n_splits", [
    (32, 8, 128, 256, 0), (4, 2, 128, 600, 0), (4, 4, 64, 300, 3), (6, 3, 96, 257, 0), (40, 2, 32, 256, 0), (24, 1, 64, 700, 7),
])
@pytest.mark.parametrize("kind", ["plain", "half", "interleaved"])
def test_decode_append_over_what_the_row_held(nq, nkv, d, max_ctx, n_splits, kind):
    """The new key's operands come from `k_new` and `v_new`: the same bits as with the row in the cache before the call, whatever the row held,
    where the new key is first, in the middle or last of a chunk, and for sequences without any key, whose rows stay as they are."""
    if kind == "half" and d not in (64, 128):
        pytest.skip("rotate-half rotary inside the kernel is for heads of 64 and 128")
    lens = [0, 1, 17, 32, 33, 128, 129, 255, max_ctx]
    g = torch.Generator().manual_seed(nq + d)
    normal = lambda *shape: torch.randn(*shape, generator=g).bfloat16().to(DEV)
    B = len(lens)
    q, k_new, v_new, kc, vc = normal(B, nq, d), normal(B, nkv, d), normal(B, nkv, d), normal(B, max_ctx, nkv, d), normal(B, max_ctx, nkv, d)
    ctx = torch.tensor(lens, dtype=torch.int32, device=DEV)
    rotary = None
    if kind != "plain":
        angle = torch.rand(max_ctx, d // 2, generator=g) * 6
        cos, sin = (angle.cos().to(DEV), angle.sin().to(DEV))
        if kind == "half":
            cos, sin = (torch.cat([t, t], 1).bfloat16() for t in (cos, sin))
        rotary = (cos, sin, torch.tensor([max(n - 1, 0) for n in lens], device=DEV))
    for b, n in enumerate(lens):
        kc[b, max(n - 1, 0):], vc[b, max(n - 1, 0):] = float("nan"), float("inf")
    before = kc.clone(), vc.clone()
    out = ops.decode_attention(q, kc, vc, ctx, k_new, v_new, rotary=rotary, n_splits=n_splits)
    present = ops.decode_attention(q, kc, vc, ctx, rotary=rotary, n_splits=n_splits)
    assert torch.equal(out, present) and out.isfinite().all() and not out[0].any()
    for b, n in enumerate(lens):
        if n > 0:
            assert torch.equal(vc[b, n - 1], v_new[b]) and kc[b, n - 1].isfinite().all()
            if kind == "plain":
                assert torch.equal(kc[b, n - 1], k_new[b])
        for now, held in zip((kc, vc), before):            # nothing but the new row was written
            now[b, max(n - 1, 0):n] = held[b, max(n - 1, 0):n]
            assert torch.equal(now[b].view(torch.int16), held[b].view(torch.int16))


@pytest.mark.parametrize("d", [64, 128])
def test_float16_keys_are_rounded_as_they_always_were(d):
    """The sums of a rotated float16 key are exact in float64.  Features 2 - 7 of every eight of the second half are rounded to float32 and then to
    float16, the others once.  The smaller product of each sum lies below the last bit of float32 and the larger one, of 22 bits, is a tie between two
    float16 values in one of 2000 sums, so that the two differ often enough."""
    B, nkv, g = 64, 32, torch.Generator().manual_seed(d)
    size = torch.where(torch.arange(d) < d // 2, 64.0, 2.0 ** -8)
    k, v, q = (((1 + torch.rand(B, nkv, d, generator=g)) * torch.randn(B, nkv, d, generator=g).sign()).half() for _ in range(3))
    k[::2], k[1::2] = k[::2] * size, k[1::2] * size.flip(0)
    cos, sin = (torch.cat([t, t], 1).half() for t in (0.5 + 0.5 * torch.rand(B, d // 2, generator=g), 2.0 ** -14 * (1 + torch.rand(B, d // 2, generator=g))))
    kc, vc = (torch.zeros(B, 4, nkv, d, dtype=torch.float16, device=DEV) for _ in range(2))
    ctx = torch.full((B,), 3, dtype=torch.int32, device=DEV)
    ops.decode_attention(q.to(DEV), kc, vc, ctx, k.to(DEV), v.to(DEV), rotary=(cos.to(DEV), sin.to(DEV), torch.arange(B, device=DEV)))
    x0, x1 = k.double().chunk(2, -1)
    c, s = (t[:, None, :d // 2].double() for t in (cos, sin))
    exact = torch.cat([x0 * c - x1 * s, x1 * c + x0 * s], -1)
    once = torch.from_numpy(exact.numpy().astype("float16"))
    twice = torch.from_numpy(exact.numpy().astype("float32").astype("float16"))
    feature = torch.arange(d)
    want = torch.where((feature >= d // 2) & (feature % 8 >= 2), twice, once)
    assert torch.equal(kc[:, 2].cpu(), want) and torch.equal(vc[:, 2].cpu(), v)
    assert int((want != once).sum()) > 10 and int((want != twice).sum()) > 10


# more workgroups than compute units, with sequences of different lengths, of equal ones, without keys; the most sequences that are handed out by
# length, and one more; one key too few for it; splits that are merged by the last workgroup and by a launch of their own
@pytest.mark.parametrize("B,nq,nkv,d,max_ctx,n_splits,kind", [
    (17, 32, 8, 128, 1100, 2, "half"), (17, 32, 8, 128, 1023, 2, "half"), (10, 8, 8, 64, 2048, 4, "half"), (64, 4, 1, 128, 2600, 5, "plain"),
    (65, 4, 1, 128, 2600, 5, "plain"), (5, 16, 16, 64, 2100, 4, "pairs"), (3, 24, 2, 96, 16384, 32, "plain"), (5, 40, 2, 32, 16400, 16, "pairs"),
    (63, 2, 2, 64, 1600, 3, "half"),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_decode_of_more_workgroups_than_compute_units(B, nq, nkv, d, max_ctx, n_splits, kind, dtype):
    """Workgroups find their sequence by its length: every sequence has the bits it has in a call of its own."""
    g = torch.Generator().manual_seed(B)
    normal = lambda *shape: torch.randn(*shape, generator=g).to(dtype).to(DEV)
    q, k_new, v_new, kc, vc = normal(B, nq, d), normal(B, nkv, d), normal(B, nkv, d), normal(B, max_ctx, nkv, d), normal(B, max_ctx, nkv, d)
    lens = torch.randint(1, max_ctx + 1, (B,), generator=g)
    lens[B // 2:] = lens[B // 2:].clamp(max=max_ctx // 3)  # several of one length
    lens[0], lens[-1] = max_ctx, 0
    ctx, pos, rotary = lens.int().to(DEV), (lens - 1).clamp(min=0).to(DEV), None
    if kind != "plain":
        angle = torch.rand(max_ctx, d // 2, generator=g) * 6
        cos, sin = (angle.cos().to(DEV), angle.sin().to(DEV))
        if kind == "half":
            cos, sin = (torch.cat([t, t], 1).to(dtype) for t in (cos, sin))
        rotary = (cos, sin, pos)
    alone = []
    for b in range(B):
        one = [t[b:b + 1].clone() for t in (kc, vc)]
        row = None if rotary is None else (*rotary[:2], pos[b:b + 1].contiguous())
        alone.append([ops.decode_attention(q[b:b + 1], *one, ctx[b:b + 1], k_new[b:b + 1], v_new[b:b + 1], rotary=row, n_splits=n_splits), *one])
    want = [torch.cat(t) for t in zip(*alone)]
    for workspace in (None, ops.decode_workspace(B, nq, d, max_ctx, DEV)):
        caches = kc.clone(), vc.clone()
        for _ in range(2):
            out = ops.decode_attention(q, *caches, ctx, k_new, v_new, rotary=rotary, n_splits=n_splits, workspace=workspace)
            assert all(torch.equal(a, c) for a, c in zip((out, *caches), want))
    assert not workspace.tickets.any()


@pytest.mark.parametrize("kind", ["plain", "half", "pairs"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,nq,nkv,n_splits", [(33, 16, 8, 0), (48, 6, 6, 0), (24, 8, 8, 2)])
def test_workgroups_that_share_a_compute_unit(B, nq, nkv, n_splits, dtype, kind):
    """Up to 2048 keys the new row of heads of 64 waits for its chunk in LDS, with one more in registers: the same bits, and the oracle's values."""
    g, d, lens = torch.Generator().manual_seed(B + nq), 64, [1, 31, 32, 33, 255, 256, 257, 600, 2048, 0]
    normal = lambda *shape: torch.randn(*shape, generator=g).to(dtype).to(DEV)
    q, k_new, v_new, kc, vc = normal(B, nq, d), normal(B, nkv, d), normal(B, nkv, d), normal(B, 2049, nkv, d), normal(B, 2049, nkv, d)
    ctx = torch.tensor((lens * 5)[:B], dtype=torch.int32, device=DEV)
    pos, rotary = (ctx.long() - 1).clamp(min=0), None
    if kind != "plain":
        angle = torch.rand(2048, d // 2, generator=g) * 6
        cos, sin = (angle.cos().to(DEV), angle.sin().to(DEV))
        if kind == "half":
            cos, sin = (torch.cat([t, t], 1).to(dtype) for t in (cos, sin))
        rotary = (cos, sin, pos)
    results = []
    for max_ctx in (2048, 2049):
        caches = kc.clone(), vc.clone()
        call = lambda: results.append([ops.decode_attention(q, *(c[:, :max_ctx] for c in caches), ctx, k_new, v_new, rotary=rotary, n_splits=n_splits), *caches])
        call()
    assert all(torch.equal(a, b) for a, b in zip(*results))
    for b in range(min(B, 10)):
        assert torch.equal(vc[b, lens[b]:], results[0][2][b, lens[b]:]) and torch.equal(kc[b, :max(lens[b] - 1, 0)], results[0][1][b, :max(lens[b] - 1, 0)])
        if lens[b] > 0:
            assert torch.equal(results[0][2][b, lens[b] - 1], v_new[b])
    rotated = q if rotary is None else (ops.rotary_embedding if kind == "half" else ops.rotary_embedding_complex)(q, cos, sin, pos)
    some = [b for b in range(10) if lens[b] > 0]
    for b in some:
        keys, values = (t[b, :lens[b]].float().repeat_interleave(nq // nkv, 1) for t in results[0][1:])
        p = torch.einsum("hd,thd->ht", rotated[b].float().cpu(), keys.cpu()).mul(d ** -0.5).softmax(-1)
        want = torch.einsum("ht,thd->hd", p, values.cpu())
        # P is rounded to 16 bits before it meets V, the result once more; q by the rotary, once or twice
        assert float((results[0][0][b].float().cpu() - want).norm()) <= (2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -10) * float(want.norm()), b
