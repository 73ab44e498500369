"""The two families of 16-bit attention kernels - tiled, and the ones for short contexts that small calls go to - over the same cases,
each pinned by its flag: against the oracle, and with the rotary inside against each other."""

import math
import random

import pytest
import torch

import oracle
from scaling_amd import _lib, ops
from tests import attn_utils as U
from tests.parity import check
from tests.kernels import launched
from tests.test_gpu_attention import CASES

pytestmark = pytest.mark.gpu
DEV = "cuda"
SHORT, TILED = 128, 256


@pytest.mark.parametrize("flags", [SHORT, TILED])
@pytest.mark.parametrize("b,s,nq,nkv,d,causal,cuts", CASES)
def test_attention_routes_parity(b, s, nq, nkv, d, causal, cuts, flags):
    print(f"case route={flags} b={b} s={s} nq={nq} nkv={nkv} d={d} causal={causal} cuts={cuts}", flush=True)
    q, k, v, do = U.make_qkv(b, s, nq, nkv, d, seed=b * 1000 + s + d)
    cu = U.make_cu(b, s, cuts)
    scale = 1.0 / math.sqrt(d)
    ref = U.oracle_attention(q, k, v, cu, b, s, causal, scale, torch.float32, do)
    ref_o = U.oracle_attention(q, k, v, cu, b, s, causal, scale, torch.bfloat16, do)
    qd, kd, vd, dod, cud = (t.to(DEV) for t in (q, k, v, do, cu))
    o, lse = ops.attention_forward(qd, kd, vd, cud, None, causal, scale, flags=flags)
    dq, dk, dv = ops.attention_backward(dod, qd, kd, vd, o, lse, cud, None, causal, scale, flags=flags)
    torch.cuda.synchronize()
    check("route.o", o, ref[0], ref_o[0], kind="o")
    check("route.dq", dq, ref[1], ref_o[1], kind="grad")
    check("route.dk", dk, ref[2], ref_o[2], kind="grad")
    check("route.dv", dv, ref[3], ref_o[3], kind="grad")


# q of another length than k (one document per row), documents without a key for the first queries, and more documents than lanes
@pytest.mark.parametrize("lens_q,lens_k", [((40, 7, 90), (100, 7, 33)), ((1,) * 70, (5,) * 70), ((129,), (32,))])
@pytest.mark.parametrize("causal", [True, False])
def test_attention_routes_agree_on_unequal_lengths(lens_q, lens_k, causal):
    print(f"case unequal lengths q={lens_q} k={lens_k} causal={causal}", flush=True)
    g = torch.Generator().manual_seed(len(lens_q))
    nq, nkv, d = 4, 2, 64
    cu_q, cu_k = (torch.tensor([0] + list(torch.tensor(x).cumsum(0)), dtype=torch.int32, device=DEV) for x in (lens_q, lens_k))
    q, do = (torch.randn(sum(lens_q), nq, d, generator=g).half().to(DEV) for _ in range(2))
    k, v = (torch.randn(sum(lens_k), nkv, d, generator=g).half().to(DEV) for _ in range(2))
    out = []
    for flags in (SHORT, TILED):
        o, lse = ops.attention_forward(q, k, v, cu_q, cu_k, causal, None, flags=flags)
        out.append([o, lse] + list(ops.attention_backward(do, q, k, v, o, lse, cu_q, cu_k, causal, None, flags=flags)))
    for name, x, y in zip(("o", "lse", "dq", "dk", "dv"), *out):
        if name == "lse":
            assert torch.equal(torch.isinf(x), torch.isinf(y)) and torch.allclose(x, y, atol=1e-5)      # sums of exponentials in another order
        else:
            # probabilities and dS are rounded to float16 relative to other maxima: two roundings each way, 4 x 2^-11 in the 2-norm
            assert float((x.float() - y.float()).norm()) <= 2.0 ** -9 * float(y.float().norm()) + 1e-6, name


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("interleaved", [False, True])
def test_attention_routes_agree_with_rotary(d, interleaved):
    print(f"case routes rotary d={d} interleaved={interleaved}", flush=True)
    total, nq, nkv = 333, 8, 2
    g = torch.Generator().manual_seed(d)
    q, do = (torch.randn(total, nq, d, generator=g).bfloat16().to(DEV) for _ in range(2))
    k, v = (torch.randn(total, nkv, d, generator=g).bfloat16().to(DEV) for _ in range(2))
    cu = torch.tensor([0, 100, 101, 300, total], dtype=torch.int32)
    pos = U.position_ids_from_cu(cu, total).to(DEV)
    cu = cu.to(DEV)
    if interleaved:
        ang = torch.outer(torch.arange(512).float(), 1.0 / (10000.0 ** (torch.arange(0, d, 2).float() / d))).to(DEV)
        cos, sin = ang.cos().contiguous(), ang.sin().contiguous()
        k_rot = ops.rotary_embedding_complex(k, cos, sin, pos, total)
    else:
        tabs = oracle.rotary_tables(d, 512, 10000, torch.bfloat16)
        cos, sin = tabs.cos.to(DEV).view(512, d), tabs.sin.to(DEV).view(512, d)
        k_rot = ops.rotary_embedding(k, cos, sin, pos, total)
    out = []
    for flags in (SHORT, TILED):
        o, lse, q_rot = ops.attention_forward(q, k_rot, v, cu, None, True, None, rotary=(cos, sin, pos, None), flags=flags, return_rotated_q=True)
        out.append([o, lse, q_rot] + list(ops.attention_backward(do, q_rot, k_rot, v, o, lse, cu, None, True, None, flags=flags, rotary=(cos, sin, pos, pos))))
    fused, _ = ops.attention_forward(q, k, v, cu, None, True, None, rotary=(cos, sin, pos, pos), flags=SHORT)
    assert torch.equal(fused, out[0][0])                   # k rotated in the kernel or before it
    assert torch.equal(out[0][2], out[1][2])               # the same rotation, bit for bit
    for name, x, y in zip(("o", "lse", "q_rot", "dq", "dk", "dv"), *out):
        assert float((x.float() - y.float()).norm()) <= 2.0 ** -6 * float(y.float().norm()), name      # as above, bfloat16


# each side of the lines that choose between the two, forward and backward: (heads, KV heads, features, tokens, documents, causal) and the
# routes of a call that pins none
@pytest.mark.parametrize("nq,nkv,d,total,docs,causal,fwd,bwd", [
    (4, 4, 64, 8192, 1, True, SHORT, SHORT), (4, 4, 64, 8192, 1, False, SHORT, SHORT), (8, 8, 64, 8192, 1, False, TILED, TILED),
    (16, 16, 64, 4096, 8, True, SHORT, TILED),             # documents of whole blocks
    (16, 16, 64, 4095, 8, True, SHORT, SHORT), (32, 8, 64, 2048, 1, False, TILED, SHORT),
    (8, 8, 128, 4096, 1, True, SHORT, TILED), (8, 8, 128, 4096, 8, True, SHORT, TILED), (8, 8, 128, 4090, 20, True, SHORT, TILED),
    (8, 8, 128, 2048, 4, True, SHORT, TILED), (4, 4, 128, 8192, 1, False, TILED, TILED), (4, 4, 128, 4096, 1, False, SHORT, TILED),
    (4, 4, 128, 16384, 1, True, TILED, TILED), (32, 8, 128, 2048, 1, True, TILED, TILED), (32, 8, 128, 1056, 1, False, TILED, TILED),
    (8, 8, 128, 1152, 4, True, SHORT, SHORT), (4, 4, 128, 3584, 1, True, SHORT, SHORT), (32, 8, 128, 768, 1, False, SHORT, SHORT),
    (8, 8, 64, 16380, 40, True, TILED, SHORT),
])
def test_route_of_a_call(nq, nkv, d, total, docs, causal, fwd, bwd):
    print(f"case route of a call nq={nq} nkv={nkv} d={d} total={total} docs={docs} causal={causal}", flush=True)
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the lines are per compute unit; these sizes are for 256")
    g = torch.Generator(device=DEV).manual_seed(total)
    q, do = (torch.randn(total, nq, d, generator=g, device=DEV).bfloat16() for _ in range(2))
    k, v = (torch.randn(total, nkv, d, generator=g, device=DEV).bfloat16() for _ in range(2))
    cu = torch.tensor([total * i // docs for i in range(docs + 1)], dtype=torch.int32, device=DEV)
    o, lse = ops.attention_forward(q, k, v, cu, None, causal, None)
    dq, dk, dv = ops.attention_backward(do, q, k, v, o, lse, cu, None, causal, None)
    for flags in (SHORT, TILED):
        o2, _ = ops.attention_forward(q, k, v, cu, None, causal, None, flags=flags)
        grads = ops.attention_backward(do, q, k, v, o, lse, cu, None, causal, None, flags=flags)
        # sums in another order: some element of so many rounds the other way
        assert torch.equal(o, o2) == (flags == fwd)
        assert all(torch.equal(x, y) == (flags == bwd) for x, y in zip((dq, dk, dv), grads))


# sizes around the lines between the routes, which lie where measurements put them: whichever is taken is one of the two, bit for bit, and the
# two agree to the rounding of P and dS
@pytest.mark.parametrize("nq,nkv,d,total,docs,causal", [
    (8, 8, 128, 4096, 1, True), (8, 8, 128, 2048, 4, True), (4, 4, 128, 4096, 1, False), (32, 8, 128, 2048, 1, True), (12, 12, 96, 2560, 4, True),
    (16, 16, 64, 4190, 1, True), (32, 1, 64, 2520, 3, True), (12, 12, 128, 877, 16, True), (8, 8, 64, 6000, 20, False),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_backward_takes_one_of_two_routes_that_agree(nq, nkv, d, total, docs, causal, dtype):
    g = torch.Generator(device=DEV).manual_seed(total)
    q, do = (torch.randn(total, nq, d, generator=g, device=DEV).to(dtype) for _ in range(2))
    k, v = (torch.randn(total, nkv, d, generator=g, device=DEV).to(dtype) for _ in range(2))
    cu = torch.tensor([i * total // docs for i in range(docs + 1)], dtype=torch.int32, device=DEV)
    o, lse = ops.attention_forward(q, k, v, cu, None, causal, None)
    run = lambda flags: ops.attention_backward(do, q, k, v, o, lse, cu, None, causal, None, flags=flags)
    taken, short, tiled = run(0), run(SHORT), run(TILED)
    assert any(all(torch.equal(a, b) for a, b in zip(taken, route)) for route in (short, tiled))
    for name, a, b in zip(("dq", "dk", "dv"), short, tiled):
        # both round the same P and dS but for the last bits of their float32 sums, and each its own results: two roundings each way
        assert float((a.float() - b.float()).norm()) <= 2.0 ** (-6 if dtype == torch.bfloat16 else -9) * float(b.float().norm()), name


# where a launch in front of the dK / dV blocks leaves delta: one of its own for long chains, or the dQ blocks' (single long documents above
# 64 features, by the size of the call)
@pytest.mark.parametrize("nq,nkv,d,lens,flags,kernel", [
    (1, 1, 64, (1100,), SHORT, "attn_bwd_delta"), (8, 1, 32, (1021,), SHORT, None), (2, 1, 128, (530,), SHORT, "attn_bwd_delta"),
    (2, 1, 96, (500, 17), SHORT, None), (4, 4, 128, (3601,), 0, "attn_short_dq"), (16, 4, 128, (1663,), 0, "attn_short_dq"),
])
def test_backward_with_delta_of_another_launch(nq, nkv, d, lens, flags, kernel):
    print(f"case delta nq={nq} nkv={nkv} d={d} lens={lens} flags={flags}", flush=True)
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the lines are per compute unit; these sizes are for 256")
    g = torch.Generator(device=DEV).manual_seed(d)
    q, do = (torch.randn(sum(lens), nq, d, generator=g, device=DEV).half() for _ in range(2))
    k, v = (torch.randn(sum(lens), nkv, d, generator=g, device=DEV).half() for _ in range(2))
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32, device=DEV)
    o, lse = ops.attention_forward(q, k, v, cu, None, True, None)
    run = lambda f: ops.attention_backward(do, q, k, v, o, lse, cu, None, True, None, flags=f)
    grads, tiled, names = run(flags), run(TILED), launched(lambda: run(flags))
    assert any("attn_short_bwd" in n for n in names)
    assert [n for n in ("attn_bwd_delta", "attn_short_dq") if any(n in x for x in names)] == ([kernel] if kernel else [])
    for name, x, y in zip(("dq", "dk", "dv"), grads, tiled):
        # P and dS round the same values to float16 but for the last bits of delta and of their exponents: two roundings each way
        assert float((x.float() - y.float()).norm()) <= 2.0 ** -9 * float(y.float().norm()), name


@pytest.mark.parametrize("d", [32, 64, 96, 128])
@pytest.mark.parametrize("nq,nkv,dtype", [(2, 2, torch.float16), (3, 1, torch.bfloat16)])
def test_delta_is_the_same_whoever_forms_it(nq, nkv, d, dtype):
    """A document of 35 blocks of 32 rows: its gradients alone, where a launch in front leaves delta, have the bits they have beside seven short
    documents, where the blocks of the second launch form it."""
    g = torch.Generator(device=DEV).manual_seed(d)
    lens = (1120,) + 7 * (16,)
    q, do = (torch.randn(sum(lens), nq, d, generator=g, device=DEV).to(dtype) for _ in range(2))
    k, v = (torch.randn(sum(lens), nkv, d, generator=g, device=DEV).to(dtype) for _ in range(2))
    results = []
    for docs in (1, 8):
        n = sum(lens[:docs])
        cu = torch.tensor([0] + list(torch.tensor(lens[:docs]).cumsum(0)), dtype=torch.int32, device=DEV)
        rows = [t[:n].contiguous() for t in (do, q, k, v)]
        o, lse = ops.attention_forward(*rows[1:], cu, None, True, None, flags=SHORT)
        run = lambda: ops.attention_backward(*rows, o, lse, cu, None, True, None, flags=SHORT)
        assert any("attn_bwd_delta" in x for x in launched(run)) == (docs == 1)
        results.append([t[:lens[0]] for t in (o, *run())])
    for name, x, y in zip(("o", "dq", "dk", "dv"), *results):
        assert torch.equal(x, y), name


# float32 backward with dS kept by the dK/dV kernel (a workspace that has room for it) against the dQ kernel that recomputes it: the same
# bits.  Triangle and whole plane, documents that end inside tiles, keys and queries of different lengths (rows that see nothing among
# them), few KV heads, several passes over the heads (4128 tokens of 64 heads; 8192 of 12 and 16384 of 8, whose passes alone have fewer
# query blocks than decide for a split of the keys), each head_dim.
@pytest.mark.parametrize("nq,nkv,d,causal,lens_q,lens_k", [
    (32, 32, 128, True, [1101], None), (32, 32, 64, False, [500, 37, 590], None), (64, 32, 96, True, [33, 1, 700, 331], None),
    (16, 16, 128, True, [1000, 1200, 3], [900, 1300, 2]), (16, 16, 64, False, [700, 900], [1500, 617]), (16, 1, 128, True, [4099], None),
    (64, 64, 64, True, [4128], None), (12, 12, 64, True, [8192], None), (12, 12, 96, False, [8190], None), (8, 8, 64, True, [16384], None),
])
def test_float32_backward_with_kept_scores(nq, nkv, d, causal, lens_q, lens_k):
    print(f"case f32 kept nq={nq} nkv={nkv} d={d} causal={causal} q={lens_q} k={lens_k}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(d + nq)
    cu = lambda lens: torch.tensor([0] + lens, dtype=torch.int32, device="cuda").cumsum(0, dtype=torch.int32)
    cu_q, cu_k = cu(lens_q), None if lens_k is None else cu(lens_k)
    tq, tk = sum(lens_q), sum(lens_k or lens_q)
    rand = lambda n, h: torch.randn(n, h, d, generator=g, device="cuda")
    q, k, v, do = rand(tq, nq), rand(tk, nkv), rand(tk, nkv), rand(tq, nq)
    o, lse = ops.attention_forward(q, k, v, cu_q, cu_k, causal)
    lib = _lib.load()
    least = lib.mi_attn_bwd_workspace_bytes_kv(tq, tk, nq, nkv, d)
    best = lib.mi_attn_bwd_workspace_bytes_for(ops._fill_attn_args(q, k, v, o, lse, cu_q, cu_k, causal, 1.0 / d ** 0.5))
    room = (least + 255) // 256 * 64                       # dS lies behind what the smaller workspace holds
    assert best > least
    run = lambda bytes_: (torch.empty_like(q), torch.empty_like(k), torch.empty_like(v), torch.full(((bytes_ + 3) // 4,), float("nan"), device="cuda"))
    small, large = run(least), run(best)
    want = ops.attention_backward(do, q, k, v, o, lse, cu_q, cu_k, causal, buffers=small)
    got = ops.attention_backward(do, q, k, v, o, lse, cu_q, cu_k, causal, buffers=large)
    kept = large[3][room:]
    assert bool((kept == kept).any()), "the kept route was not taken"
    own = ops.attention_backward(do, q, k, v, o, lse, cu_q, cu_k, causal)
    assert all(torch.equal(a, b) for a, b in zip(got, own))
    for name, a, b in zip(("dq", "dk", "dv"), got, want):
        assert torch.equal(a, b), f"{name}: {(a - b).abs().max().item()}"


def test_float32_backward_in_a_program_near_its_limit():
    """Where the room for dS is not there the pass takes the small workspace at once: nothing is thrown out of the allocator's cache, the bits stay."""
    g = torch.Generator(device="cuda").manual_seed(1)
    q, do = (torch.randn(4096, 32, 64, generator=g, device="cuda") for _ in range(2))
    k, v = (torch.randn(4096, 32, 64, generator=g, device="cuda") for _ in range(2))
    cu = torch.tensor([0, 4096], dtype=torch.int32, device="cuda")
    for t in (q, k, v):
        t.requires_grad_()
    o = ops.attention(q, k, v, cu)
    grads = lambda: torch.autograd.grad(o, (q, k, v), do, retain_graph=True)
    want = grads()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    try:
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (512 << 20)) / total)
        cached = torch.empty(64 << 20, dtype=torch.uint8, device="cuda")        # a block of the cache, for the next step
        del cached
        before = torch.cuda.memory_stats()
        for _ in range(3):
            got = grads()
        after = torch.cuda.memory_stats()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert all(after[n] == before[n] for n in ("num_alloc_retries", "num_ooms")), (before["num_alloc_retries"], after["num_alloc_retries"])
    assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_float32_step_with_kept_scores_in_a_graph():
    """The room for dS comes from the graph's own pool: replays between eager steps give the eager bits."""
    g = torch.Generator(device="cuda").manual_seed(1)
    q, k, v, do = (torch.randn(1101, 32, 64, generator=g, device="cuda") for _ in range(4))
    cu = torch.tensor([0, 600, 1101], dtype=torch.int32, device="cuda")
    for t in (q, k, v):
        t.requires_grad_()
    step = lambda: torch.autograd.grad(ops.attention(q, k, v, cu), (q, k, v), do)
    want = step()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = step()
    for _ in range(3):
        for t in got:
            t.zero_()
        graph.replay()
        assert all(torch.equal(a, b) for a, b in zip(step(), want))
        assert all(torch.equal(a, b) for a, b in zip(got, want))


# blocks of two wavefronts, and which way goes to them: a last block that is not whole, empty documents, one much longer than the others, q of another
# length than k, rotary on the load of q
@pytest.mark.parametrize("nq,nkv,d,total,docs,causal,fwd,bwd", [
    (24, 24, 64, 2081, 9, True, 2, 2), (24, 24, 64, 2049, 9, False, 4, 2), (16, 4, 128, 2600, 13, True, 2, 4), (12, 12, 32, 2500, 20, False, 4, 2),
    (12, 12, 64, 2047, 6, True, 4, 2), (12, 12, 64, 2047, 5, True, 4, 4), (16, 16, 96, 2561, 30, True, 2, 4), (32, 32, 64, 4096, 40, True, 2, 2),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("kind", ["self", "cross", "rotary"])
def test_blocks_of_two_wavefronts(nq, nkv, d, total, docs, causal, fwd, bwd, dtype, kind):
    print(f"case two wavefronts nq={nq} nkv={nkv} d={d} total={total} docs={docs} causal={causal} {dtype} {kind}", flush=True)
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the lines are per compute unit; these sizes are for 256")
    if kind == "rotary" and d not in (64, 128):
        pytest.skip("rotary inside: 64 and 128 features")
    g = torch.Generator(device=DEV).manual_seed(total)
    cut = [0] + sorted(random.Random(docs).sample(range(1, total), docs - 2)) + [total, total]              # the last document is empty
    cu = torch.tensor(cut, dtype=torch.int32, device=DEV)
    cu_k = torch.clamp(cu, max=total - 40) if kind == "cross" else cu
    total_k = int(cu_k[-1])
    q, do = (torch.randn(total, nq, d, generator=g, device=DEV).to(dtype) for _ in range(2))
    k, v = (torch.randn(total_k, nkv, d, generator=g, device=DEV).to(dtype) for _ in range(2))
    forward = backward = {}
    if kind == "rotary":
        tabs = oracle.rotary_tables(d, total, 10000, dtype)
        cos, sin, pos = tabs.cos.to(DEV).view(total, d), tabs.sin.to(DEV).view(total, d), torch.arange(total, device=DEV)
        k = ops.rotary_embedding(k, cos, sin, pos, total)
        forward, backward = dict(rotary=(cos, sin, pos, None), return_rotated_q=True), dict(rotary=(cos, sin, pos, pos))
    out = []
    for flags in (SHORT, TILED):
        names = []
        run = lambda: ops.attention_forward(q, k, v, cu, cu_k, causal, None, flags=flags, **forward)
        o, lse, *rotated = run()
        qr = rotated[0] if rotated else q
        grads = lambda: ops.attention_backward(do, qr, k, v, o, lse, cu, cu_k, causal, None, flags=flags, **backward)
        out.append([o, *rotated, *grads()])
        if flags == SHORT:
            names = launched(lambda: (run(), grads()))
            assert any(f"attn_short_fwd_kernel<{d}, {1 if kind == 'rotary' else 0}, false, {fwd}>" in n for n in names), names
            assert any(f"attn_short_bwd_kernel<{d}, {bwd}, " in n for n in names), names
    for i, (a, b) in enumerate(zip(*out)):
        # as above: the two round the same P and dS and their own results
        assert float((a.float() - b.float()).norm()) <= 2.0 ** (-6 if dtype == torch.bfloat16 else -9) * float(b.float().norm()) + 1e-6, i
