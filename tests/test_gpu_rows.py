"""Products of a few rows (mi_rows_product, and ops.linear / ops.projections that reach it) against float64 products of the same rounded
operands, and a native decode step of a layer against the modules it stands for."""

import ctypes

import pytest
import torch

from scaling_amd import _lib, ops
from scaling_amd.config import TransformerArchitectureConfig
from scaling_amd.inference import TransformerInferenceModule

pytestmark = pytest.mark.gpu
DEV = "cuda"
HALF_ULP = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def _rand(shape, dtype, seed, std=1.0):
    return (torch.randn(shape, generator=torch.Generator(device=DEV).manual_seed(seed), device=DEV) * std).to(dtype)


# contractions: one product, fewer than wavefronts, a last wavefront with less than the others, several rounds of prefetch; widths of
# less than a block of 16, ragged, past the line of four (1024 blocks) and of two-block (2048 blocks) workgroups
@pytest.mark.parametrize("rows,k,outs", [(1, 32, (8,)), (16, 96, (24, 8, 40)), (3, 1056, (1032, 264)), (5, 4096, (72,)), (2, 2816, (16, 16, 16400)),
                                         (16, 544, (33000,)),
                                         # past 16 rows: the tiled kernel
                                         (17, 3064, (72, 40)), (17, 3072, (72, 40))])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_few_rows_through_linear(rows, k, outs, dtype):
    print(f"case rows rows={rows} k={k} outs={outs} dtype={dtype}", flush=True)
    x, ws = _rand((rows, k), dtype, 1), [_rand((o, k), dtype, 2 + i, 0.1) for i, o in enumerate(outs)]
    bs = [_rand((o,), dtype, 9) if i != 1 else None for i, o in enumerate(outs)]
    res = _rand((rows, outs[0]), dtype, 10)
    got = ops.projections(x, ws, bs) + [ops.linear(x, ws[0], bs[0], res)]
    for i, y in enumerate(got):
        w, b = (ws + ws)[i] if i < len(ws) else ws[0], bs[i] if i < len(ws) else bs[0]
        ref, mag = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
        if b is not None:
            ref, mag = ref + b.double(), mag + b.double().abs()
        bound = HALF_ULP[dtype] * ref.abs() + (k + 1) * 2.0 ** -24 * mag + 2.0 ** -25
        if i == len(ws):                                   # the rounded product, then one more rounding of the sum
            ref = ref + res.double()
            bound = bound + HALF_ULP[dtype] * (ref.abs() + bound)
        assert bool(((y.double() - ref).abs() <= bound * 1.001).all()), i


@pytest.mark.parametrize("rows,k,n,glu", [(1, 32, 16, True), (3, 1024, 2816, True), (16, 288, 40, False), (7, 2048, 50257, False), (4, 64, 16416, True)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_few_rows_with_norm(rows, k, n, glu, dtype):
    print(f"case rows norm rows={rows} k={k} n={n} glu={glu} dtype={dtype}", flush=True)
    store = _rand((rows, 3, k), dtype, 3)
    x, g = store[:, 1], (1.0 + _rand((k,), torch.float32, 4, 0.1)).to(dtype)       # rows of a larger tensor
    ws = [_rand((n, k), dtype, 5 + i, k ** -0.5) for i in range(2)]
    out, count = torch.empty(rows, n, dtype=dtype, device=DEV), torch.arange(rows, dtype=torch.int32, device=DEV)
    a = _lib.MiRowsArgs()
    a.x, a.norm_weight, a.ldx, a.k, a.rows, a.eps, a.glu = x.data_ptr(), g.data_ptr(), x.stride(0), k, rows, 1e-5, int(glu)
    a.n_weights, a.dtype, a.stream, a.count_up = 1 + int(glu), _lib.dtype_code(dtype), _lib.stream_ptr(), count.data_ptr()
    for i in range(1 + int(glu)):
        a.w[i], a.n[i], a.ldw[i], a.out[i], a.ldo[i] = ws[i].data_ptr(), n, k, out.data_ptr(), n
    _lib.check(_lib.load().mi_rows_product(ctypes.byref(a)), "mi_rows_product")
    xd = x.double()
    normed = (xd * torch.rsqrt(xd.square().mean(-1, keepdim=True) + 1e-5) * g.double()).to(dtype).double()
    p = [normed @ w.double().t() for w in ws]
    u = HALF_ULP[dtype]
    # a normalised element may round to the neighbour where float32 and float64 norms straddle a tie: 2 u of its size
    e = [u * p[i].abs() + (2 * u + (k + 1) * 2.0 ** -24) * (normed.abs() @ ws[i].double().abs().t()) for i in range(2)]
    ref, bound = p[0], e[0]
    if glu:
        silu = torch.nn.functional.silu(p[0])
        ref = silu * p[1]
        bound = 1.1 * e[0] * (p[1].abs() + e[1]) + silu.abs() * e[1] + 2 * u * ref.abs()     # |silu'| < 1.1
    err = (out.double() - ref).abs()
    assert bool((err <= bound * 1.01 + 2.0 ** -25).all())
    assert float(err.norm() / ref.norm()) < 3 * u                                     # the bound's straddled ties are few
    assert count.tolist() == list(range(1, rows + 1))
    a.k = 33
    assert _lib.load().mi_rows_product(ctypes.byref(a)) == -3


# both sides of the lines between whole, half and quarter blocks (64, 128, 256 and 384 of 16 features); slices that are shorter than others or empty
@pytest.mark.parametrize("rows,k,n,glu", [(1, 32, 5, False), (4, 2816, 1024, True), (4, 544, 1025, False), (5, 544, 1024, False), (8, 1056, 2048, True),
                                          (8, 96, 2049, False), (3, 64, 4097, False), (8, 2080, 6144, True), (2, 352, 6145, False)])
@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_folded_rows_equal_whole_blocks(rows, k, n, glu, norm, dtype):
    """More than 8 rows are not folded, and a row's results do not depend on the others: the same to the bit, infinite weights included."""
    x, g = _rand((16, k), dtype, 3), (1.0 + _rand((k,), torch.float32, 4, 0.1)).to(dtype)
    ws = [_rand((n, k), dtype, 5 + i, k ** -0.5) for i in range(2)]
    ws[0][n // 2, k - 1] = float("inf")
    bias, add = _rand((n,), dtype, 7), _rand((16, n), dtype, 8)

    def product(count):
        out = torch.full((count, n), 3.0, dtype=dtype, device=DEV)
        a = _lib.MiRowsArgs()
        a.x, a.norm_weight, a.ldx, a.k, a.rows, a.eps, a.glu = x.data_ptr(), g.data_ptr() if norm else None, k, k, count, 1e-5, int(glu)
        a.n_weights, a.dtype, a.stream = 1 + int(glu), _lib.dtype_code(dtype), _lib.stream_ptr()
        for i in range(1 + int(glu)):
            a.w[i], a.n[i], a.ldw[i], a.out[i], a.ldo[i] = ws[i].data_ptr(), n, k, out.data_ptr(), n
        if not glu:
            a.bias[0], a.add[0], a.ldadd[0] = bias.data_ptr(), add.data_ptr(), n
        _lib.check(_lib.load().mi_rows_product(ctypes.byref(a)), "mi_rows_product")
        return out
    got, want = product(rows), product(16)[:rows]
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(), want.nan_to_num())
    assert int((~want.isfinite()).sum()) <= rows


# each side of the lines between the norm inside the product and a launch of its own: (features, k)
@pytest.mark.parametrize("n,k,inside", [(4096, 2048, True), (4097, 2048, False), (8192, 1024, True), (8200, 1024, False), (16, 2080, False),
                                        (1536, 4096, False), (1000, 288, True)])
def test_norm_in_front_of_a_product(n, k, inside):
    print(f"case norm in front n={n} k={k}", flush=True)
    x, w = _rand((5, k), torch.bfloat16, 1), _rand((n, k), torch.bfloat16, 2, k ** -0.5)
    g = (1.0 + _rand((k,), torch.float32, 4, 0.1)).bfloat16()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        out = ops.norm_linear_rows(x, g, 1e-5, w)
        torch.cuda.synchronize()
    names = [e.key for e in prof.key_averages() if "kernel" in e.key]
    assert any("rows_kernel" in name for name in names) and any("rmsnorm" in name for name in names) == (not inside), names
    xd = x.double()
    normed = (xd * torch.rsqrt(xd.square().mean(-1, keepdim=True) + 1e-5) * g.double()).bfloat16().double()
    ref, mag = normed @ w.double().t(), normed.abs() @ w.double().abs().t()
    u = HALF_ULP[torch.bfloat16]
    # as in test_few_rows_with_norm: a normalised element may round to the neighbour
    err = (out.double() - ref).abs()
    assert bool((err <= (u * ref.abs() + (2 * u + (k + 1) * 2.0 ** -24) * mag) * 1.01).all())
    assert float(err.norm() / ref.norm()) < 3 * u


@pytest.mark.parametrize("batch,heads,kv,dtype", [(1, 4, 2, torch.bfloat16), (3, 8, 8, torch.float16), (16, 4, 1, torch.bfloat16), (17, 4, 2, torch.bfloat16)])
def test_native_decode_step_equals_the_modules(batch, heads, kv, dtype):
    print(f"case native decode batch={batch} heads={heads}/{kv} dtype={dtype}", flush=True)
    hidden = 64 * heads
    cfg = TransformerArchitectureConfig.from_dict(dict(
        vocab_size=1003, hidden_size=hidden, num_layers=2, num_attention_heads=heads, attention_num_kv_heads=kv, attention_qkv_in_one=False,
        norm_type="rms", mlp_type="swiglu", mlp_factor=2.75, attention_bias=False, mlp_bias=False, sequence_length=64,
        precision="bfloat16" if dtype == torch.bfloat16 else "float16", weight_tying=True, masked_softmax={"kernel": "hip"}))
    model = TransformerInferenceModule(cfg, device=DEV, init_std=0.05, seed=3)
    with torch.no_grad():
        model._layers[0].embedding.weight.mul_(20.0)       # tied embeddings of unit scale: a sure greedy choice
    ids = torch.randint(1, 1003, (batch, 9), generator=torch.Generator().manual_seed(batch))
    tokens, logits = model.generate(6, ids)
    caches = [layer.self_attention.cache[0] for layer in model._layers[1:-2]]
    native = [(c.k.clone(), c.v.clone(), c.ctx_len.clone(), c.length) for c in caches]
    calls = []
    handles = [layer.mlp.register_forward_hook(lambda *a: calls.append(1)) for layer in model._layers[1:-2]]   # a hooked module is called
    tokens2, logits2 = model.generate(6, ids)
    for h in handles:
        h.remove()
    assert len(calls) == 12 and tokens == tokens2
    tol = 4 * HALF_ULP[dtype]                              # two layers, each with two rounded residual sums
    assert float((logits.float() - logits2.float()).norm() / logits2.float().norm()) < tol
    for c, (k, v, ctx, length) in zip(caches, native):
        assert torch.equal(c.ctx_len, ctx) and c.length == length == 14
        for x, y in ((c.k, k), (c.v, v)):
            assert float((x.float() - y.float()).norm() / x.float().norm()) < tol
    short, _ = model.generate(6, ids[:1], stop_tokens=[tokens[0][2]])
    assert short[0] == tokens[0][:tokens[0].index(tokens[0][2]) + 1]


# one vector, less than a wavefront, both sides of a round of 1024 threads x 8 vectors, rows off a 16-byte boundary
@pytest.mark.parametrize("rows,n,offset", [(1, 1, 0), (3, 7, 1), (4, 1000, 3), (16, 32000, 0), (5, 65537, 2), (2, 131072 + 9, 0), (300, 515, 5)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_argmax_of_rows(rows, n, offset, dtype):
    print(f"case argmax rows={rows} n={n} offset={offset} dtype={dtype}", flush=True)
    x = _rand((rows * (n + offset) + offset,), dtype, n)[offset:].view(rows, n + offset)[:, :n]
    cases = [x, x.clone().clamp_(max=0.0), torch.full_like(x, -float("inf")), -torch.zeros_like(x)]     # ties from clamping, at -inf and at -0
    if n > 8:
        at = torch.randint(0, n, (rows, 2), generator=torch.Generator(device=DEV).manual_seed(1), device=DEV)
        cases += [x.scatter(1, at, float("inf")), x.scatter(1, at, float("nan")), cases[3].scatter(1, at, 0.0)]
    for i, c in enumerate(cases):
        ref = torch.argmax(c.float().cpu(), dim=-1)
        if i == 6:
            assert ref.tolist() == [0] * rows              # -0 and +0 are equal
        assert torch.equal(ops.argmax_rows(c).cpu(), ref), i
    assert ops.argmax_rows(x[:0]).numel() == 0


# one vector, more of them than threads, a padded table with more rows than are chosen from
@pytest.mark.parametrize("rows,n,hidden,pad", [(1, 1, 8, 0), (3, 32000, 1024, 0), (5, 1001, 12288, 8), (300, 515, 264, 16)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_argmax_with_its_embedding(rows, n, hidden, pad, dtype):
    x, table = _rand((rows, n), dtype, n), _rand((n + 3, hidden + pad), dtype, 2)[:, :hidden]
    x[0, n // 2] = float("nan")                            # above everything
    with torch.no_grad():
        index, out = ops.argmax_embed(x, table)
        assert torch.equal(index, ops.argmax_rows(x)) and int(index[0]) == n // 2 and torch.equal(out, table[index])
        for refused in (table[:n - 1], table[:, :hidden - 1], table.double(), table.t()):
            assert ops.argmax_embed(x, refused) is None
    assert ops.argmax_embed(x, table.clone().requires_grad_()) is None


def test_generation_calls_a_watched_embedding():
    cfg = TransformerArchitectureConfig.from_dict(dict(
        vocab_size=512, hidden_size=256, num_layers=2, num_attention_heads=4, attention_num_kv_heads=2, sequence_length=64, precision="bfloat16", norm_type="rms",
        mlp_type="swiglu", mlp_factor=2.75, attention_bias=False, mlp_bias=False, attention_qkv_in_one=False, masked_softmax={"kernel": "hip"}))
    model, ids, calls = TransformerInferenceModule(cfg, DEV, seed=3), torch.arange(1, 21).view(2, 10), []
    tokens, logits = model.generate(6, ids)
    handle = model._layers[0].embedding.register_forward_hook(lambda *a: calls.append(1))
    tokens2, logits2 = model.generate(6, ids)
    handle.remove()
    assert len(calls) == 6 and tokens == tokens2 and torch.equal(logits, logits2)
