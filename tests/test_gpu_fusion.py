"""Fused launches of the layer step against the separate launches they replace: residual add + norm (forward and
backward), the packed-QKV attention node, column sums."""

from unittest import mock

import pytest
import torch

from scaling_amd import _lib, ops
from scaling_amd.config import RotaryConfig, TransformerArchitectureConfig
from scaling_amd.layer import InferenceSettings, TransformerLayer, TransformerLayerIO
from scaling_amd.nn import KVCache, RotaryEmbedding
from tests.kernels import launched

pytestmark = pytest.mark.gpu
DEV = "cuda"


# one per tiling of the norm kernels: 16 and 64 lanes a row, wide rows of one and two vectors per thread at each width
@pytest.mark.parametrize("rows,hidden", [(1, 64), (7, 264), (257, 1024), (1025, 2048), (300, 4096), (33, 8192), (5, 12288)])
@pytest.mark.parametrize("layer_norm", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_residual_through_the_norm_matches_separate_launches(rows, hidden, layer_norm, dtype):
    if dtype == torch.float32:
        hidden = min(hidden, 8192)           # the widest float32 row the norms take
    print(f"case add_norm rows={rows} hidden={hidden} layer_norm={layer_norm} dtype={dtype}", flush=True)
    g = torch.Generator().manual_seed(rows + hidden)
    x, r, dy, ds = (torch.randn(rows, hidden, generator=g).to(dtype).to(DEV) for _ in range(4))
    w, b = ((k + 0.1 * torch.randn(hidden, generator=g)).to(dtype).to(DEV) for k in (1.0, 0.0))
    b = b if layer_norm else None

    def separate(with_residual):
        a, c, wt = x.clone().requires_grad_(), r.clone().requires_grad_(), w.clone().requires_grad_()
        bt = b.clone().requires_grad_() if b is not None else None
        s = a + c if with_residual else a
        y = ops.layer_norm(s, wt, bt, 1e-5) if layer_norm else ops.rms_norm(s, wt, 1e-5)
        torch.autograd.backward([s * 1.0, y], [ds, dy])
        return [s.detach(), y.detach(), a.grad, c.grad, wt.grad, bt.grad if bt is not None else None]

    def fused(with_residual):
        a, c, wt = x.clone().requires_grad_(), r.clone().requires_grad_(), w.clone().requires_grad_()
        bt = b.clone().requires_grad_() if b is not None else None
        s, y = ops.add_norm(a, c if with_residual else None, wt, bt, 1e-5, layer_norm)
        torch.autograd.backward([s, y], [ds, dy])
        return [s.detach(), y.detach(), a.grad, c.grad, wt.grad, bt.grad if bt is not None else None]

    for with_residual in (True, False):
        for name, want, got in zip(("sum", "y", "dx", "dresidual", "dw", "db"), separate(with_residual), fused(with_residual)):
            assert (want is None) == (got is None), name
            if want is None:
                continue
            if dtype == torch.float32 and name in ("dx", "dresidual"):
                # the compiler contracts the norm's last multiplication with the added gradient: the fused result lacks the
                # rounding of the norm's dx (half an ulp of it), and each side rounds its own sum (half an ulp each)
                bound = 2.0 ** -24 * (1.01 * (want - ds).abs() + 2.01 * want.abs()) + 2.0 ** -126
                assert bool(((want - got).abs() <= bound).all()), (name, with_residual)
            else:                            # the same arithmetic in the same order: the same bits
                assert torch.equal(want, got), (name, with_residual)


def test_norm_outputs_that_do_not_reach_the_loss():
    x = torch.randn(9, 128, device=DEV, requires_grad=True)
    w = torch.ones(128, device=DEV, requires_grad=True)
    s, y = ops.add_norm(x, None, w, None, 1e-5, False)
    s.sum().backward()
    assert torch.equal(x.grad, torch.ones_like(x)) and w.grad is None
    x.grad = None
    s, y = ops.add_norm(x, x, w, None, 1e-5, False)          # both addends are the same tensor
    y.sum().backward()
    a = x.detach().clone().requires_grad_()
    ops.rms_norm(a + a, w.detach(), 1e-5).sum().backward()
    assert torch.equal(x.grad, a.grad)


def _offset(t):
    """The same values one element off a 16-byte boundary."""
    flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:]
    return flat.copy_(t.reshape(-1)).view(t.shape)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("layer_norm", [False, True])
def test_residual_stream_off_a_vector_boundary(layer_norm, dtype):
    """A sum takes its addends and its gradient wherever they lie: the same bits."""
    g = torch.Generator(DEV).manual_seed(5)
    x, r, dy, ds = (torch.randn(37, 264, generator=g, device=DEV).to(dtype) for _ in range(4))
    w = torch.ones(264, dtype=dtype, device=DEV, requires_grad=True)
    out = []
    for place in (lambda t: t, _offset):
        a, c = place(x).requires_grad_(), place(r).requires_grad_()
        s, y = ops.add_norm(a, c, w, None, 1e-5, layer_norm)
        out.append([s, y] + list(torch.autograd.grad([s, y], [a, c, w], [place(ds), dy])))
    assert all(torch.equal(p, q) for p, q in zip(*out))


def _layer(dtype, default, hidden=256, inter=2.75, heads=4, **options):
    """The default block (LayerNorm, one QKV projection, GELU MLP, biases) or RMSNorm, grouped heads, SwiGLU without biases."""
    torch.manual_seed(7)
    own = dict(mlp_type="default", mlp_factor=4.0) if default else dict(norm_type="rms", mlp_type="swiglu", mlp_factor=inter, attention_bias=False,
                                                                        mlp_bias=False, attention_qkv_in_one=False, attention_num_kv_heads=heads // 2)
    cfg = TransformerArchitectureConfig.from_dict(dict(
        vocab_size=64, hidden_size=hidden, num_layers=1, num_attention_heads=heads, sequence_length=512, precision=dtype,
        dropout_embedding=0.0, dropout_attention_probs=0.0, dropout_after_attention=0.0, dropout_after_mlp=0.0,
        masked_softmax={"kernel": "hip"}, **own, **options))
    return TransformerLayer(cfg, 0, device=torch.device(DEV))


def _io(x):
    b, s, _ = x.shape
    return TransformerLayerIO(activations=x, position_ids=torch.arange(s, device=DEV).repeat(b, 1),
                              cumulative_seq_lengths=torch.arange(0, b * s + 1, s, dtype=torch.int32, device=DEV))


def _step(layer, forward, x, dy):
    """Output and every gradient of one step."""
    layer.zero_grad(set_to_none=True)
    x = x.clone().requires_grad_()
    y = forward(x)
    y.backward(dy)
    return [y.detach(), x.grad] + [p.grad for p in layer.parameters()]


def _blocks(layer, x):
    """The layer's two blocks, with every residual sum a launch of its own."""
    io = _io(x)
    return layer.mlp_block(layer.attention_block(io.activations, io.cumulative_seq_lengths, io.position_ids))


@pytest.mark.parametrize("default", [True, False])
def test_layer_with_an_output_gradient_off_a_vector_boundary(default):
    """Every product of that gradient moves to the library: float32 sums in another order."""
    layer = _layer("float32", default)
    x, dy = (torch.randn(2, 100, 256, device=DEV, generator=torch.Generator(DEV).manual_seed(s)) for s in (1, 2))
    for p, q in zip(_step(layer, lambda t: layer(_io(t)).activations, x, dy), _step(layer, lambda t: layer(_io(t)).activations, x, _offset(dy))):
        assert float((p - q).norm()) <= 1e-5 * float(p.norm()) + 1e-4     # the gradient of a key bias is a sum that cancels to nothing


@pytest.mark.parametrize("default", [True, False])
def test_float32_layer_under_autocast(default):
    """The projections run in bf16 and the residual stream stays float32.  The fused norms' float32 input gradients may differ in the
    last place, which can turn a bf16 rounding further down: less than one such rounding of a gradient altogether."""
    layer = _layer("float32", default)
    x, dy = (torch.randn(2, 100, 256, device=DEV, generator=torch.Generator(DEV).manual_seed(s)) for s in (1, 2))
    with torch.autocast("cuda", dtype=torch.bfloat16):
        want, got = _step(layer, lambda t: _blocks(layer, t), x, dy), _step(layer, lambda t: layer(_io(t)).activations, x, dy)
    assert got[0].dtype == torch.float32 and torch.equal(want[0], got[0])
    for a, b in zip(want, got):
        assert a.dtype == b.dtype and float((a - b).norm()) <= 2.0 ** -8 * float(a.norm())


@pytest.mark.parametrize("default", [True, False])
@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
def test_layer_with_activations_kept_on_the_host(default, dtype):
    """What saved-tensor hooks bring back has other addresses and may have other strides; the step is the same to the bit."""
    layer = _layer(dtype, default)
    x, dy = (torch.randn(2, 100, 256, device=DEV, generator=torch.Generator(DEV).manual_seed(s)).to(getattr(torch, dtype)) for s in (1, 2))

    def forward(t):
        return layer(_io(t)).activations
    want = _step(layer, forward, x, dy)
    with torch.autograd.graph.save_on_cpu():
        got = _step(layer, forward, x, dy)
    assert all(torch.equal(a, b) for a, b in zip(want, got))


def _watch(layer, how, path, calls):
    """Lets `calls` see every call of the module at `path`; returns what undoes a global registration."""
    name = path.split(".")[-1]
    parent = layer.get_submodule(path[:-len(name)].rstrip("."))
    module = getattr(parent, name)
    if how == "hook":
        module.register_forward_hook(lambda m, a, y: calls.append(path))
    elif how == "global hook":
        return torch.nn.modules.module.register_module_forward_hook(lambda m, a, y: calls.append(path) if m is module else None)
    elif how == "own forward":
        inner = module.forward
        module.forward = lambda *a, **k: (calls.append(path), inner(*a, **k))[1]
    else:
        class Replacement(torch.nn.Module):
            def __init__(self):
                super().__init__()
                self.inner = module

            def forward(self, x):
                calls.append(path)
                return self.inner(x)
        setattr(parent, name, Replacement())


WATCHED = ["input_layernorm", "post_attention_layernorm", "dropout_attention", "dropout_mlp", "self_attention.dense", "mlp", "mlp.dense_in",
           "mlp.siglu_weight", "mlp.dense_out"]


@pytest.mark.parametrize("how", ["hook", "global hook", "own forward", "replaced"])
@pytest.mark.parametrize("path", WATCHED + ["self_attention.query", "self_attention.value"])
def test_watched_or_replaced_modules_are_called(how, path):
    """A module that somebody observes or replaces is called in a training step and (but for the stacked q / k / v of inference) in a
    cached decode step, whose results stay what they were."""
    print(f"case watched {how} {path}", flush=True)
    layer = _layer("bfloat16", False)
    x, dy = (torch.randn(2, 40, 256, device=DEV, generator=torch.Generator(DEV).manual_seed(s)).bfloat16() for s in (1, 2))

    def decode():
        layer.eval()
        with torch.no_grad():
            io = _io(x)
            io.inference_settings = InferenceSettings(use_cache=True, reset_cache=True)
            layer(io)
            calls.clear()
            one = TransformerLayerIO(activations=x[:, :1].contiguous(), position_ids=torch.full((2, 1), 40, device=DEV),
                                     cumulative_seq_lengths=torch.arange(3, dtype=torch.int32, device=DEV),
                                     inference_settings=InferenceSettings(use_cache=True, reset_cache=False))
            y = layer(one).activations
        layer.train()
        return y
    calls = []
    want, token = _step(layer, lambda t: layer(_io(t)).activations, x, dy), decode()
    handle = _watch(layer, how, path, calls)
    try:
        calls.clear()
        got = _step(layer, lambda t: layer(_io(t)).activations, x, dy)
        assert calls == [path]
        # the same outputs; gradients of projections that share their input are rounded before they are summed, and the products of a
        # decode step are summed in another order: one rounding at each of the eight places where either stores a result
        assert torch.equal(want[0], got[0])
        assert float((want[1] - got[1]).float().norm()) <= 8 * 2.0 ** -8 * float(want[1].float().norm())
        if path in WATCHED:
            y = decode()
            assert calls == [path]
            assert float((y - token).float().norm()) <= 8 * 2.0 ** -8 * float(token.float().norm())
    finally:
        if handle is not None:
            handle.remove()


class _WideProjection(torch.nn.Module):
    """The projection `inner` as the first columns of a wider product."""

    def __init__(self, inner):
        super().__init__()
        self.inner = inner

    def forward(self, x):
        y = self.inner(x)
        return torch.cat([y, y[..., :8]], -1)[..., :y.shape[-1]]


class _OwnCore(torch.nn.Module):
    """An attention core with the token-major call alone."""

    def __init__(self, inner):
        super().__init__()
        self.inner, self.called = inner, 0

    def forward_tokens(self, *args, **kw):
        self.called += 1
        return self.inner.forward_tokens(*args, **kw)


@pytest.mark.parametrize("how", ["projection", "core", "core's method"])
def test_packed_qkv_with_a_replaced_projection_or_core(how):
    layer = _layer("bfloat16", True)
    x, dy = (torch.randn(2, 40, 256, device=DEV, generator=torch.Generator(DEV).manual_seed(s)).bfloat16() for s in (1, 2))

    def forward(t):
        return layer(_io(t)).activations
    want = _step(layer, forward, x, dy)
    att = layer.self_attention
    core, calls = att.scaled_dot_product_attention, []
    if how == "projection":
        att.query_key_value = _WideProjection(att.query_key_value)
    elif how == "core":
        att.scaled_dot_product_attention = _OwnCore(core)
    else:
        own = core.forward_tokens
        core.forward_tokens = lambda *a, **k: (calls.append(1), own(*a, **k))[1]
    got = _step(layer, forward, x, dy)
    assert torch.equal(want[0], got[0]) and torch.equal(want[1], got[1])
    assert how == "projection" or (calls or att.scaled_dot_product_attention.called == 1)


@pytest.mark.parametrize("heads,d,rotary,causal,docs", [(3, 64, True, True, (40,)), (2, 128, True, False, ()), (2, 96, False, True, (7, 100)), (4, 32, False, True, ())])
def test_packed_qkv_attention_matches_three_slices(heads, d, rotary, causal, docs):
    print(f"case attention_qkv heads={heads} d={d} rotary={rotary}", flush=True)
    tokens = 150
    g = torch.Generator().manual_seed(d)
    qkv = torch.randn(tokens, heads, 3 * d, generator=g).bfloat16().to(DEV)
    do = torch.randn(tokens, heads, d, generator=g).bfloat16().to(DEV)
    cu = torch.tensor([0, *docs, tokens], dtype=torch.int32, device=DEV)
    rot = None
    if rotary:
        ang = torch.outer(torch.arange(tokens).float(), 1.0 / 10000 ** (torch.arange(0, d, 2).float() / d))
        ang = torch.cat((ang, ang), -1)
        pos = torch.arange(tokens, device=DEV)
        rot = (ang.cos().bfloat16().to(DEV), ang.sin().bfloat16().to(DEV), pos, pos)
    a = qkv.clone().requires_grad_()
    o = ops.attention(a[..., :d], a[..., d:2 * d], a[..., 2 * d:], cu, None, causal, rotary=rot)
    o.backward(do)
    b = qkv.clone().requires_grad_()
    o2 = ops.attention_qkv(b, cu, None, causal, rotary=rot)
    o2.backward(do)
    assert torch.equal(o, o2) and torch.equal(a.grad, b.grad)


@pytest.mark.parametrize("rows,cols,stride", [(1, 8, 8), (63, 72, 80), (512, 64, 64), (513, 136, 136), (4084, 1024, 3072)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_column_sum(rows, cols, stride, dtype):
    """Rows fewer than the row groups of a workgroup, one whole prefetch round, and remainders of both axes; the bound is one
    rounding of the result plus rows fp32 additions."""
    x = torch.randn(rows, stride, generator=torch.Generator().manual_seed(rows)).to(dtype).to(DEV)
    out = torch.empty(cols, dtype=dtype, device=DEV)
    _lib.check(_lib.load().mi_column_sum(x.data_ptr(), stride, rows, cols, out.data_ptr(), _lib.dtype_code(dtype), _lib.stream_ptr()), "mi_column_sum")
    xd = x[:, :cols].double()
    u = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -24}[dtype]
    bound = u * xd.sum(0).abs() + (rows + 1) * 2.0 ** -24 * xd.abs().sum(0) + 2.0 ** -25
    assert bool(((out.double() - xd.sum(0)).abs() <= bound).all())


@pytest.mark.parametrize("rows,cols,stride", [(1, 8, 8), (63, 72, 80), (64, 64, 64), (65, 136, 136), (200, 1000, 1008)])
def test_transpose16(rows, cols, stride):
    """Exact; one row and column past a tile, one short of it, rows of a wider matrix; the padding of the result becomes zero up to
    a whole vector and stays as it is behind."""
    x = torch.randn(rows, stride, generator=torch.Generator().manual_seed(rows)).bfloat16().to(DEV)
    ld = (rows + 63) // 64 * 64
    out = torch.full((cols, ld), 7.0, dtype=torch.bfloat16, device=DEV)
    _lib.check(_lib.load().mi_transpose16(x.data_ptr(), stride, rows, cols, out.data_ptr(), ld, _lib.stream_ptr()), "mi_transpose16")
    whole = (rows + 7) // 8 * 8
    assert torch.equal(out[:, :rows], x[:, :cols].t())
    assert bool((out[:, rows:whole] == 0).all()) and bool((out[:, whole:] == 7).all())


@pytest.mark.parametrize("rows,ins,outs", [(4001, 2048, (8196, 4096)), (3001, 8196, (2056,)), (2500, 4096, (5004,))])
def test_weight_gradients_through_a_transposed_operand(rows, ins, outs):
    """Wide projections that the package's kernels do not take (features that are no whole vectors): the input or (one projection that narrows)
    the output gradient is transposed first; the same products in the same precision, so one rounding of the result and fp32 sums of `rows` terms against float64 on sampled rows."""
    print(f"case transposed weight gradient rows={rows} {ins}->{outs}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(ins)
    x = torch.randn(rows, ins, generator=g, device=DEV).bfloat16().requires_grad_()
    ws = [(torch.randn(o, ins, generator=g, device=DEV) * 0.02).bfloat16().requires_grad_() for o in outs]
    dys = [torch.randn(rows, o, generator=g, device=DEV).bfloat16() for o in outs]
    ys = ops.projections(x, ws, [None] * len(ws))
    names = launched(lambda: torch.autograd.backward(ys, dys))
    assert any("transpose_kernel" in k for k in names) and not any("wide_kernel" in k for k in names), names
    for w, dy in zip(ws, dys):
        pick = torch.tensor([0, 7, w.shape[0] // 2, w.shape[0] - 1], device=DEV)
        a, b = dy[:, pick].double().t().contiguous(), x.detach().double()
        bound = 2.0 ** -8 * (a @ b).abs() + (rows + 1) * 2.0 ** -24 * (a.abs() @ b.abs())
        assert bool(((w.grad[pick].double() - a @ b).abs() <= bound * 1.01).all())


def _native_calls(call):
    """How many layers of a call go through the native layer."""
    with mock.patch.object(ops, "layer", wraps=ops.layer) as native:
        call()
    return native.call_count


# norms, MLPs, projections, types and rotaries of a layer; a step, and the two forms of a pass without gradients
@pytest.mark.parametrize("dtype", ["bfloat16", "float16", "float32"])
@pytest.mark.parametrize("default,options", [
    (True, {}), (False, {}), (True, dict(relative_position_embedding_type="none")), (False, dict(rotary_percentage=0.5)),
    (False, dict(relative_position_embedding_type="rotary_complex")), (True, dict(relative_position_embedding_type="rotary_complex")),
    (False, dict(causal=False)),
])
def test_layer_in_one_call_equals_its_modules(dtype, default, options):
    layer = _layer(dtype, default, **options)
    x = torch.randn(2, 93, 256, generator=torch.Generator().manual_seed(5)).to(layer.self_attention.dtype).to(DEV)
    dy = torch.randn(2, 93, 256, generator=torch.Generator().manual_seed(6)).to(x.dtype).to(DEV)
    io = TransformerLayerIO(activations=x, position_ids=(torch.arange(93, device=DEV) % 60).repeat(2, 1),
                            cumulative_seq_lengths=torch.tensor([0, 60, 93, 153, 186], dtype=torch.int32, device=DEV))

    def run(train, grad):
        layer.train(train)
        x.grad = None
        x.requires_grad_(grad)
        for p in layer.parameters():
            p.grad = None
        with torch.set_grad_enabled(grad):
            out = layer(io).activations
        if not grad:
            return [out]
        out.backward(dy)
        return [out.detach(), x.grad] + [p.grad for p in layer.parameters()]

    for train, grad in ((True, True), (False, True), (True, False), (False, False)):
        assert _native_calls(lambda: run(train, grad)) == 1
        native = run(train, grad)
        seen = []
        handle = layer.self_attention.register_forward_hook(lambda *a: seen.append(1))      # whoever watches a module sees it called
        modules = run(train, grad)
        handle.remove()
        assert seen == [1]
        for i, (a, b) in enumerate(zip(native, modules)):
            assert torch.equal(a, b), (train, grad, i)


@pytest.mark.parametrize("b,s,max_ctx,nkv,d", [(1, 1, 1, 1, 64), (3, 67, 80, 2, 64), (2, 130, 130, 8, 128)])
@pytest.mark.parametrize("interleaved", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_prefill_attention_fills_the_cache(b, s, max_ctx, nkv, d, interleaved, dtype):
    """The rotated rows and the rest of the cache, the lengths and the attention of the launches that it replaces."""
    nq, g = 2 * nkv, torch.Generator().manual_seed(s)
    qkv = torch.randn(b * s, nq + 2 * nkv, d, generator=g).to(dtype).to(DEV)
    q, k, v = qkv[:, :nq], qkv[:, nq:nq + nkv], qkv[:, nq + nkv:]
    pos = torch.arange(s, device=DEV).repeat(b) + 3
    ang = torch.outer(torch.arange(max_ctx + 3).float(), 1.0 / (10000.0 ** (torch.arange(0, d, 2).float() / d))).to(DEV)
    cos, sin = (t if interleaved else torch.cat((t, t), -1).to(dtype) for t in (ang.cos(), ang.sin()))
    cu = torch.arange(0, b * s + 1, s, dtype=torch.int32, device=DEV)
    kc, vc = (torch.full((b, nkv, max_ctx, d), 7.0, dtype=dtype, device=DEV).transpose(1, 2) for _ in range(2))
    ctx = torch.zeros(b, dtype=torch.int32, device=DEV)
    o = _lib.host().prefill_attention(q, k, v, cu, pos, cos, sin, interleaved, d ** -0.5, b, kc, vc, ctx)
    rotate = ops.rotary_embedding_complex if interleaved else ops.rotary_embedding
    k_rot = rotate(k, cos, sin, pos)
    got = kc[:, :s].reshape(b * s, nkv, d)
    if dtype == torch.float16:
        # the rotary kernel rounds some of its float32 sums twice (float32, float16) and some once (mixed-precision fma): one ulp apart
        assert torch.allclose(got.float(), k_rot.float(), rtol=2.0 ** -10, atol=2.0 ** -24)
        k_rot = got.contiguous()
    assert torch.equal(got, k_rot) and torch.equal(vc[:, :s].reshape(b * s, nkv, d), v)
    assert bool((kc[:, s:] == 7).all()) and bool((vc[:, s:] == 7).all()) and ctx.tolist() == [s] * b
    assert torch.equal(o, ops.attention_forward(q, k_rot, v, cu, None, True, d ** -0.5, rotary=(cos, sin, pos, None))[0])
    with pytest.raises(RuntimeError, match="fit the rows"):
        _lib.host().prefill_attention(q, k, v, cu, pos, cos, sin, interleaved, d ** -0.5, b, kc, vc, ctx[:0])


@pytest.mark.parametrize("d,b,s", [(64, 1, 1), (64, 3, 67), (128, 2, 130), (128, 1, 509)])
@pytest.mark.parametrize("kind", ["rotary", "rotary_complex"])
@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
def test_prefill_in_one_call_equals_its_modules(dtype, kind, d, b, s):
    """Output, cache and lengths of a prefill, a prefill into a cache that is there and longer, and the step that follows, in every bit: float16
    too, whose rotary sums the kernels round once or twice."""
    layer = _layer(dtype, False, hidden=4 * d, relative_position_embedding_type=kind).eval()
    g = torch.Generator().manual_seed(s)
    normal = lambda *shape: torch.randn(*shape, generator=g).to(layer.self_attention.dtype).to(DEV)
    x, x2, x3, step = normal(b, s, 4 * d), normal(b, s, 4 * d), normal(b, max(s - 1, 1), 4 * d), normal(b, 1, 4 * d)

    def io(x, position, reset):
        io = _io(x)
        io.position_ids, io.inference_settings = io.position_ids + position, InferenceSettings(use_cache=True, reset_cache=reset)
        return io

    def run(watched):
        layer.self_attention.cache.clear()
        seen, out = [], []
        for x_ in (x, x2, x3):
            handle = layer.self_attention.register_forward_hook(lambda *a: seen.append(1)) if watched else None
            with torch.no_grad():
                out.append(layer(io(x_, 0, True)).activations)
            if handle is not None:
                handle.remove()
            cache = layer.self_attention.cache[0]
            assert cache.length == x_.shape[1]
            out += [cache.k.clone(), cache.v.clone(), cache.ctx_len.clone()]
        with torch.no_grad():
            out.append(layer(io(step, x3.shape[1], False)).activations)
        return out + [cache.k, cache.v], seen

    assert _native_calls(lambda: run(False)) == 3 and _native_calls(lambda: run(True)) == 0
    native, _ = run(False)
    modules, seen = run(True)
    assert len(seen) == 3
    for i, (a, c) in enumerate(zip(native, modules)):
        assert torch.equal(a, c), i


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("interleaved", [False, True])
@pytest.mark.parametrize("d", [64, 128])
def test_cached_keys_are_those_of_the_rotary_kernel(d, interleaved, dtype):
    """The rounding of float16 sums included: 131072 rotated features."""
    nkv, s, g = 8, 16384 // d, torch.Generator().manual_seed(d)
    q, k, v = (torch.randn(s, nkv, d, generator=g).to(dtype).to(DEV) for _ in range(3))
    pos = torch.arange(s, device=DEV)
    ang = torch.outer(torch.arange(s).float(), 1.0 / (10000.0 ** (torch.arange(0, d, 2).float() / d))).to(DEV)
    cos, sin = (t if interleaved else torch.cat((t, t), -1).to(dtype) for t in (ang.cos(), ang.sin()))
    cu = torch.tensor([0, s], dtype=torch.int32, device=DEV)
    kc, vc = (torch.zeros(1, s, nkv, d, dtype=dtype, device=DEV) for _ in range(2))
    _lib.host().prefill_attention(q, k, v, cu, pos, cos, sin, interleaved, d ** -0.5, 1, kc, vc, torch.zeros(1, dtype=torch.int32, device=DEV))
    assert torch.equal(kc[0], (ops.rotary_embedding_complex if interleaved else ops.rotary_embedding)(k, cos, sin, pos)) and torch.equal(vc[0], v)


def _watched(layer, io):
    """The layer's activations from its modules, which a hook keeps from being passed by."""
    handle = layer.self_attention.register_forward_hook(lambda *a: None)
    try:
        return layer(io).activations
    finally:
        handle.remove()


@pytest.mark.parametrize("default", [False, True])
@pytest.mark.parametrize("tables", ["float32", "other16", "narrow"])
def test_rotary_tables_that_the_kernels_cannot_read(tables, default):
    """Tables of another type or of fewer features than a head, as casts and replaced modules leave them: refused where the attention core rotates, as
    the modules refuse them; a prefill with float32 tables is computed, as the modules compute it."""
    layer = _layer("bfloat16", default)
    att, x = layer.self_attention, torch.randn(2, 40, 256, generator=torch.Generator().manual_seed(1)).bfloat16().to(DEV)
    if tables == "narrow":
        att.rotary_embedding = RotaryEmbedding(RotaryConfig(dimensions=32, max_seq_length=512, base=10000), torch.device(DEV), torch.bfloat16)
    else:
        att.rotary_embedding.to(torch.float32 if tables == "float32" else torch.float16)
    for train in (True, False):
        layer.train(train)
        with torch.set_grad_enabled(train), pytest.raises(AssertionError, match="fused rotary"):
            layer(_io(x))
    if default:
        return
    io = _io(x)
    io.inference_settings = InferenceSettings(use_cache=True, reset_cache=True)
    with torch.no_grad():
        if tables == "other16":
            with pytest.raises(RuntimeError, match="table dtype"):
                layer(io)
            return
        y, cache = layer(io).activations, att.cache[0]
        y, k, n = y.clone(), cache.k.clone(), cache.ctx_len.tolist()
        assert torch.equal(y, _watched(layer, io)) and torch.equal(k, cache.k) and n == [40, 40] and y.isfinite().all()


@pytest.mark.parametrize("cos_dtype,width,interleaved", [(torch.float32, 64, False), (torch.float16, 64, False), (torch.bfloat16, 32, False),
                                                         (torch.bfloat16, 32, True), (torch.float32, 64, True)])
def test_prefill_attention_refuses_tables_that_do_not_fit(cos_dtype, width, interleaved):
    q, k, v = (torch.zeros(8, 2, 64, dtype=torch.bfloat16, device=DEV) for _ in range(3))
    cos, sin = (torch.zeros(16, width, dtype=cos_dtype, device=DEV) for _ in range(2))
    kc, vc = (torch.full((1, 8, 2, 64), 3.0, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    cu, ctx = torch.tensor([0, 8], dtype=torch.int32, device=DEV), torch.zeros(1, dtype=torch.int32, device=DEV)
    with pytest.raises(RuntimeError, match="tables have to fit"):
        _lib.host().prefill_attention(q, k, v, cu, torch.arange(8, device=DEV), cos, sin, interleaved, 0.125, 1, kc, vc, ctx)
    assert bool((kc == 3).all()) and int(ctx) == 0


@pytest.mark.parametrize("default", [False, True])
@pytest.mark.parametrize("owner", ["attention", "core"])
def test_mask_of_a_layer_is_its_cores(owner, default):
    """`causal` of the attention module decides whether a cache may be filled, that of its core what is masked."""
    layer, x = _layer("bfloat16", default).eval(), torch.randn(2, 70, 256, generator=torch.Generator().manual_seed(2)).bfloat16().to(DEV)
    with torch.no_grad():
        y = layer(_io(x)).activations
        target = layer.self_attention if owner == "attention" else layer.self_attention.scaled_dot_product_attention
        target.causal = False
        changed = layer(_io(x)).activations
        assert torch.equal(changed, _watched(layer, _io(x))) and torch.equal(changed, y) == (owner == "attention")
        if default:
            return
        io = _io(x)
        io.inference_settings = InferenceSettings(use_cache=True, reset_cache=True)
        if owner == "attention":
            with pytest.raises(ValueError, match="causal"):
                layer(io)
        else:
            assert torch.equal(layer(io).activations, _watched(layer, io))


@pytest.mark.parametrize("on_class", [False, True])
@pytest.mark.parametrize("default,where,name", [
    (False, "self_attention", "_project"), (True, "self_attention", "_fill_cache"), (False, "self_attention", "_fill_cache"),
    (False, "self_attention.rotary_embedding", "rotate_tokens"), (True, "self_attention.scaled_dot_product_attention", "forward_qkv"),
    (False, "self_attention.scaled_dot_product_attention", "forward_tokens"), (False, "input_layernorm", "with_residual"),
    (True, "post_attention_layernorm", "with_residual"), (False, "mlp", "forward"), (True, "mlp", "forward"), (True, "self_attention.dense", "forward"),
])
def test_functions_that_somebody_set_anew_are_called(where, name, default, on_class, monkeypatch):
    """A function of the layer's modules that is replaced, on the module or on its class, is called wherever the modules call it: in a pass without a
    cache or in a prefill (which only the layer without one QKV projection can take here)."""
    layer = _layer("bfloat16", default).eval()
    x = torch.randn(2, 30, 256, generator=torch.Generator().manual_seed(3)).bfloat16().to(DEV)
    module = layer.get_submodule(where)
    calls, own = [], getattr(type(module), name)
    io = _io(x)
    with torch.no_grad():
        y = layer(io).activations
        if name in ("_fill_cache", "rotate_tokens"):       # called in a prefill alone
            io.inference_settings = InferenceSettings(use_cache=True, reset_cache=True)
            y = layer(io).activations

        def replaced(self, *args, **kwargs):
            calls.append(name)
            return own(self, *args, **kwargs)

        if on_class:
            monkeypatch.setattr(type(module), name, replaced)
        else:
            monkeypatch.setattr(module, name, lambda *args, **kwargs: replaced(module, *args, **kwargs))
        assert torch.equal(layer(io).activations, y) and calls


@pytest.mark.parametrize("case", ["float16", "strides"])
def test_prefill_into_a_cache_of_another_kind(case):
    """A cache that is there and long enough is filled, whatever its type (a model that was cast in between) and strides, as the modules fill it."""
    layer = _layer("bfloat16", False).eval()
    att, x = layer.self_attention, torch.randn(2, 30, 256, generator=torch.Generator().manual_seed(4)).bfloat16().to(DEV)
    io = _io(x)
    io.inference_settings = InferenceSettings(use_cache=True, reset_cache=True)
    results = []
    for run in (lambda: layer(io).activations, lambda: _watched(layer, io)):
        cache = att.cache[0] = KVCache(2, 512, 2, 64, torch.float16 if case == "float16" else torch.bfloat16, torch.device(DEV))
        if case == "strides":
            cache.v = cache.v.contiguous()
        with torch.no_grad():
            results.append([run(), cache.k, cache.v, cache.ctx_len])
        assert att.cache[0] is cache and cache.length == 30
    assert all(torch.equal(a, b) for a, b in zip(*results)) and results[0][1].any()


# on the line up to which a layer is one autograd node, above it, and with rows that end inside a tile
@pytest.mark.parametrize("default,dtype,options,b,s", [
    (True, "float32", {}, 2, 93), (True, "bfloat16", dict(relative_position_embedding_type="none"), 1, 1), (False, "bfloat16", {}, 8, 256),
    (False, "bfloat16", {}, 9, 228), (False, "float16", dict(rotary_percentage=0.5), 3, 67),
])
def test_gradients_of_a_layer_that_is_one_node(default, dtype, options, b, s):
    """Any choice of gradients, a kept graph and a graph of the gradients: to the bit what the nodes of the modules give."""
    layer = _layer(dtype, default, **options)
    x = torch.randn(b, s, 256, generator=torch.Generator().manual_seed(5)).to(getattr(torch, dtype)).to(DEV).requires_grad_()
    io, parameters = _io(x), dict(layer.named_parameters())
    first = "self_attention.query_key_value.weight" if default else "self_attention.key.weight"

    def gradients(forward, inputs, **how):
        y = forward()
        return [torch.autograd.grad(y, inputs, torch.cos(y.detach()), **how) for _ in range(2 if how else 1)]

    def native():
        y = layer(io).activations
        assert y.grad_fn.name().endswith("::Layer>") == (b * s * 256 <= 2 ** 19)
        return y
    for names in (["x"], ["input_layernorm.weight"], [first], ["self_attention.dense.weight", "x"], ["post_attention_layernorm.weight"],
                  ["mlp.dense_in.weight"], ["mlp.dense_out.weight"], ["x", *parameters]):
        inputs = [x if n == "x" else parameters[n] for n in names]
        for how in ({}, dict(retain_graph=True), dict(create_graph=True)):
            for got, want in zip(gradients(native, inputs, **how), gradients(lambda: _watched(layer, io), inputs, **how)):
                assert all(torch.equal(p, q) for p, q in zip(got, want)), (names, how)
    for n, p in parameters.items():                        # frozen: everything but one
        p.requires_grad_(n == first)
    io.activations = x.detach()
    assert all(torch.equal(p, q) for p, q in zip(gradients(native, [parameters[first]])[0], gradients(lambda: _watched(layer, io), [parameters[first]])[0]))


@pytest.mark.parametrize("case", ["retained", "hooks", "shared", "twice", "frozen since"])
def test_graph_of_gradients_of_a_layer_that_is_one_node(case):
    """Gradients with a graph of their own meet hooks, retained gradients and parameters in several places as often as those of the modules' nodes, and
    that graph is theirs: to the bit, and where it is differentiated again up to the order of float32 sums of a few terms."""
    layer = _layer("float32", True)
    if case == "shared":
        layer.post_attention_layernorm.weight = layer.input_layernorm.weight
        layer.mlp.dense_out.bias = layer.self_attention.dense.bias
    leaf = torch.randn(2, 33, 256, generator=torch.Generator().manual_seed(8)).to(DEV).requires_grad_()
    parameters = dict(layer.named_parameters())
    dy = torch.randn(2, 33, 256, generator=torch.Generator().manual_seed(9)).to(DEV).requires_grad_()
    where = ["self_attention.query_key_value.weight", "mlp.dense_in.bias", "post_attention_layernorm.weight"]

    def gradients(forward):
        layer.zero_grad(set_to_none=True)
        leaf.grad = None
        x = leaf * layer.input_layernorm.weight if case in ("retained", "twice") else leaf
        handles = [p.register_hook(lambda g: 2 * g) for p in (x, *(parameters[n] for n in where))] if case == "hooks" else []
        if case == "retained":
            x.retain_grad()
        y = forward(x)
        if case == "twice":
            y = forward(y)
        if case == "frozen since":                         # its gradient is wanted all the same: what the graph was made with counts
            parameters[where[1]].requires_grad_(False)
        if case in ("retained", "frozen since"):
            torch.autograd.backward(y, dy, create_graph=True)
            got = [x.grad, *(p.grad for p in (leaf, *parameters.values()) if p.requires_grad)]
        else:
            got = list(torch.autograd.grad(y, [leaf, *parameters.values()], dy, create_graph=True))
        parameters[where[1]].requires_grad_(True)
        connected = [g for g in got if g.requires_grad]
        again = torch.autograd.grad(sum((g * torch.cos(g.detach())).sum() for g in connected), [leaf, dy, *parameters.values()], allow_unused=True)
        for handle in handles:
            handle.remove()
        for p in (x, leaf, *parameters.values()):
            p.grad = None
        return [g.detach() for g in got], [g.requires_grad for g in got], again

    def native(x):
        y = layer(_io(x)).activations
        assert y.grad_fn.name().endswith("::Layer>")
        return y
    (got, graph, again), (want, want_graph, want_again) = gradients(native), gradients(lambda x: _watched(layer, _io(x)))
    assert all(torch.equal(p, q) for p, q in zip(got, want)) and graph == want_graph and any(graph)
    assert [g is None for g in again] == [g is None for g in want_again]
    for p, q in zip(again, want_again):
        if q is not None:
            assert (p - q).abs().max() <= 1e-5 * q.abs().max()


@pytest.mark.parametrize("name", ["mlp.dense_out.bias", "input_layernorm.bias", "self_attention.dense.bias", "self_attention.query_key_value.weight", "lengths"])
def test_graph_of_gradients_of_a_layer_changed_since(name):
    """What the forward pass read and nothing saved, changed in place before the backward pass: a graph of the gradients, which is made from it, is refused,
    and gradients without one are those of the pass that was."""
    layer = _layer("float32", True)
    for n, p in layer.named_parameters():                  # nothing in front of the first projection takes a gradient: its weight is not saved
        p.requires_grad_(not n.startswith("input_layernorm"))
    io = _io(torch.randn(2, 33, 256, generator=torch.Generator().manual_seed(8)).to(DEV))
    wanted = [layer.mlp.dense_in.weight, layer.self_attention.query_key_value.bias]
    y = layer(io).activations
    assert y.grad_fn.name().endswith("::Layer>")
    before = torch.autograd.grad(y.sum(), wanted, retain_graph=True)
    torch.autograd.grad(y.sum(), wanted, create_graph=True)
    with torch.no_grad():
        if name == "lengths":
            io.cumulative_seq_lengths[1] += 1
        else:
            layer.get_parameter(name).add_(1.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(y.sum(), wanted, create_graph=True)
    if name != "lengths":
        assert all(torch.equal(p, q) for p, q in zip(before, torch.autograd.grad(y.sum(), wanted)))


@pytest.mark.parametrize("to", [torch.bfloat16, torch.float16])
def test_graph_of_gradients_of_a_layer_under_autocast(to):
    """Autocast around the backward pass alone: what the modules' nodes give under it, to the bit, and no forward pass in another type."""
    layer = _layer("float32", True)
    x = torch.randn(2, 33, 256, generator=torch.Generator().manual_seed(8)).to(DEV).requires_grad_()
    inputs = [x, *layer.parameters()]

    def gradients(y):
        with torch.autocast("cuda", dtype=to):
            return torch.autograd.grad(y, inputs, torch.cos(y.detach()), create_graph=True)
    y = layer(_io(x)).activations
    assert y.grad_fn.name().endswith("::Layer>")
    assert all(torch.equal(p, q) for p, q in zip(gradients(y), gradients(_watched(layer, _io(x)))))


@pytest.mark.parametrize("default", [False, True])
@pytest.mark.parametrize("trained", ["everything", "mlp.dense_out.weight", "mlp.dense_in.weight"])
def test_memory_of_a_layer_that_is_one_node(default, trained):
    """What is kept for the backward pass, and the most that is held during it, beside the modules' nodes: no more than x, which a graph of the gradients would
    need, and the gradient that goes past the MLP."""
    layer = _layer("bfloat16", default)
    if trained != "everything":
        layer.requires_grad_(False).get_parameter(trained).requires_grad_()
    x = torch.randn(8, 256, 256, generator=torch.Generator().manual_seed(8)).to(torch.bfloat16).to(DEV)
    io, dy = _io(x), torch.randn(8, 256, 256, generator=torch.Generator().manual_seed(9)).to(torch.bfloat16).to(DEV)

    def held(forward):
        layer.zero_grad(set_to_none=True)
        torch.cuda.synchronize()
        start = torch.cuda.memory_allocated()
        y = forward()
        kept = torch.cuda.memory_allocated() - start
        torch.cuda.reset_peak_memory_stats()
        torch.autograd.backward(y, dy)
        return kept, torch.cuda.max_memory_allocated() - start

    def native():
        y = layer(io).activations
        assert y.grad_fn.name().endswith("::Layer>")
        return y
    for forward in (native, lambda: _watched(layer, io)):  # workspaces
        held(forward)
    (kept, most), (want, want_most) = held(native), held(lambda: _watched(layer, io))
    size = x.numel() * x.element_size()
    assert kept <= want + size and most <= want_most + 2 * size, (kept / size, want / size, most / size, want_most / size)


def test_parts_of_a_layer_that_is_one_node_look_at_their_own():
    """A weight changed in place since the forward pass is refused by gradients that take it, and by no others; a graph is used up once."""
    layer = _layer("bfloat16", False)
    x = torch.randn(2, 33, 256, generator=torch.Generator().manual_seed(8)).to(torch.bfloat16).to(DEV).requires_grad_()
    y = layer(_io(x)).activations
    assert y.grad_fn.name().endswith("::Layer>")
    wanted = [layer.mlp.dense_out.weight, layer.mlp.dense_in.weight]
    before = torch.autograd.grad(y.sum(), wanted, retain_graph=True)
    with torch.no_grad():
        layer.self_attention.query.weight.mul_(2.0)
    assert all(torch.equal(p, q) for p, q in zip(before, torch.autograd.grad(y.sum(), wanted, retain_graph=True)))
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(y.sum(), x, retain_graph=True)
    assert all(torch.equal(p, q) for p, q in zip(before, torch.autograd.grad(y.sum(), wanted)))
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(y.sum(), wanted)


@pytest.mark.parametrize("case", ["no module", "instance's module", "instance's weight", "class's module"])
def test_layer_whose_parts_are_not_where_modules_keep_them(case):
    """A layer reads its parts as attributes do: an identity that is no module, entries of the instance and properties of a derived class count."""
    layer, other = _layer("float32", True), _layer("float32", True)
    with torch.no_grad():
        other.mlp.dense_in.weight.mul_(2.0)
    io = _io(torch.randn(2, 33, 256, generator=torch.Generator().manual_seed(8)).to(DEV))
    plain = layer(io).activations
    if case == "no module":
        del layer.dropout_attention, layer.dropout_mlp
        layer.dropout_attention = layer.dropout_mlp = lambda x: x
    elif case == "instance's module":
        layer.__dict__["mlp"] = other.mlp
    elif case == "instance's weight":
        layer.mlp.dense_in.__dict__["weight"] = other.mlp.dense_in.weight
    else:
        layer.__class__ = type("Derived", (TransformerLayer,), dict(mlp=property(lambda self: other.mlp)))
    got, want = layer(io).activations, _watched(layer, io)
    assert torch.equal(got, want) and torch.equal(got, plain) == (case == "no module")


def test_training_of_a_small_layer_on_an_inference_tensor():
    """x from inference mode, a frozen norm in front of what is trained: nothing that may not be kept has to be."""
    layer = _layer("bfloat16", True)
    layer.input_layernorm.requires_grad_(False)
    with torch.inference_mode():
        x = torch.randn(2, 33, 256, device=DEV).to(torch.bfloat16)
    io, inputs = _io(x), [p for p in layer.parameters() if p.requires_grad]
    got, want = (torch.autograd.grad(y.float().sum(), inputs) for y in (layer(io).activations, _watched(layer, io)))
    assert all(torch.equal(p, q) for p, q in zip(got, want))
