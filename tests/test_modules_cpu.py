"""CPU-only checks of the host-side mirror of the reference interface: config surface, index
construction (bit-exact against the oracle and the reference's known answers), module / parameter
names (checkpoint contract) and the documented error behaviour.  No kernel is launched."""

import os

import pytest
import torch

import oracle
from scaling_amd import config as C
from scaling_amd import data as D
from scaling_amd.layer import LayerNormWrapper, TransformerLayer
from scaling_amd.nn import ParallelSelfAttention, ParallelSwiGLUMLP, RMSNorm, RotaryEmbedding
from tests.golden import known_answers as KA

CPU = torch.device("cpu")


def _arch(**kw):
    d = dict(vocab_size=64, hidden_size=256, num_layers=2, num_attention_heads=4, attention_num_kv_heads=2,
             attention_qkv_in_one=False, norm_type="rms", mlp_type="swiglu", mlp_factor=2.6875, attention_bias=False,
             mlp_bias=False, precision="bfloat16", sequence_length=128, masked_softmax={"kernel": "hip"}, weight_tying=False)
    d.update(kw)
    return C.TransformerArchitectureConfig.from_dict(d)


# ---- config surface ------------------------------------------------------------------------------------
def test_masked_softmax_config_defaults_and_new_member():
    c = C.MaskedSoftmaxConfig()
    assert c.kernel == C.MaskedSoftmaxKernel.TORCH and c.softmax_in_fp32 is False and c.scale == 1.0
    assert c.deterministic_flash_attn_bwd is False
    assert [k.value for k in C.MaskedSoftmaxKernel] == ["torch", "flash_attention", "hip"]
    assert C.MaskedSoftmaxConfig(kernel="hip").as_dict()["kernel"] == "hip"
    with pytest.raises(Exception):
        C.MaskedSoftmaxConfig(kernel="cuda")
    with pytest.raises(Exception):
        C.MaskedSoftmaxConfig(unknown_key=1)           # extra = forbid
    with pytest.raises(Exception):
        c.scale = 2.0                                  # frozen


def test_architecture_config_round_trip_and_defaults():
    a = C.TransformerArchitectureConfig()
    assert a.norm_type == C.NormType.LAYERNORM and a.mlp_type == C.MLPType.DEFAULT and a.mlp_factor == 4.0
    assert a.attention_qkv_in_one and a.attention_num_kv_heads is None and a.rotary_embedding_base == 10000
    assert a.sequence_length == 2048 and a.causal and a.precision == C.Precision.FLOAT32
    assert a.relative_position_embedding_type == C.RelativePositionEmbeddingType.ROTARY
    assert C.RotaryConfig().max_seq_length == 2048 and C.LayerNormConfig().layernorm_epsilon == 1e-5
    b = _arch()
    assert C.TransformerArchitectureConfig.from_dict(b.as_dict()) == b
    assert C.TransformerArchitectureConfig.from_str(b.as_str()) == b
    assert b.rotary_config() == C.RotaryConfig(dimensions=64, max_seq_length=128, base=10000)
    assert b.precision.dtype == torch.bfloat16


def test_example_architecture_block_validates(tmp_path):
    # the transformer_architecture block of the reference's example config (values restated as data)
    block = {"weight_tying": False, "vocab_size": 128000, "hidden_size": 256, "num_layers": 4, "num_attention_heads": 2,
             "rotary_embedding_base": 10000, "sequence_length": 64, "norm_type": "rms",
             "relative_position_embedding_type": "rotary_complex", "attention_bias": False, "mlp_type": "swiglu",
             "mlp_factor": 2.5, "mlp_bias": False, "masked_softmax": {"kernel": "flash_attention", "softmax_in_fp32": True,
                                                                      "deterministic_flash_attn_bwd": False, "scale": 1.0},
             "layernorm": {"optimization_type": "torch", "layernorm_epsilon": 1e-5}, "precision": "bfloat16",
             "dropout_embedding": 0.1, "dropout_attention_probs": 0.1, "dropout_after_attention": 0.1,
             "dropout_after_mlp": 0.1, "bitfit_bias_config": None, "softprompt_config": None, "adapter_config": None,
             "lora_config": None, "image_encoder": False, "dropout_image_encoder": 0.0}
    import yaml
    f = tmp_path / "config.yml"
    f.write_text(yaml.safe_dump({"transformer_architecture": block}))
    a = C.architecture_from_config_file(f, kernel=None)
    assert a.masked_softmax.kernel == C.MaskedSoftmaxKernel.FLASH_ATTENTION
    assert C.architecture_from_config_file(f, kernel="hip").masked_softmax.kernel == C.MaskedSoftmaxKernel.HIP


# ---- index construction -----------------------------------------------------------------------------------
def test_data_utils_known_answers():
    ids = torch.tensor(KA.TOKEN_IDS)
    assert D.get_cumulative_seq_lengths(ids).tolist() == KA.CU_WITH_RESET
    assert D.get_cumulative_seq_lengths(ids).dtype == torch.int32
    assert D.get_cumulative_seq_lengths(ids, reset_attention_mask=False).tolist() == KA.CU_WITHOUT_RESET
    assert D.get_position_ids(ids).tolist() == KA.POSITION_IDS_WITH_RESET
    assert D.get_position_ids(ids, reset_position_ids=False).tolist() == KA.POSITION_IDS_WITHOUT_RESET
    padded = D.add_cumulative_seq_lengths_padding(torch.tensor(KA.PADDING_INPUT), KA.PADDING_PAD_TO)
    assert padded.tolist() == KA.PADDING_EXPECTED
    assert D.remove_cumulative_seq_lengths_padding(padded).tolist() == KA.PADDING_INPUT


def test_data_utils_bit_exact_against_oracle():
    g = torch.Generator().manual_seed(0)
    for _ in range(20):
        b, s = int(torch.randint(1, 5, (1,), generator=g)), int(torch.randint(1, 40, (1,), generator=g))
        ids = torch.randint(0, 4, (b, s), generator=g)
        for reset in (True, False):
            a, o = D.get_cumulative_seq_lengths(ids, reset), oracle.get_cumulative_seq_lengths(ids, reset)
            assert a.dtype == o.dtype and torch.equal(a, o)
            a, o = D.get_position_ids(ids, reset), oracle.get_position_ids(ids, reset)
            assert a.dtype == o.dtype and torch.equal(a, o)


def test_get_max_seq_length_matches_oracle():
    cu = torch.tensor(KA.CU_WITH_RESET, dtype=torch.int32)
    assert D.get_max_seq_length(cu) == oracle.get_max_seq_length(cu) == max(b - a for a, b in zip(KA.CU_WITH_RESET[:-1], KA.CU_WITH_RESET[1:]))


def test_scaled_dot_product_attention_and_masked_softmax_mirror_the_reference_classes():
    """attention.py:280-304 and masked_softmax.py:37-52: attribute names, the module tree under
    `scaled_dot_product_attention`, NotImplementedError for a kernel this package does not provide, and the
    assert of a fused kernel's softmax module when it is called directly."""
    from scaling_amd.nn import MaskedSoftmax, ScaledDotProductAttention
    hip = C.MaskedSoftmaxConfig(kernel="hip", scale=2.0, deterministic_flash_attn_bwd=True)
    sdpa = ScaledDotProductAttention(head_dim=64, dropout_p=0.1, masked_softmax_config=hip, causal=True)
    assert sdpa.head_dim == 64 and sdpa.dropout_p == 0.1 and sdpa.causal and not sdpa.use_matmul
    assert sdpa.query_key_scaling_factor == 1 / 8 and sdpa.softmax_scale == 0.25 and sdpa.masked_softmax_config is hip
    assert isinstance(sdpa.softmax_fn, MaskedSoftmax) and isinstance(sdpa.dropout_fn, torch.nn.Dropout)
    assert sdpa.softmax_fn.kernel is None and sdpa.softmax_fn.config is hip
    with pytest.raises(AssertionError):
        sdpa.softmax_fn(torch.zeros(1, 1, 2, 2), torch.zeros(1, 1, 2, 2, dtype=torch.bool))
    for kernel in ("torch", "flash_attention"):
        with pytest.raises(NotImplementedError, match="not implemented"):
            MaskedSoftmax(C.MaskedSoftmaxConfig(kernel=kernel))
    att = ParallelSelfAttention(256, 4, hip, dtype=torch.bfloat16, device=CPU, rotary_config=C.RotaryConfig(dimensions=64))
    names = dict(att.named_modules())
    assert "scaled_dot_product_attention" in names and "scaled_dot_product_attention.softmax_fn" in names
    assert att.softmax_scale == sdpa.softmax_scale
    assert not any(k.startswith("scaled_dot_product_attention") for k in att.state_dict())   # no parameters: checkpoints unchanged


class _Seen(torch.Tensor):
    """An operand that takes over torch functions."""
    functions = []

    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        cls.functions.append(func)
        return super().__torch_function__(func, types, args, kwargs or {})


def test_projections_are_seen_by_operands_and_modes_that_take_over_torch_functions():
    from torch.overrides import TorchFunctionMode

    from scaling_amd import ops
    functions = []

    class Mode(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            functions.append(func)
            return func(*args, **(kwargs or {}))
    x, w, b = torch.randn(3, 8), torch.randn(4, 8), torch.randn(4)
    want = torch.nn.functional.linear(x, w, b)
    for call, n in ((lambda v: ops.linear(x, v, b), 1), (lambda v: ops.linear(x, v, b, torch.zeros(3, 4)), 1),
                    (lambda v: ops.projections(x, [v, w], [b, b])[0], 2)):
        _Seen.functions.clear()
        y = call(w.as_subclass(_Seen))
        assert isinstance(y, _Seen) and torch.nn.functional.linear in _Seen.functions and torch.equal(y.as_subclass(torch.Tensor), want)
        functions.clear()
        with Mode():
            y = call(w)
        assert functions.count(torch.nn.functional.linear) == n and torch.equal(y, want)
        assert torch.equal(call(w), want)


# ---- module / checkpoint contract ---------------------------------------------------------------------------
def test_a_default_device_changes_no_projection(monkeypatch):
    from scaling_amd import _lib, ops

    class Host:
        @staticmethod
        def linear(*_):
            return "native"
        projections = linear
    monkeypatch.setattr(_lib, "host", lambda: Host)
    x, w = torch.randn(3, 8), torch.nn.Parameter(torch.randn(4, 8))
    for call in (lambda v: ops.linear(x, v), lambda v: ops.projections(x, [v, w], [None, None])):
        assert call(w) == "native"
        with torch.device("cpu"):
            assert call(w) == "native" and call(w.detach().as_subclass(_Seen)) != "native"


def test_row_products_leave_operands_and_modes_that_take_over_torch_functions_alone(monkeypatch):
    from torch.overrides import TorchFunctionMode

    from scaling_amd import _lib, ops

    class Host:
        @staticmethod
        def norm_linear_rows(*_):
            return "native"
        decode_layer = norm_linear_rows
    monkeypatch.setattr(_lib, "host", lambda: Host)
    x, norm, w, ids = torch.randn(3, 8), torch.ones(8), torch.randn(4, 8), torch.zeros(3, dtype=torch.int64)

    def head(i=None):
        x_, norm_, w_ = (t.as_subclass(_Seen) if j == i else t for j, t in enumerate((x, norm, w)))
        return ops.norm_linear_rows(x_, norm_, 1e-5, w_)

    def step(i=None):
        t = [norm, w, w, w, w, norm, w, w, w]
        if i is not None:
            t[i] = t[i].as_subclass(_Seen)
        arguments = ops.decode_layer_arguments(t[0], 1e-5, t[1:4], t[4], t[5], 1e-5, *t[6:], 8, *[None] * 3, (w, w), 1.0, None, torch.float32)
        return arguments and ops.decode_layer(x, ids, arguments)
    for call, n in ((head, 3), (step, 9)):
        assert call() == "native" and all(call(i) is None for i in range(n))
        with TorchFunctionMode():
            assert call() is None
        with torch.device("cpu"):
            assert call() == "native"


def test_layer_parameter_names_match_reference_checkpoint(golden_dir):
    legacy = torch.load(os.path.join(golden_dir, "legacy_layer_state.pt"), weights_only=True)
    layer = TransformerLayer(_arch(attention_qkv_in_one=True, attention_num_kv_heads=None), layer_index=0, device=CPU)
    assert set(layer.state_dict().keys()) == set(legacy.keys())      # rotary tables are not persistent
    names = [n for n, _ in layer.named_children()]
    assert names == ["input_layernorm", "self_attention", "dropout_attention", "post_attention_layernorm", "mlp", "dropout_mlp"]
    gqa = TransformerLayer(_arch(), layer_index=1, device=CPU).state_dict()
    assert {"self_attention.query.weight", "self_attention.key.weight", "self_attention.value.weight",
            "self_attention.dense.weight", "mlp.dense_in.weight", "mlp.siglu_weight.weight", "mlp.dense_out.weight",
            "input_layernorm.weight", "post_attention_layernorm.weight"} == set(gqa.keys())
    assert gqa["self_attention.key.weight"].shape == (128, 256) and gqa["mlp.dense_in.weight"].shape == (688, 256)
    assert list(LayerNormWrapper(_arch(), layer_index=2, device=CPU).state_dict().keys()) == ["norm.weight"]
    biased = ParallelSelfAttention(256, 4, C.MaskedSoftmaxConfig(kernel="hip"), rotary_config=C.RotaryConfig(dimensions=64),
                                   dtype=torch.bfloat16, device=CPU)
    assert "query_key_value.bias" in biased.state_dict() and "dense.bias" in biased.state_dict()
    assert biased.state_dict()["query_key_value.weight"].shape == (768, 256)


def test_rotary_tables_match_oracle_and_are_not_persistent():
    r = RotaryEmbedding(C.RotaryConfig(dimensions=64, max_seq_length=128, base=500000), CPU, torch.bfloat16)
    t = oracle.rotary_tables(64, 128, 500000, torch.bfloat16)
    cos, sin = r.tables()
    assert r.cos.shape == (128, 1, 1, 64) and torch.equal(cos, t.cos) and torch.equal(sin, t.sin)
    assert len(r.state_dict()) == 0


def test_unsupported_options_raise():
    hip = C.MaskedSoftmaxConfig(kernel="hip")
    with pytest.raises(NotImplementedError, match="hip"):
        ParallelSelfAttention(256, 4, C.MaskedSoftmaxConfig(kernel="torch"), dtype=torch.bfloat16, device=CPU)
    assert ParallelSelfAttention(256, 4, hip, dropout_attention_probs=0.1, dtype=torch.bfloat16, device=CPU,
                                 rotary_config=C.RotaryConfig(dimensions=64)).dropout_attention_probs == 0.1
    # float32 (the reference's default precision) is accepted: exact-fp32 kernels, stand-alone rotary, no dropout
    f32 = ParallelSelfAttention(256, 4, hip, dtype=torch.float32, device=CPU, rotary_config=C.RotaryConfig(dimensions=64))
    assert f32.dtype == torch.float32 and not f32._fusable_rotary and f32.query_key_value.weight.dtype == torch.float32
    with pytest.raises(NotImplementedError, match="dropout"):
        ParallelSelfAttention(256, 4, hip, dropout_attention_probs=0.1, dtype=torch.float32, device=CPU,
                              rotary_config=C.RotaryConfig(dimensions=64))
    with pytest.raises(NotImplementedError, match="float32"):
        ParallelSelfAttention(256, 4, hip, dtype=torch.float64, device=CPU, rotary_config=C.RotaryConfig(dimensions=64))
    cplx = ParallelSelfAttention(256, 4, hip, dtype=torch.bfloat16, device=CPU, rotary_config=C.RotaryConfig(dimensions=64, max_seq_length=16),
                                 relative_position_embedding_type=C.RelativePositionEmbeddingType.ROTARY_COMPLEX)
    assert cplx.rotary_embedding.freqs_cis_real.shape == (16, 32) and cplx._fusable_rotary
    real, imag = cplx.rotary_embedding.tables()      # the fused kernels take fp32 [rows, d / 2] tables
    assert real.dtype == torch.float32 and real.shape == (16, 32) and imag.shape == (16, 32)
    partial = ParallelSelfAttention(256, 4, hip, dtype=torch.bfloat16, device=CPU, rotary_config=C.RotaryConfig(dimensions=32, max_seq_length=16))
    assert not partial._fusable_rotary               # rotary over part of the head: stand-alone kernel
    with pytest.raises(AssertionError, match="LoRa"):   # same failure as the reference without a LoRA configuration
        partial.merge_lora_weights()
    assert all("freqs_cis" not in k for k in cplx.state_dict())
    with pytest.raises(AssertionError, match="kv heads"):
        ParallelSelfAttention(256, 4, hip, dtype=torch.bfloat16, device=CPU, num_kv_heads=2, qkv_in_one=True,
                              rotary_config=C.RotaryConfig(dimensions=64))
    with pytest.raises(AssertionError):
        ParallelSwiGLUMLP(10, 0.33, device=CPU)
    # the reference's default architecture (LayerNorm + GELU MLP) builds, with the reference's parameter names
    dflt = TransformerLayer(_arch(mlp_type="default", norm_type="layernorm", mlp_factor=4.0, mlp_bias=True), 0, device=CPU)
    names = set(dflt.state_dict())
    assert {"input_layernorm.weight", "input_layernorm.bias", "post_attention_layernorm.bias", "mlp.dense_in.weight",
            "mlp.dense_in.bias", "mlp.dense_out.weight"} <= names and "mlp.siglu_weight.weight" not in names
    with pytest.raises(NotImplementedError):
        TransformerLayer(_arch(umup={"enable": True}), 0, device=CPU)
    assert RMSNorm(16, CPU).weight.tolist() == [1.0] * 16


def test_checked_once_handles_inference_tensors_and_caches_by_version():
    """The validation cache keys on the version counter; tensors made under torch.inference_mode() have none and
    must be validated on every call instead of raising."""
    from scaling_amd import nn as N
    calls = []

    def compute():
        calls.append(1)
        return True

    t = torch.arange(4)
    assert N._checked_once("test_kind", t, (1,), compute) and N._checked_once("test_kind", t, (1,), compute)
    assert len(calls) == 1                      # second call is a cache hit
    t.add_(1)                                   # in-place write bumps the version: validated again
    assert N._checked_once("test_kind", t, (1,), compute) and len(calls) == 2
    with torch.inference_mode():
        u = torch.arange(4)
        assert N._checked_once("test_kind", u, (1,), compute) and N._checked_once("test_kind", u, (1,), compute)
    assert len(calls) == 4                      # no version counter: no caching, no exception
    att = ParallelSelfAttention(256, 4, C.MaskedSoftmaxConfig(kernel="hip"), dtype=torch.bfloat16, device=CPU,
                                rotary_config=C.RotaryConfig(dimensions=64, max_seq_length=16))
    with torch.inference_mode():
        att._check_positions(torch.arange(16))
        with pytest.raises(IndexError):
            att._check_positions(torch.arange(17))
        assert att._rows_are_single_documents(torch.tensor([0, 8, 16], dtype=torch.int32), 2, 8)
        assert not att._rows_are_single_documents(torch.tensor([0, 5, 16], dtype=torch.int32), 2, 8)


def test_greedy_choice_takes_batch_position_vocabulary():
    from scaling_amd.inference import sample_argmax

    logits = torch.tensor([[[5.0, 1.0, 2.0], [0.0, 3.0, 3.0]], [[1.0, 0.0, 9.0], [4.0, -1.0, float("nan")]]])
    assert sample_argmax(logits).tolist() == [1, 2]
    with pytest.raises(IndexError):
        sample_argmax(logits[0])
