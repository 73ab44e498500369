"""Tensor-level entry points of the HIP kernels (through the C ABI) and their autograd wrappers.

Every function here launches a hand-written gfx950 kernel on the current stream.  None of them falls
back to PyTorch arithmetic: tensors must live on the GPU, and shapes or dtypes a kernel does not
support raise.  The checks are here; argument blocks, allocations, launches and autograd nodes are native
(csrc/host.cpp).  The nodes keep tensors with ``save_for_backward`` only, so they work
under saved-tensor hooks (activation checkpointing) and are deterministic under recomputation.
"""

import ctypes  # noqa: F401 - for callers that fill an argument block with _fill_attn_args and hand it to the C ABI
import math
from typing import Optional, Tuple

import torch
from torch.overrides import _get_current_function_mode_stack, has_torch_function
from torch.utils._device import DeviceContext

from . import _lib
from ._lib import MiAttnArgs, check, dtype_code, ptr, stream_ptr

__all__ = [
    "rms_norm", "swiglu", "rotary_embedding", "rotary_embedding_complex", "attention", "attention_forward", "attention_backward",
    "decode_attention", "rms_norm_forward", "rms_norm_backward", "swiglu_forward", "swiglu_backward",
    "cross_entropy", "cross_entropy_forward", "linear_cross_entropy", "weighted_cross_entropy", "add_rms_norm",
]


def _need_cuda(*tensors):
    _lib.require_device()
    for t in tensors:
        if t is not None and not t.is_cuda:
            raise RuntimeError("scaling_amd ops take GPU tensors only (got a CPU tensor); there is no CPU path")


# ------------------------------------------------------------------------------------------------
# RMSNorm
# ------------------------------------------------------------------------------------------------
def add_rms_norm(x: torch.Tensor, residual: torch.Tensor, weight: torch.Tensor, eps: float) -> Tuple[torch.Tensor, torch.Tensor]:
    """(x + residual, rms_norm(x + residual) * weight) in one launch (inference; no autograd).  The sum is rounded
    to the tensor dtype before it is normalised, as the separate add and norm would do."""
    _need_cuda(x, residual, weight)
    assert x.shape == residual.shape and x.dtype == residual.dtype == weight.dtype and x.shape[-1] == weight.shape[0]
    with torch.no_grad():
        return _lib.host().add_norm(x, residual, weight, None, eps, False)


def add_norm(x: torch.Tensor, residual: Optional[torch.Tensor], weight: torch.Tensor, bias: Optional[torch.Tensor], eps: float,
             layer_norm: bool) -> Tuple[torch.Tensor, torch.Tensor]:
    """(s, norm(s)) with s = x + residual, or s = x without a residual, in one launch; differentiable, with the gradient that
    reaches s directly added inside the norm's backward kernel.  LayerNorm or RMSNorm (no bias)."""
    _need_cuda(x, residual, weight, bias)
    assert x.shape[-1] == weight.shape[0] and weight.dtype == x.dtype and (residual is None or residual.shape == x.shape)
    return _lib.host().add_norm(x, residual, weight, bias, eps, layer_norm)


def rms_norm_forward(x: torch.Tensor, weight: torch.Tensor, eps: float) -> torch.Tensor:
    _need_cuda(x, weight)
    assert x.shape[-1] == weight.shape[0] and weight.dtype == x.dtype
    return _lib.host().rms_norm_forward(x, weight, eps)


def rms_norm_backward(x: torch.Tensor, weight: torch.Tensor, dy: torch.Tensor, eps: float):
    _need_cuda(x, weight, dy)
    return _lib.host().rms_norm_backward(x, weight, dy, eps)


def rms_norm(x: torch.Tensor, weight: torch.Tensor, eps: float = 1e-5) -> torch.Tensor:
    """y = x * rsqrt(mean(x^2, -1) + eps) * weight (fp32 math, one rounding)."""
    _need_cuda(x, weight)
    assert x.shape[-1] == weight.shape[0] and weight.dtype == x.dtype
    return _lib.host().rms_norm(x, weight, eps)


# ------------------------------------------------------------------------------------------------
# LayerNorm, GELU (the reference's default norm / activation)
# ------------------------------------------------------------------------------------------------
def layer_norm_forward(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor], eps: float,
                       save_stats: bool = False):
    """y, or (y, stats) with stats an fp32 [2, n_rows] tensor (row means, then reciprocal standard deviations)
    for layer_norm_backward when save_stats is set."""
    _need_cuda(x, weight, bias)
    assert x.shape[-1] == weight.shape[0] and weight.dtype == x.dtype
    y, stats = _lib.host().layer_norm_forward(x, weight, bias, eps, save_stats)
    return (y, stats) if save_stats else y


def layer_norm_backward(x: torch.Tensor, weight: torch.Tensor, dy: torch.Tensor, eps: float, need_bias_grad: bool = True,
                        stats: Optional[torch.Tensor] = None):
    """(dx, dweight, dbias).  `stats` is what layer_norm_forward(save_stats=True) returned for the same x, or
    None to have the statistics recomputed."""
    _need_cuda(x, weight, dy)
    if stats is not None and x.numel() != 0:
        assert stats.dtype == torch.float32 and stats.is_contiguous() and stats.shape == (2, x.numel() // x.shape[-1])
    return _lib.host().layer_norm_backward(x, weight, dy, eps, need_bias_grad, stats)


def layer_norm(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor] = None, eps: float = 1e-5) -> torch.Tensor:
    """(x - mean) * rsqrt(var + eps) * weight + bias over the last dimension (fp32 math, one rounding)."""
    _need_cuda(x, weight, bias)
    assert x.shape[-1] == weight.shape[0] and weight.dtype == x.dtype
    return _lib.host().layer_norm(x, weight, bias, eps)


def gelu_forward(x: torch.Tensor) -> torch.Tensor:
    _need_cuda(x)
    return _lib.host().gelu_forward(x)


def gelu_backward(x: torch.Tensor, dy: torch.Tensor) -> torch.Tensor:
    _need_cuda(x, dy)
    return _lib.host().gelu_backward(x, dy)


def gelu(x: torch.Tensor) -> torch.Tensor:
    """Exact (erf) GELU."""
    _need_cuda(x)
    return _lib.host().gelu(x)


# ------------------------------------------------------------------------------------------------
# SwiGLU
# ------------------------------------------------------------------------------------------------
def swiglu_forward(a: torch.Tensor, gate: torch.Tensor) -> torch.Tensor:
    _need_cuda(a, gate)
    assert a.shape == gate.shape and a.dtype == gate.dtype
    return _lib.host().swiglu_forward(a, gate)


def swiglu_backward(a: torch.Tensor, gate: torch.Tensor, dout: torch.Tensor):
    _need_cuda(a, gate, dout)
    return _lib.host().swiglu_backward(a, gate, dout)


def swiglu(a: torch.Tensor, gate: torch.Tensor) -> torch.Tensor:
    """silu(a) * gate."""
    _need_cuda(a, gate)
    assert a.shape == gate.shape and a.dtype == gate.dtype
    return _lib.host().swiglu(a, gate)


# ------------------------------------------------------------------------------------------------
# linear projections
# ------------------------------------------------------------------------------------------------
def _taken_over(operands: tuple) -> bool:
    """Whether an operand or a mode takes over torch functions, and so has to see them.  A default device (torch.set_default_device,
    `with torch.device(...)`) is such a mode too, which does nothing to a call on tensors that are there."""
    if not has_torch_function(operands):
        return False
    return any(not isinstance(mode, DeviceContext) for mode in _get_current_function_mode_stack()) or \
        any(t is not None and type(t) is not torch.Tensor and type(t).__torch_function__ is not torch._C._disabled_torch_function_impl
            for t in operands)


def linear(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor] = None,
           residual: Optional[torch.Tensor] = None, inference: bool = False) -> torch.Tensor:
    """x W^T + b (torch.nn.functional.linear) (+ residual), on the matrix kernel of this package where the product is too small to fill
    the chip and on the library product elsewhere.  `inference`: no gradients follow, so the forward product alone decides; the same value
    gives the same bits with and without gradients."""
    if _taken_over((x, weight, bias, residual)):
        y = torch.nn.functional.linear(x, weight, bias)
        return y if residual is None else y + residual
    return _lib.host().linear(x, weight, bias, residual, inference)


def projections(x: torch.Tensor, weights, biases, inference: bool = False):
    """[linear(x, w, b) for up to three (w, b)] of one input, whose gradient is then one sum inside the products."""
    if _taken_over((x, *weights, *biases)):
        return [torch.nn.functional.linear(x, w, b) for w, b in zip(weights, biases)]
    return _lib.host().projections(x, weights, biases, inference)


# ------------------------------------------------------------------------------------------------
# rotary (stand-alone kernel)
# ------------------------------------------------------------------------------------------------
def _check_rotary(x, cos, sin, position_ids):
    _need_cuda(x, cos, sin, position_ids)
    assert x.dim() == 3 and x.stride(2) == 1
    assert cos.is_contiguous() and sin.is_contiguous() and cos.shape == sin.shape and cos.dim() == 2
    assert position_ids is None or (position_ids.dtype == torch.int64 and position_ids.numel() == x.shape[0])


def _rotary_launch(x, cos, sin, position_ids, seq_len_for_null_ids, inverse):
    """x: [tokens, heads, head_dim] view whose last dim is contiguous; cos/sin: [rows, rot_dim]."""
    _check_rotary(x, cos, sin, position_ids)
    return _lib.host().rotary_launch(x, cos, sin, position_ids, int(seq_len_for_null_ids), bool(inverse), False)


def rotary_embedding(x: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor,
                     position_ids: Optional[torch.Tensor] = None, seq_len_for_null_ids: int = 0) -> torch.Tensor:
    """Rotate-half rotary on x [tokens, heads, head_dim]; position_ids int64 [tokens] (flattened (b s))."""
    _check_rotary(x, cos, sin, position_ids)
    return _lib.host().rotary(x, cos, sin, position_ids, int(seq_len_for_null_ids), False)


def rotary_embedding_complex(x: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor,
                             position_ids: Optional[torch.Tensor] = None, seq_len_for_null_ids: int = 0) -> torch.Tensor:
    """Interleaved-pair rotary on x [tokens, heads, head_dim]; cos / sin fp32 [rows, head_dim/2]."""
    _check_rotary(x, cos, sin, position_ids)
    assert cos.dtype == torch.float32 and sin.dtype == torch.float32 and cos.shape[1] * 2 == x.shape[2]
    return _lib.host().rotary(x, cos, sin, position_ids, int(seq_len_for_null_ids), True)


# ------------------------------------------------------------------------------------------------
# cross entropy over vocabulary rows
# ------------------------------------------------------------------------------------------------
def cross_entropy_forward(logits: torch.Tensor, targets: torch.Tensor, row_scale: Optional[torch.Tensor] = None,
                          dlogits: Optional[torch.Tensor] = None, want_lse: bool = False):
    """One launch over logits [rows, vocab]: returns (losses fp32 [rows], argmax int32 [rows]) (+ lse if asked).

    With ``dlogits`` (same shape and dtype, may be ``logits`` itself) the gradient
    ``row_scale[r] * (softmax(x_r) - onehot(t_r))`` is written in the same pass."""
    _need_cuda(logits, targets, row_scale, dlogits)
    assert logits.dim() == 2 and logits.stride(1) == 1, "logits must be [rows, vocab] with contiguous vocab"
    assert targets.dtype == torch.int64 and targets.is_contiguous() and targets.numel() == logits.shape[0]
    if row_scale is not None:
        assert row_scale.dtype == torch.float32 and row_scale.is_contiguous() and row_scale.numel() == logits.shape[0]
    if dlogits is not None:
        assert dlogits.shape == logits.shape and dlogits.dtype == logits.dtype and dlogits.stride(1) == 1
    n, v = logits.shape
    losses = torch.empty(n, dtype=torch.float32, device=logits.device)
    argmax = torch.empty(n, dtype=torch.int32, device=logits.device)
    # with a gradient, rows that are very long, not a whole number of 16-byte vectors or not 16-byte aligned take two
    # launches that hand the log-sum-exp over: always supply the (rows x 4 bytes) buffer
    need_lse = want_lse or dlogits is not None
    lse = torch.empty(n, dtype=torch.float32, device=logits.device) if need_lse else None
    check(_lib.load().mi_cross_entropy(ptr(logits), ptr(targets), ptr(row_scale), ptr(losses), ptr(lse), ptr(argmax), ptr(dlogits),
                                       n, v, logits.stride(0), dlogits.stride(0) if dlogits is not None else 0,
                                       dtype_code(logits.dtype), stream_ptr()), "mi_cross_entropy")
    return (losses, argmax, lse) if want_lse else (losses, argmax)


class _CrossEntropy(torch.autograd.Function):
    @staticmethod
    def forward(ctx, logits, targets):
        losses, argmax = cross_entropy_forward(logits, targets)
        ctx.save_for_backward(logits, targets)
        ctx.mark_non_differentiable(argmax)
        return losses, argmax

    @staticmethod
    def backward(ctx, dlosses, _dargmax):
        logits, targets = ctx.saved_tensors
        dlogits = torch.empty_like(logits)
        cross_entropy_forward(logits, targets, row_scale=dlosses.float().contiguous(), dlogits=dlogits)
        return dlogits, None


def cross_entropy(logits: torch.Tensor, targets: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor]:
    """Differentiable per-row losses (fp32) and the row argmax (int32) of logits [rows, vocab]."""
    if logits.stride(1) != 1:
        logits = logits.contiguous()
    return _CrossEntropy.apply(logits, targets.contiguous())


def weighted_cross_entropy(logits: torch.Tensor, targets: torch.Tensor, weights: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor]:
    """(loss, accuracy) of logits [rows, vocab]: loss = sum(w * CE) / sum(w), accuracy = hit rate of the row argmax among the
    rows with w > 0; weights float32 [rows], not differentiable here.  Two launches forward, one backward."""
    _need_cuda(logits, targets, weights)
    if logits.stride(1) != 1:
        logits = logits.contiguous()
    return _lib.host().weighted_cross_entropy(logits, targets.contiguous(), weights.contiguous())


def linear_cross_entropy(h: torch.Tensor, weight: torch.Tensor, targets: torch.Tensor, loss_weights: torch.Tensor,
                         chunk_rows: int = 8192) -> Tuple[torch.Tensor, torch.Tensor]:
    """LM head + weighted cross entropy, chunked over rows.  h [rows, hidden], weight [vocab, hidden].
    The transient logits take chunk_rows * vocab * 2 bytes (2.1 GB at the default and a 128k vocabulary); larger
    chunks keep the three GEMMs efficient and the fp32 accumulation of dweight rare (measured at 8192 rows x 128256:
    23.4 ms with one chunk, 28.4 ms with four, 39.9 ms with eight).

    Returns (loss, argmax int32 [rows]); the gradients of h and weight are computed in the forward pass."""
    return _linear_cross_entropy(h, weight, targets, loss_weights, chunk_rows)[:2]


def _linear_cross_entropy(h, weight, targets, loss_weights, chunk_rows):
    """(loss, argmax, accuracy)"""
    _need_cuda(h, weight, targets, loss_weights)
    assert h.dim() == 2 and weight.dim() == 2 and h.shape[1] == weight.shape[1] and h.dtype == weight.dtype
    return _lib.host().linear_cross_entropy(h.contiguous(), weight, targets.contiguous().view(-1),
                                            loss_weights.detach().float().contiguous().view(-1), int(chunk_rows))


# ------------------------------------------------------------------------------------------------
# attention core
# ------------------------------------------------------------------------------------------------
def _fused_rotary_kind(cos: torch.Tensor, sin: torch.Tensor, head_dim: int, dtype: torch.dtype) -> bool:
    """Checks the tables of a fused rotary; True for the interleaved-pair variant (fp32 tables [rows, head_dim / 2],
    RotaryEmbeddingComplex), False for rotate-half (tables [rows, head_dim] in the tensors' dtype)."""
    assert cos.is_contiguous() and sin.is_contiguous() and cos.shape == sin.shape and cos.dim() == 2
    if cos.dtype == torch.float32 and cos.shape[1] * 2 == head_dim and dtype != torch.float32:
        assert sin.dtype == torch.float32
        return True
    assert cos.dtype == dtype and sin.dtype == dtype and cos.shape[1] == head_dim, \
        "fused rotary takes [rows, head_dim] tables in the data dtype or fp32 [rows, head_dim / 2] tables (interleaved pairs)"
    return False


def _fill_attn_args(q, k, v, o, lse, cu_q, cu_k, causal, scale, rotary=None, flags=0, dropout=None, q_rot=None) -> MiAttnArgs:
    a = MiAttnArgs()
    a.flags = int(flags)
    a.q, a.k, a.v, a.o, a.lse = ptr(q), ptr(k), ptr(v), ptr(o), ptr(lse)
    a.cu_seqlens_q, a.cu_seqlens_k = ptr(cu_q), ptr(cu_k)
    a.n_docs = cu_q.numel() - 1
    a.causal = int(bool(causal))
    a.total_q, a.total_k = q.shape[0], k.shape[0]
    a.n_q_heads, a.n_kv_heads, a.head_dim = q.shape[1], k.shape[1], q.shape[2]
    a.dtype = dtype_code(q.dtype)
    a.q_stride_token, a.q_stride_head = q.stride(0), q.stride(1)
    a.k_stride_token, a.k_stride_head = k.stride(0), k.stride(1)
    a.v_stride_token, a.v_stride_head = v.stride(0), v.stride(1)
    a.o_stride_token, a.o_stride_head = o.stride(0), o.stride(1)
    a.softmax_scale = float(scale)
    if rotary is not None:
        cos, sin, pos_q, pos_k = rotary
        a.rotary_cos, a.rotary_sin = ptr(cos), ptr(sin)
        a.position_ids_q, a.position_ids_k = ptr(pos_q), ptr(pos_k)
        a.rotary_table_rows = cos.shape[0]
        a.rotary_interleaved = int(_fused_rotary_kind(cos, sin, q.shape[2], q.dtype))
        a.q_rot_out = ptr(q_rot)
    if dropout is not None and dropout[0] > 0.0:
        a.dropout_p, a.dropout_seed = float(dropout[0]), int(dropout[1]) & 0xFFFFFFFFFFFFFFFF
    a.stream = stream_ptr()
    return a


def _check_qkv(q, k, v, cu_q, cu_k):
    _need_cuda(q, k, v, cu_q, cu_k)
    for t in (q, k, v):
        assert t.dim() == 3 and t.stride(2) == 1, "q/k/v must be [tokens, heads, head_dim] with contiguous features"
    assert k.shape == v.shape and q.shape[2] == k.shape[2]
    assert cu_q.dtype == torch.int32 and cu_q.is_contiguous()
    if cu_k is not None:
        assert cu_k.dtype == torch.int32 and cu_k.is_contiguous() and cu_k.numel() == cu_q.numel()


def _dropout_args(dropout):
    """(p, seed as an unsigned 64-bit integer) of an optional (p, seed) pair."""
    return (float(dropout[0]), int(dropout[1]) & 0xFFFFFFFFFFFFFFFF) if dropout is not None and dropout[0] > 0.0 else (0.0, 0)


SPLIT_P = 4   # MI_ATTN_SPLIT_P


def attention_forward(q, k, v, cu_seqlens_q, cu_seqlens_k=None, causal=True, softmax_scale=None, rotary=None, flags=0,
                      dropout=None, return_rotated_q=False, precise=False):
    """Returns (o [tokens, n_q_heads, head_dim], lse fp32 [n_q_heads, tokens]) (+ the rotated q if asked).

    rotary: optional (cos, sin, position_ids_q, position_ids_k), q and k are rotated while they are loaded:
    rotate-half with [rows, head_dim] tables in q's dtype, interleaved pairs with fp32 [rows, head_dim / 2] tables.
    position_ids_k = None: k is rotated already, only q is rotated in the kernel (the cheaper arrangement, see
    include/mi355_layer.h); return_rotated_q then also returns the rotated q (strides of q) for the backward.

    dropout: optional (p, seed) for dropout on the attention probabilities; the backward needs the same pair.

    flags: 0 lets the library pick the tiling; 1 / 2 pin one / two query groups per wavefront.
    precise: accuracy mode (probabilities enter P V as two bf16 terms; no dropout, rotary on q only)."""
    _check_qkv(q, k, v, cu_seqlens_q, cu_seqlens_k)
    if softmax_scale is None:
        softmax_scale = 1.0 / math.sqrt(q.shape[2])
    if precise:
        flags |= SPLIT_P
    cos = sin = pos_q = pos_k = None
    interleaved = False
    if rotary is not None:
        cos, sin, pos_q, pos_k = rotary
        interleaved = _fused_rotary_kind(cos, sin, q.shape[2], q.dtype)
        assert pos_q.dtype == torch.int64 and pos_q.is_contiguous() and pos_q.numel() == q.shape[0]
        assert pos_k is None or (pos_k.dtype == torch.int64 and pos_k.is_contiguous() and pos_k.numel() == k.shape[0])
    else:
        assert not return_rotated_q
    p, seed = _dropout_args(dropout)
    o, lse, q_rot = _lib.host().attention_forward(q, k, v, cu_seqlens_q, cu_seqlens_k, bool(causal), float(softmax_scale), int(flags), p, seed,
                                                  cos, sin, pos_q, pos_k, interleaved, bool(return_rotated_q))
    return (o, lse, q_rot) if return_rotated_q else (o, lse)


def attention_backward(do, q, k, v, o, lse, cu_seqlens_q, cu_seqlens_k=None, causal=True, softmax_scale=None,
                       flags=0, buffers=None, dropout=None, rotary=None, precise=False):
    """Returns (dq, dk, dv).  The summation order is fixed: results are bit-reproducible
    (what masked_softmax.deterministic_flash_attn_bwd asks of the reference's fused kernel holds always).

    rotary = (cos, sin, position_ids_q, position_ids_k): q and k are the ROTATED tensors the forward attended with, and
    dq / dk come back as gradients of the unrotated ones (rotated back inside the kernels, one rounding).

    flags: 0 runs the whole backward; 16 / 32 / 64 run only the delta / dK-dV / dQ kernel (timing aid).
    buffers: optional (dq, dk, dv, workspace) to reuse across calls.
    precise: accuracy mode (P and dS enter their MFMAs as two bf16 terms each; no dropout)."""
    _check_qkv(q, k, v, cu_seqlens_q, cu_seqlens_k)
    if precise:
        flags |= SPLIT_P
    if softmax_scale is None:
        softmax_scale = 1.0 / math.sqrt(q.shape[2])
    dq, dk, dv, ws = buffers if buffers is not None else (None, None, None, None)
    assert dq is None or dq.stride() == q.stride()
    cos = sin = pos_q = pos_k = None
    interleaved = False
    if rotary is not None:
        cos, sin, pos_q, pos_k = rotary
        interleaved = _fused_rotary_kind(cos, sin, q.shape[2], q.dtype)
    p, seed = _dropout_args(dropout)
    return _lib.host().attention_backward(do, q, k, v, o, lse, cu_seqlens_q, cu_seqlens_k, bool(causal), float(softmax_scale), int(flags), p, seed,
                                          cos, sin, pos_q, pos_k, interleaved, dq, dk, dv, ws)


def next_dropout_seed(device: torch.device) -> int:
    """A fresh 64-bit seed from the device's default generator without touching the GPU: (seed, offset) of the
    Philox state, with the offset advanced as torch's own random kernels do.  The state is part of what
    torch.utils.checkpoint saves and restores, so a recomputed forward draws the same seed."""
    gen = torch.cuda.default_generators[device.index if device.index is not None else torch.cuda.current_device()]
    seed, offset = gen.initial_seed(), gen.get_offset()
    gen.set_offset(offset + 4)
    return (seed * 0x9E3779B97F4A7C15 + offset * 0xD1B54A32D192ED03 + 0x2545F4914F6CDD1D) & 0xFFFFFFFFFFFFFFFF


def attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, cu_seqlens_q: torch.Tensor,
              cu_seqlens_k: Optional[torch.Tensor] = None, causal: bool = True,
              softmax_scale: Optional[float] = None, dropout_p: float = 0.0,
              dropout_seed: Optional[int] = None, rotary=None, deterministic: bool = False, precise: bool = False) -> torch.Tensor:
    """Differentiable attention core on q [tokens, n_q, d], k/v [tokens_k, n_kv, d] (bfloat16, float16 or float32;
    float32 tensors run separate kernels on the fp32 matrix pipe with exact fp32 probabilities, without dropout).

    Tokens are the flattened (batch seq) axis; cu_seqlens are int32 offsets on it.  Returns
    o [tokens, n_q, d].  dropout_p > 0 drops attention probabilities (attention.py:204-207) with a mask that
    is a function of (dropout_seed, head, query, key); without a seed one is drawn from the device generator.
    The drop probability is quantised to round(256 p) / 256.

    rotary = (cos, sin, position_ids_q, position_ids_k) applies the rotary embedding of the whole head to q and k
    (attention.py:836-845; table formats as for attention_forward) and differentiates through it: q is rotated while
    the forward kernel loads it, k by one stand-alone launch, and the backward kernels rotate dq / dk back in their
    epilogues, with or without autograd, with or without dropout.
    deterministic mirrors masked_softmax.deterministic_flash_attn_bwd of the reference; the kernels sum in a fixed
    order whatever its value.
    precise selects the accuracy mode of forward and backward: P and dS enter their products as two bf16 terms, which
    brings outputs and gradients within max-abs 2e-2 / mean-relative 1e-3 of the fp32 reference (the default mode
    rounds P once to bf16 as the reference does); bench.py times both modes (`accuracy_mode.time_over_default`); no
    dropout.  Exception: with `rotary` the rotated q and k are rounded once to the I/O dtype before the score product
    in either mode, which leaves a mean-relative error of about 2e-3 against the fp32 reference (0.5 - 0.75 x what the
    reference's own bf16 path shows there).
    """
    if softmax_scale is None:
        softmax_scale = 1.0 / math.sqrt(q.shape[2])
    if dropout_p > 0.0 and dropout_seed is None:
        dropout_seed = next_dropout_seed(q.device)
    cos = sin = pos_q = pos_k = None
    if rotary is not None and q.dtype == torch.float32:
        # float32 tensors: the rotation runs as the stand-alone (differentiable) kernel in front of the fp32 attention core
        cos, sin, pos_q, pos_k = rotary
        rot = rotary_embedding_complex if cos.shape[1] * 2 == q.shape[2] else rotary_embedding
        q, k = rot(q, cos, sin, pos_q), rot(k, cos, sin, pos_k)
        rotary = cos = sin = pos_q = pos_k = None
    _check_qkv(q, k, v, cu_seqlens_q, cu_seqlens_k)
    interleaved = False
    if rotary is not None:
        cos, sin, pos_q, pos_k = rotary
        interleaved = _fused_rotary_kind(cos, sin, q.shape[2], q.dtype)
        assert pos_q.dtype == torch.int64 and pos_q.is_contiguous() and pos_q.numel() == q.shape[0]
        assert pos_k.dtype == torch.int64 and pos_k.is_contiguous() and pos_k.numel() == k.shape[0]
    p, seed = _dropout_args((dropout_p, dropout_seed if dropout_seed is not None else 0))
    return _lib.host().attention(q, k, v, cu_seqlens_q, cu_seqlens_k, bool(causal), float(softmax_scale), p, seed, cos, sin, pos_q, pos_k,
                                 interleaved, bool(precise))


def attention_qkv(qkv: torch.Tensor, cu_seqlens_q: torch.Tensor, cu_seqlens_k: Optional[torch.Tensor] = None, causal: bool = True,
                  softmax_scale: Optional[float] = None, dropout_p: float = 0.0, dropout_seed: Optional[int] = None, rotary=None) -> torch.Tensor:
    """`attention` on one projection output qkv [tokens, heads, 3 d] (per head q, then k, then v), whose gradient comes back in
    the same layout."""
    d = qkv.shape[2] // 3
    if softmax_scale is None:
        softmax_scale = 1.0 / math.sqrt(d)
    if dropout_p > 0.0 and dropout_seed is None:
        dropout_seed = next_dropout_seed(qkv.device)
    cos = sin = pos_q = pos_k = None
    interleaved = False
    if rotary is not None:
        cos, sin, pos_q, pos_k = rotary
        interleaved = _fused_rotary_kind(cos, sin, d, qkv.dtype)
        assert pos_q.dtype == torch.int64 and pos_q.is_contiguous() and pos_q.numel() == qkv.shape[0]
        assert pos_k.dtype == torch.int64 and pos_k.is_contiguous() and pos_k.numel() == qkv.shape[0]
    p, seed = _dropout_args((dropout_p, dropout_seed if dropout_seed is not None else 0))
    return _lib.host().attention_qkv(qkv, cu_seqlens_q, cu_seqlens_k, bool(causal), float(softmax_scale), p, seed, cos, sin, pos_q, pos_k, interleaved)


# ------------------------------------------------------------------------------------------------
# decode attention over a pre-allocated KV cache
# ------------------------------------------------------------------------------------------------
def _decode_scratch(batch: int, n_q_heads: int, head_dim: int, max_ctx: int, device) -> torch.Tensor:
    nbytes = _lib.load().mi_attn_decode_workspace_bytes(batch, n_q_heads, head_dim, max_ctx)
    return torch.empty(nbytes // 4, dtype=torch.float32, device=device)


def decode_workspace(batch: int, n_q_heads: int, head_dim: int, max_ctx: int, device) -> torch.Tensor:
    """Scratch of `decode_attention` for calls that do not overlap.  With it come the arrival counts (attribute `tickets`, int32, zero
    between calls) by which the last workgroup of a small call merges the splits of the keys in the same launch; a workspace without them (a
    slice, a tensor of the caller's own) takes a second launch for the same result.  The counts are cleared on the current stream, so a first call
    on another stream waits for this one; and where calls on one workspace overlapped all the same, not these calls alone are spoilt: counts
    that are not zero again make later ones merge too early or never, until `tickets` is cleared (`workspace.tickets.zero_()`)."""
    workspace = _decode_scratch(batch, n_q_heads, head_dim, max_ctx, device)
    workspace.tickets = torch.zeros(max(batch * n_q_heads, 0), dtype=torch.int32, device=device)
    return workspace


def decode_attention(q: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor, ctx_len: torch.Tensor,
                     k_new: Optional[torch.Tensor] = None, v_new: Optional[torch.Tensor] = None,
                     rotary: Optional[Tuple[torch.Tensor, torch.Tensor, torch.Tensor]] = None,
                     softmax_scale: Optional[float] = None, workspace: Optional[torch.Tensor] = None,
                     n_splits: int = 0, out: Optional[torch.Tensor] = None, static_scratch: bool = False) -> torch.Tensor:
    """One decode step.  q [B, n_q, d]; caches [B, max_ctx, n_kv, d]; ctx_len int32 [B] counts the valid
    keys INCLUDING the token appended by this call (k_new/v_new [B, n_kv, d], written at ctx_len-1).
    rotary = (cos, sin, position_ids[B]) rotates q and k_new inside the kernels (table formats as for
    attention_forward: rotate-half or interleaved pairs).  q, k_new and v_new may be
    column slices of one projection output: only their [heads, d] part has to be contiguous.
    static_scratch=True calls the entry point that allocates nothing (partial results in the library's static
    device array; `out` should be given too, and calls on one GPU must not overlap)."""
    _need_cuda(q, k_cache, v_cache, ctx_len)
    B, nq, d = q.shape

    def _check_rows(t):
        assert t.stride(2) == 1 and t.stride(1) == d and t.stride(0) % 8 == 0, "each sequence's [heads, d] block must be contiguous"

    assert k_cache.dim() == 4 and k_cache.shape == v_cache.shape
    assert k_cache.stride() == v_cache.stride() and k_cache.stride(3) == 1
    assert ctx_len.dtype == torch.int32 and ctx_len.numel() == B
    if softmax_scale is None:
        softmax_scale = 1.0 / math.sqrt(d)
    if workspace is None and not static_scratch:
        workspace = _decode_scratch(B, nq, d, k_cache.shape[1], q.device)
    if out is None:
        out = torch.empty((B, nq, d), dtype=q.dtype, device=q.device)
    _check_rows(q)
    if k_new is not None:
        assert k_new.shape == (B, k_cache.shape[2], d) and v_new.shape == k_new.shape
        _check_rows(k_new)
        _check_rows(v_new)
    cos = sin = pos = None
    interleaved = False
    if rotary is not None:
        cos, sin, pos = rotary
        interleaved = _fused_rotary_kind(cos, sin, d, q.dtype)
        assert pos.dtype == torch.int64 and pos.numel() == B and pos.is_contiguous()
    _lib.host().decode_attention(q, k_cache, v_cache, ctx_len, k_new, v_new, cos, sin, pos, interleaved, float(softmax_scale),
                                 None if static_scratch else workspace, None if static_scratch else getattr(workspace, "tickets", None),
                                 int(n_splits), out, bool(static_scratch))
    return out


def layer(*arguments) -> torch.Tensor:
    """A pre-norm layer in one native call (csrc/host.cpp op_layer); the callers check what it takes."""
    return _lib.host().layer(*arguments)


ROWS_MAX = 16   # MI_ROWS_MAX


def norm_linear_rows(x: torch.Tensor, norm_weight: torch.Tensor, eps: float, weight: torch.Tensor) -> Optional[torch.Tensor]:
    """rms_norm(x) @ weight.T of up to 16 rows [rows, k] (inference); None where the kernel does not apply."""
    if _taken_over((x, norm_weight, weight)):
        return None
    return _lib.host().norm_linear_rows(x, norm_weight, eps, weight)


def argmax_rows(x: torch.Tensor) -> torch.Tensor:
    """torch.argmax(x, dim=-1) of x [rows, n]."""
    index = None if _taken_over((x,)) or not x.is_cuda else _lib.host().argmax_rows(x)
    return torch.argmax(x, dim=-1) if index is None else index


def argmax_embed(x: torch.Tensor, table: torch.Tensor) -> Optional[Tuple[torch.Tensor, torch.Tensor]]:
    """(argmax_rows(x), table[argmax_rows(x)]) of x [rows, n] and table [at least n, hidden] in one launch (inference); None where the kernel does not apply."""
    return None if _taken_over((x, table)) or not x.is_cuda else _lib.host().argmax_embed(x, table)


def decode_layer_arguments(norm1, eps1, qkv_weights, dense, norm2, eps2, w_in, w_gate, w_out, head_dim, k_cache, v_cache, ctx_len, tables,
                           softmax_scale, workspace, dtype) -> Optional[tuple]:
    """What `decode_layer` takes beside the token: the layer's weights, its caches and rotary tables.  None for weights that have to see
    the functions they are used in."""
    if _taken_over((norm1, *qkv_weights, dense, norm2, w_in, w_gate, w_out)):
        return None
    cos, sin = tables
    interleaved = _fused_rotary_kind(cos, sin, head_dim, dtype)
    return (norm1, eps1, list(qkv_weights), dense, norm2, eps2, w_in, w_gate, w_out, head_dim, k_cache, v_cache, ctx_len, cos, sin, interleaved,
            float(softmax_scale), workspace)


def decode_layer(x: torch.Tensor, position_ids: torch.Tensor, arguments: tuple) -> Optional[torch.Tensor]:
    """A cached decode step of a whole layer, x [batch, 1, hidden] of up to 16 sequences, position_ids int64 [batch]: raises the context
    lengths by one, appends to the caches and returns the layer's output.  None, with nothing done, where the kernels do not apply."""
    if _taken_over((x, position_ids)):
        return None
    return _lib.host().decode_layer(x, position_ids, *arguments)
