"""Bindings of libmi355_layer.so (C ABI declared in include/mi355_layer.h): ctypes, and the native host path `mi355_host`
(csrc/host.cpp), a Python extension module that calls the same C ABI.

Both are loaded lazily.  There is no CPU or PyTorch fallback: if a shared object has not
been built, or a kernel returns an error status, a RuntimeError is raised.
"""

import ctypes
import importlib.util
import os
from ctypes import c_uint64, POINTER, Structure, c_char_p, c_float, c_int, c_int32, c_int64, c_size_t, c_void_p

import torch

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "csrc", "libmi355_layer.so")
HOST_PATH = os.path.join(_HERE, "csrc", "mi355_host.so")

MI_BF16, MI_F16, MI_F32 = 0, 1, 2
_DTYPE_CODE = {torch.bfloat16: MI_BF16, torch.float16: MI_F16, torch.float32: MI_F32}

EXPORTS = (
    "mi_version", "mi_last_error", "mi_status_string", "mi_check_device",
    "mi_rmsnorm_fwd", "mi_add_rmsnorm_fwd", "mi_rmsnorm_bwd_workspace_bytes", "mi_rmsnorm_bwd",
    "mi_layernorm_fwd", "mi_layernorm_bwd_workspace_bytes", "mi_layernorm_bwd", "mi_gelu_fwd", "mi_gelu_bwd", "mi_cross_entropy",
    "mi_cross_entropy_padded", "mi_argmax", "mi_argmax_embed", "mi_cross_entropy_mean_grad", "mi_loss_reduce", "mi_loss_row_scale", "mi_scale_inplace",
    "mi_swiglu_fwd", "mi_swiglu_bwd", "mi_rotary", "mi_rotary_complex", "mi_rotary_two",
    "mi_attn_fwd", "mi_attn_bwd_workspace_bytes", "mi_attn_bwd_workspace_bytes_kv", "mi_attn_bwd_workspace_bytes_for", "mi_attn_bwd",
    "mi_gemm", "mi_gemm_workspace_bytes", "mi_gemm_with_workspace", "mi_rows_product", "mi_transpose16", "mi_column_sum", "mi_add_rmsnorm_bwd", "mi_add_layernorm_fwd", "mi_add_layernorm_bwd", "mi_attn_decode_workspace_bytes", "mi_attn_decode", "mi_attn_decode_with_tickets", "mi_fill_cache", "mi_attn_decode_static_scratch_bytes", "mi_attn_decode_static",
)


class MiAttnArgs(Structure):
    _fields_ = [
        ("q", c_void_p), ("k", c_void_p), ("v", c_void_p), ("o", c_void_p), ("lse", c_void_p),
        ("cu_seqlens_q", c_void_p), ("cu_seqlens_k", c_void_p),
        ("n_docs", c_int32), ("causal", c_int32),
        ("total_q", c_int64), ("total_k", c_int64),
        ("n_q_heads", c_int32), ("n_kv_heads", c_int32), ("head_dim", c_int32), ("dtype", c_int32),
        ("q_stride_token", c_int64), ("q_stride_head", c_int64),
        ("k_stride_token", c_int64), ("k_stride_head", c_int64),
        ("v_stride_token", c_int64), ("v_stride_head", c_int64),
        ("o_stride_token", c_int64), ("o_stride_head", c_int64),
        ("softmax_scale", c_float), ("flags", c_int32),
        ("rotary_cos", c_void_p), ("rotary_sin", c_void_p),
        ("position_ids_q", c_void_p), ("position_ids_k", c_void_p),
        ("rotary_table_rows", c_int64),
        ("stream", c_void_p),
        ("dropout_p", c_float), ("dropout_seed", c_uint64), ("rotary_interleaved", c_int32),
        ("q_rot_out", c_void_p),
    ]


class MiAttnBwdArgs(Structure):
    _fields_ = [
        ("fwd", MiAttnArgs),
        ("d_o", c_void_p), ("dq", c_void_p), ("dk", c_void_p), ("dv", c_void_p),
        ("dk_stride_token", c_int64), ("dk_stride_head", c_int64),
        ("dv_stride_token", c_int64), ("dv_stride_head", c_int64),
        ("workspace", c_void_p), ("workspace_bytes", c_size_t),
    ]


class MiDecodeArgs(Structure):
    _fields_ = [
        ("q", c_void_p), ("k_cache", c_void_p), ("v_cache", c_void_p), ("o", c_void_p),
        ("ctx_len", c_void_p), ("k_new", c_void_p), ("v_new", c_void_p),
        ("rotary_cos", c_void_p), ("rotary_sin", c_void_p), ("position_ids", c_void_p),
        ("rotary_table_rows", c_int64),
        ("batch", c_int32), ("max_ctx", c_int32), ("n_q_heads", c_int32), ("n_kv_heads", c_int32),
        ("head_dim", c_int32), ("dtype", c_int32),
        ("cache_stride_batch", c_int64), ("cache_stride_token", c_int64), ("cache_stride_head", c_int64),
        ("softmax_scale", c_float), ("n_splits", c_int32),
        ("workspace", c_void_p), ("workspace_bytes", c_size_t),
        ("stream", c_void_p),
        ("q_stride_batch", c_int64), ("k_new_stride_batch", c_int64), ("v_new_stride_batch", c_int64),
        ("rotary_interleaved", c_int32),
    ]


class MiGemmSegment(Structure):
    _fields_ = [("p", c_void_p), ("q", c_void_p), ("ldp", c_int64), ("ldq", c_int64), ("k", c_int32)]


class MiGemmProblem(Structure):
    _fields_ = [
        ("segments", MiGemmSegment * 3),
        ("c", c_void_p), ("bias", c_void_p), ("add", c_void_p), ("p_sum", c_void_p),
        ("ldc", c_int64), ("ldadd", c_int64),
        ("n_segments", c_int32), ("p_kmajor", c_int32), ("q_kmajor", c_int32), ("m", c_int32), ("n", c_int32),
    ]


class MiRowsArgs(Structure):
    _fields_ = [
        ("x", c_void_p), ("norm_weight", c_void_p), ("w", c_void_p * 3), ("bias", c_void_p * 3), ("add", c_void_p * 3), ("out", c_void_p * 3),
        ("ldx", c_int64), ("ldw", c_int64 * 3), ("ldadd", c_int64 * 3), ("ldo", c_int64 * 3), ("count_up", c_void_p), ("n", c_int32 * 3),
        ("n_weights", c_int32), ("rows", c_int32), ("k", c_int32), ("glu", c_int32), ("dtype", c_int32), ("eps", c_float), ("stream", c_void_p),
    ]


class MiRotaryRows(Structure):
    _fields_ = [("x", c_void_p), ("out", c_void_p), ("x_stride_token", c_int64), ("x_stride_head", c_int64), ("out_stride_token", c_int64),
                ("out_stride_head", c_int64), ("n_heads", c_int32)]


_lib = None
_host = None
_device_checked = False


def _declare(lib):
    lib.mi_version.restype = c_int
    lib.mi_last_error.restype = c_char_p
    lib.mi_status_string.restype = c_char_p
    lib.mi_status_string.argtypes = [c_int]
    lib.mi_check_device.restype = c_int
    lib.mi_rmsnorm_fwd.restype = c_int
    lib.mi_rmsnorm_fwd.argtypes = [c_void_p, c_void_p, c_void_p, c_void_p, c_int64, c_int64, c_float, c_int, c_void_p]
    lib.mi_rmsnorm_bwd_workspace_bytes.restype = c_size_t
    lib.mi_add_rmsnorm_fwd.restype = c_int
    lib.mi_add_rmsnorm_fwd.argtypes = [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int64, c_int64, c_float, c_int, c_void_p]
    lib.mi_rmsnorm_bwd_workspace_bytes.argtypes = [c_int64, c_int64]
    lib.mi_rmsnorm_bwd.restype = c_int
    lib.mi_rmsnorm_bwd.argtypes = [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_size_t, c_int64,
                                   c_int64, c_float, c_int, c_void_p]
    lib.mi_layernorm_fwd.restype = c_int
    lib.mi_layernorm_fwd.argtypes = [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int64, c_int64, c_float,
                                     c_int, c_void_p]
    lib.mi_layernorm_bwd_workspace_bytes.restype = c_size_t
    lib.mi_layernorm_bwd_workspace_bytes.argtypes = [c_int64, c_int64]
    lib.mi_layernorm_bwd.restype = c_int
    lib.mi_layernorm_bwd.argtypes = [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p,
                                     c_void_p, c_size_t, c_int64, c_int64, c_float, c_int, c_void_p]
    lib.mi_gelu_fwd.restype = c_int
    lib.mi_gelu_fwd.argtypes = [c_void_p, c_void_p, c_int64, c_int, c_void_p]
    lib.mi_gelu_bwd.restype = c_int
    lib.mi_gelu_bwd.argtypes = [c_void_p, c_void_p, c_void_p, c_int64, c_int, c_void_p]
    lib.mi_cross_entropy.restype = c_int
    lib.mi_cross_entropy.argtypes = [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int64, c_int64,
                                     c_int64, c_int64, c_int, c_void_p]
    lib.mi_cross_entropy_padded.restype = c_int
    lib.mi_cross_entropy_padded.argtypes = [c_void_p] * 6 + [c_int64, c_int64, c_int64, c_int, c_void_p]
    lib.mi_cross_entropy_mean_grad.restype = c_int
    lib.mi_cross_entropy_mean_grad.argtypes = [c_void_p] * 7 + [c_int64, c_int64, c_int64, c_int64, c_int, c_void_p]
    lib.mi_rotary_two.restype = c_int
    lib.mi_rotary_two.argtypes = [POINTER(MiRotaryRows), c_void_p, c_void_p, c_void_p, c_int64, c_int32, c_int32, c_int64, c_int64, c_int, c_int, c_int, c_int,
                                  c_void_p]
    lib.mi_argmax.restype = c_int
    lib.mi_argmax.argtypes = [c_void_p, c_int64, c_int64, c_int64, c_void_p, c_int, c_void_p]
    lib.mi_argmax_embed.restype = c_int
    lib.mi_argmax_embed.argtypes = [c_void_p, c_int64, c_int64, c_int64, c_void_p, c_void_p, c_int64, c_int64, c_int64, c_void_p, c_int, c_void_p]
    lib.mi_loss_reduce.restype = c_int
    lib.mi_loss_reduce.argtypes = [c_void_p] * 4 + [c_int64, c_void_p, c_void_p, c_void_p, c_void_p]
    lib.mi_loss_row_scale.restype = c_int
    lib.mi_loss_row_scale.argtypes = [c_void_p, c_int64, c_void_p, c_void_p]
    lib.mi_scale_inplace.restype = c_int
    lib.mi_scale_inplace.argtypes = [c_void_p, c_int64, c_void_p, c_int, c_void_p]
    lib.mi_swiglu_fwd.restype = c_int
    lib.mi_swiglu_fwd.argtypes = [c_void_p, c_void_p, c_void_p, c_int64, c_int, c_void_p]
    lib.mi_swiglu_bwd.restype = c_int
    lib.mi_swiglu_bwd.argtypes = [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int64, c_int, c_void_p]
    lib.mi_rotary.restype = c_int
    lib.mi_rotary.argtypes = [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int64, c_int32, c_int32, c_int32,
                              c_int64, c_int64, c_int64, c_int64, c_int64, c_int64, c_int, c_int, c_int, c_void_p]
    lib.mi_rotary_complex.restype = c_int
    lib.mi_rotary_complex.argtypes = [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int64, c_int32, c_int32,
                                      c_int64, c_int64, c_int64, c_int64, c_int64, c_int64, c_int, c_int, c_void_p]
    lib.mi_gemm.restype = c_int
    lib.mi_gemm.argtypes = [POINTER(MiGemmProblem), c_int, c_int, c_void_p]
    lib.mi_gemm_workspace_bytes.restype = c_size_t
    lib.mi_gemm_workspace_bytes.argtypes = [POINTER(MiGemmProblem), c_int, c_int]
    lib.mi_gemm_with_workspace.restype = c_int
    lib.mi_gemm_with_workspace.argtypes = [POINTER(MiGemmProblem), c_int, c_int, c_void_p, c_size_t, c_void_p]
    lib.mi_rows_product.restype = c_int
    lib.mi_rows_product.argtypes = [POINTER(MiRowsArgs)]
    lib.mi_transpose16.restype = c_int
    lib.mi_transpose16.argtypes = [c_void_p, c_int64, c_int64, c_int64, c_void_p, c_int64, c_void_p]
    lib.mi_column_sum.restype = c_int
    lib.mi_column_sum.argtypes = [c_void_p, c_int64, c_int64, c_int64, c_void_p, c_int, c_void_p]
    lib.mi_add_rmsnorm_bwd.restype = c_int
    lib.mi_add_rmsnorm_bwd.argtypes = [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_size_t, c_int64,
                                       c_int64, c_float, c_int, c_void_p]
    lib.mi_add_layernorm_fwd.restype = c_int
    lib.mi_add_layernorm_fwd.argtypes = [c_void_p] * 8 + [c_int64, c_int64, c_float, c_int, c_void_p]
    lib.mi_add_layernorm_bwd.restype = c_int
    lib.mi_add_layernorm_bwd.argtypes = [c_void_p] * 10 + [c_size_t, c_int64, c_int64, c_float, c_int, c_void_p]
    lib.mi_attn_fwd.restype = c_int
    lib.mi_attn_fwd.argtypes = [POINTER(MiAttnArgs)]
    lib.mi_attn_bwd_workspace_bytes.restype = c_size_t
    lib.mi_attn_bwd_workspace_bytes.argtypes = [c_int64, c_int32, c_int32]
    lib.mi_attn_bwd_workspace_bytes_for.restype = c_size_t
    lib.mi_attn_bwd_workspace_bytes_for.argtypes = [POINTER(MiAttnArgs)]
    lib.mi_attn_bwd_workspace_bytes_kv.restype = c_size_t
    lib.mi_attn_bwd_workspace_bytes_kv.argtypes = [c_int64, c_int64, c_int32, c_int32, c_int32]
    lib.mi_attn_bwd.restype = c_int
    lib.mi_attn_bwd.argtypes = [POINTER(MiAttnBwdArgs)]
    lib.mi_attn_decode_workspace_bytes.restype = c_size_t
    lib.mi_attn_decode_workspace_bytes.argtypes = [c_int32, c_int32, c_int32, c_int32]
    lib.mi_attn_decode.restype = c_int
    lib.mi_attn_decode.argtypes = [POINTER(MiDecodeArgs)]
    lib.mi_attn_decode_with_tickets.restype = c_int
    lib.mi_attn_decode_with_tickets.argtypes = [POINTER(MiDecodeArgs), c_void_p, c_int64]
    lib.mi_attn_decode_static_scratch_bytes.restype = c_size_t
    lib.mi_attn_decode_static_scratch_bytes.argtypes = []
    lib.mi_attn_decode_static.restype = c_int
    lib.mi_attn_decode_static.argtypes = [POINTER(MiDecodeArgs)]


def load(path: str = LIB_PATH):
    """Returns the loaded library; raises if it has not been built."""
    global _lib
    if _lib is None:
        if not os.path.exists(path):
            raise RuntimeError(
                f"{path} is missing: the HIP extension has not been built "
                "(run `python -m scaling_amd.csrc.build`); there is no fallback path"
            )
        lib = ctypes.CDLL(path)
        _declare(lib)
        _lib = lib
    return _lib


def host():
    """Returns the native host module; raises if it has not been built."""
    global _host
    if _host is None:
        load()                           # the module links against it
        if not os.path.exists(HOST_PATH):
            raise RuntimeError(f"{HOST_PATH} is missing: the host extension has not been built "
                               "(run `python -m scaling_amd.csrc.build`); there is no fallback path")
        spec = importlib.util.spec_from_file_location("mi355_host", HOST_PATH)
        module = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(module)
        _host = module
    return _host


def check(status: int, what: str) -> None:
    if status != 0:
        lib = load()
        raise RuntimeError(
            f"{what} failed: {lib.mi_status_string(status).decode()} ({status}): {lib.mi_last_error().decode()}"
        )


def require_device() -> None:
    """Raises unless the current device is a gfx950 GPU (checked once per process)."""
    global _device_checked
    if _device_checked:
        return
    if not torch.cuda.is_available():
        raise RuntimeError("scaling_amd kernels need an MI355X (gfx950) GPU; no HIP device is visible")
    check(load().mi_check_device(), "mi_check_device")
    _device_checked = True


def dtype_code(dtype: torch.dtype) -> int:
    try:
        return _DTYPE_CODE[dtype]
    except KeyError:
        raise TypeError(f"dtype {dtype} is not supported by the HIP kernels") from None


def stream_ptr() -> int:
    return torch.cuda.current_stream().cuda_stream


def ptr(t):
    return None if t is None else t.data_ptr()
