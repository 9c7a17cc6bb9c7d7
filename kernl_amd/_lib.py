"""Binding of libkernl_hip.so (C ABI: include/kernl_hip.h): ctypes, and for the calls made per token or per layer the
CPython module `_host` (csrc/host_ops.cpp), which costs 2 us a call where ctypes and its conversions cost 10.

Both are built in-tree by `kernl_amd/csrc/Makefile` (see `kernl_amd.build`).  There is no fallback:
if a shared object is missing or a call fails, the error is raised to the caller.
"""
import ctypes
import importlib
import os
from typing import Optional, Sequence

import torch

_LIB_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "libkernl_hip.so")
_lib: Optional[ctypes.CDLL] = None
_host = None

KERNL_F16, KERNL_BF16, KERNL_F32 = 0, 1, 2
DTYPE_CODE = {torch.float16: KERNL_F16, torch.bfloat16: KERNL_BF16, torch.float32: KERNL_F32}

ACT_NONE, ACT_RELU, ACT_TANH, ACT_GELU_ERF, ACT_GELU_TANH, ACT_SILU = range(6)

# every symbol declared in include/kernl_hip.h
EXPORTED_SYMBOLS = (
    "kernl_version",
    "kernl_last_error_string",
    "kernl_attention_fwd",
    "kernl_attention_cached_fwd",
    "kernl_attention_skinny_workspace_bytes",
    "kernl_attention_skinny_fwd",
    "kernl_attention_skinny_kv8_fwd",
    "kernl_attention_kv8_fwd",
    "kernl_attention_skinny_static_max_bytes",
    "kernl_attention_skinny_static_init",
    "kernl_attention_skinny_static_fwd",
    "kernl_rope_fwd",
    "kernl_rope_tables",
    "kernl_linear_fwd",
    "kernl_linear_small_kind",
    "kernl_linear_w8_fwd",
    "kernl_linear_rms_fwd",
    "kernl_linear_scaled_fwd",
    "kernl_linear_residual_fwd",
    "kernl_linear_wide_kind",
    "kernl_linear_mid_kind",
    "kernl_linear_norm_kind",
    "kernl_linear_norm_add_fwd",
    "kernl_linear_norm_apply_fwd",
    "kernl_layernorm_rows32_fwd",
    "kernl_embedding_layernorm_fwd",
    "kernl_copy_many",
    "kernl_select_mask_fwd",
    "kernl_linear_decode_fwd",
    "kernl_linear_splitk_workspace_bytes",
    "kernl_linear_splitk_fwd",
    "kernl_linear_split_workspace_bytes",
    "kernl_linear_split_fwd",
    "kernl_linear_exchange_bytes",
    "kernl_linear_add_norm_fwd",
    "kernl_linear_fewrow_workspace_bytes",
    "kernl_linear_fewrow_fwd",
    "kernl_linear_fewrow_w8_fwd",
    "kernl_linear_glu_fwd",
    "kernl_layernorm_fwd",
    "kernl_add_layernorm_fwd",
    "kernl_add_rms_stats_fwd",
)

# the process-wide test and tuning hooks of include/kernl_hip_test.h (bound for the tests and benchmarks only)
TEST_HOOK_SYMBOLS = (
    "kernl_linear_force_tile",
    "kernl_attention_force_scalar",
    "kernl_attention_set_variant",
    "kernl_probe_rate",
)

_i64 = ctypes.c_int64
_vp = ctypes.c_void_p
_i64p = ctypes.POINTER(ctypes.c_int64)


class KernlLibraryError(RuntimeError):
    pass


def lib_path() -> str:
    return _LIB_PATH


def load() -> ctypes.CDLL:
    """Load (once) and return the shared library; raises KernlLibraryError if it has not been built."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(_LIB_PATH):
        raise KernlLibraryError(
            f"{_LIB_PATH} not found: build it with `python -m kernl_amd.build` (needs hipcc, targets gfx950)"
        )
    lib = ctypes.CDLL(_LIB_PATH)
    lib.kernl_version.restype = ctypes.c_int
    lib.kernl_version.argtypes = []
    lib.kernl_last_error_string.restype = ctypes.c_char_p
    lib.kernl_last_error_string.argtypes = []
    lib.kernl_attention_fwd.restype = ctypes.c_int
    lib.kernl_attention_fwd.argtypes = (
        [_vp] * 5 + [_i64] * 5 + [_i64p] * 6 + [ctypes.c_int, ctypes.c_float, ctypes.c_int, ctypes.c_float, ctypes.c_int, _vp]
    )
    lib.kernl_attention_cached_fwd.restype = ctypes.c_int
    lib.kernl_attention_cached_fwd.argtypes = (
        [_vp] * 5 + [_i64] * 5 + [_i64p] * 6 + [ctypes.c_int, ctypes.c_float, _i64, ctypes.c_float, ctypes.c_int, _vp]
    )
    lib.kernl_attention_kv8_fwd.restype = ctypes.c_int
    lib.kernl_attention_kv8_fwd.argtypes = (
        [_vp] * 5 + [_i64] * 5 + [_i64p] * 6
        + [ctypes.c_int, ctypes.c_float, ctypes.c_int, _i64, ctypes.c_float, ctypes.c_int, _vp]
    )
    lib.kernl_attention_skinny_workspace_bytes.restype = _i64
    lib.kernl_attention_skinny_workspace_bytes.argtypes = [_i64] * 5
    lib.kernl_attention_skinny_fwd.restype = ctypes.c_int
    lib.kernl_attention_skinny_fwd.argtypes = (
        [_vp] * 6 + [_i64] * 6 + [_i64p] * 6 + [ctypes.c_int, ctypes.c_float, ctypes.c_int, ctypes.c_float, ctypes.c_int, _vp]
    )
    lib.kernl_attention_skinny_kv8_fwd.restype = ctypes.c_int
    lib.kernl_attention_skinny_kv8_fwd.argtypes = (
        [_vp] * 6 + [_i64] * 6 + [_i64p] * 6 + [ctypes.c_int, ctypes.c_float, ctypes.c_int, ctypes.c_float, ctypes.c_int, _vp]
    )
    lib.kernl_attention_skinny_static_max_bytes.restype = _i64
    lib.kernl_attention_skinny_static_max_bytes.argtypes = []
    lib.kernl_attention_skinny_static_init.restype = ctypes.c_int
    lib.kernl_attention_skinny_static_init.argtypes = []
    lib.kernl_attention_skinny_static_fwd.restype = ctypes.c_int
    lib.kernl_attention_skinny_static_fwd.argtypes = (
        [_vp] * 5 + [_i64] * 5 + [_i64p] * 6 + [ctypes.c_int, ctypes.c_float, ctypes.c_int, ctypes.c_float, ctypes.c_int, _vp]
    )
    lib.kernl_rope_tables.restype = ctypes.c_int
    lib.kernl_rope_tables.argtypes = [_vp] * 4 + [_i64] * 3 + [_i64p] * 2 + [ctypes.c_int, ctypes.c_int, ctypes.c_float, ctypes.c_int, _vp]
    lib.kernl_rope_fwd.restype = ctypes.c_int
    lib.kernl_rope_fwd.argtypes = [_vp] * 4 + [_i64] * 4 + [_i64p] * 5 + [ctypes.c_int, ctypes.c_int, _vp]
    lib.kernl_linear_fwd.restype = ctypes.c_int
    lib.kernl_linear_fwd.argtypes = [_vp] * 5 + [_i64] * 3 + [_i64p] * 3 + [ctypes.c_int, ctypes.c_int, _vp]
    lib.kernl_linear_w8_fwd.restype = ctypes.c_int
    lib.kernl_linear_w8_fwd.argtypes = [_vp] * 5 + [_i64] * 3 + [_i64p] * 3 + [ctypes.c_int, ctypes.c_int, _vp]
    lib.kernl_linear_decode_fwd.restype = ctypes.c_int
    lib.kernl_linear_decode_fwd.argtypes = (
        [_vp, _vp, ctypes.c_float, _vp, _vp, _vp, _vp] + [_i64] * 3 + [_i64p] * 3 + [_vp, _vp] + [_i64] * 3
        + [_i64p, ctypes.c_int, ctypes.c_int, _vp]
    )
    lib.kernl_linear_splitk_workspace_bytes.restype = _i64
    lib.kernl_linear_splitk_workspace_bytes.argtypes = [_i64] * 3
    lib.kernl_linear_split_workspace_bytes.restype = _i64
    lib.kernl_linear_split_workspace_bytes.argtypes = [_i64] * 3 + [ctypes.c_int]
    lib.kernl_linear_split_fwd.restype = ctypes.c_int
    lib.kernl_linear_split_fwd.argtypes = [_vp] * 6 + [ctypes.c_float] + [_vp] * 3 + [_i64] * 7 + [ctypes.c_int, ctypes.c_int, _vp]
    lib.kernl_linear_exchange_bytes.restype = _i64
    lib.kernl_linear_exchange_bytes.argtypes = [_i64] * 3
    lib.kernl_linear_add_norm_fwd.restype = ctypes.c_int
    lib.kernl_linear_add_norm_fwd.argtypes = [_vp] * 6 + [ctypes.c_float] + [_vp] * 4 + [_i64, ctypes.c_int] + [_i64] * 6 + [ctypes.c_int, _vp]
    lib.kernl_linear_splitk_fwd.restype = ctypes.c_int
    lib.kernl_linear_splitk_fwd.argtypes = [_vp] * 6 + [_i64] * 4 + [_i64p] * 3 + [ctypes.c_int, ctypes.c_int, _vp]
    lib.kernl_linear_fewrow_workspace_bytes.restype = _i64
    lib.kernl_linear_fewrow_workspace_bytes.argtypes = [_i64] * 3 + [ctypes.c_int] * 2
    lib.kernl_linear_fewrow_fwd.restype = ctypes.c_int
    lib.kernl_linear_fewrow_fwd.argtypes = (
        [_vp, _vp, ctypes.c_float] + [_vp] * 5 + [_i64] * 4 + [_i64p] * 3 + [_vp, _vp] + [_i64] * 3
        + [_i64p] + [ctypes.c_int] * 4 + [_vp]
    )
    lib.kernl_linear_fewrow_w8_fwd.restype = ctypes.c_int
    lib.kernl_linear_fewrow_w8_fwd.argtypes = lib.kernl_linear_fewrow_fwd.argtypes
    lib.kernl_linear_rms_fwd.restype = ctypes.c_int
    lib.kernl_linear_rms_fwd.argtypes = (
        [_vp, _vp, ctypes.c_float, _vp, _vp, _vp] + [_i64] * 3 + [_i64p] * 2 + [ctypes.c_int] * 3 + [_vp]
    )
    lib.kernl_linear_scaled_fwd.restype = ctypes.c_int
    lib.kernl_linear_scaled_fwd.argtypes = [_vp] * 5 + [_i64] * 3 + [_i64p] * 2 + [ctypes.c_int] * 3 + [_vp]
    lib.kernl_linear_residual_fwd.restype = ctypes.c_int
    lib.kernl_linear_residual_fwd.argtypes = [_vp] * 5 + [_i64] * 3 + [_i64p] * 3 + [ctypes.c_int, _vp]
    lib.kernl_embedding_layernorm_fwd.restype = ctypes.c_int
    lib.kernl_embedding_layernorm_fwd.argtypes = [_vp, _vp, _i64, _i64, _i64] * 3 + [_vp, _vp, _vp, _i64, _i64, _i64,
                                                                                      ctypes.c_float, ctypes.c_int, _vp]
    lib.kernl_copy_many.restype = ctypes.c_int
    lib.kernl_copy_many.argtypes = [ctypes.c_int, ctypes.POINTER(_vp), ctypes.POINTER(_vp), _i64p, _vp]
    lib.kernl_select_mask_fwd.restype = ctypes.c_int
    lib.kernl_select_mask_fwd.argtypes = [_vp, ctypes.c_int, ctypes.c_float, ctypes.c_float, _vp, _i64, ctypes.c_int, _vp]
    lib.kernl_add_rms_stats_fwd.restype = ctypes.c_int
    lib.kernl_add_rms_stats_fwd.argtypes = [_vp] * 4 + [_i64] * 5 + [ctypes.c_float, ctypes.c_int, _vp]
    lib.kernl_linear_small_kind.restype = ctypes.c_int
    lib.kernl_linear_small_kind.argtypes = [_i64] * 3
    lib.kernl_linear_wide_kind.restype = ctypes.c_int
    lib.kernl_linear_wide_kind.argtypes = [_i64] * 3
    lib.kernl_linear_mid_kind.restype = ctypes.c_int
    lib.kernl_linear_mid_kind.argtypes = [_i64] * 3 + [ctypes.c_int]
    lib.kernl_linear_norm_kind.restype = ctypes.c_int
    lib.kernl_linear_norm_kind.argtypes = [_i64] * 3
    lib.kernl_linear_norm_add_fwd.restype = ctypes.c_int
    lib.kernl_linear_norm_add_fwd.argtypes = [_vp] * 7 + [ctypes.c_float, _vp, _vp] + [_i64] * 6 + [ctypes.c_int, _vp]
    lib.kernl_linear_norm_apply_fwd.restype = ctypes.c_int
    lib.kernl_linear_norm_apply_fwd.argtypes = [_vp] * 4 + [ctypes.c_float] + [_vp] * 3 + [_i64] * 5 + [ctypes.c_int, ctypes.c_int, _vp]
    lib.kernl_layernorm_rows32_fwd.restype = ctypes.c_int
    lib.kernl_layernorm_rows32_fwd.argtypes = [_vp] * 4 + [_i64] * 4 + [ctypes.c_float, ctypes.c_int, _vp]
    lib.kernl_linear_glu_fwd.restype = ctypes.c_int
    lib.kernl_linear_glu_fwd.argtypes = [_vp] * 4 + [_i64] * 3 + [_i64p] * 2 + [ctypes.c_int, ctypes.c_int, _vp]
    lib.kernl_layernorm_fwd.restype = ctypes.c_int
    lib.kernl_layernorm_fwd.argtypes = [_vp] * 6 + [_i64] * 6 + [ctypes.c_float, ctypes.c_int, ctypes.c_int, _vp]
    lib.kernl_add_layernorm_fwd.restype = ctypes.c_int
    lib.kernl_add_layernorm_fwd.argtypes = [_vp] * 7 + [_i64] * 8 + [ctypes.c_float, ctypes.c_int, ctypes.c_int, _vp]
    lib.kernl_linear_force_tile.restype = None
    lib.kernl_linear_force_tile.argtypes = [ctypes.c_int]
    lib.kernl_attention_force_scalar.restype = None
    lib.kernl_attention_force_scalar.argtypes = [ctypes.c_int]
    lib.kernl_attention_set_variant.restype = None
    lib.kernl_attention_set_variant.argtypes = [ctypes.c_int]
    lib.kernl_probe_rate.restype = ctypes.c_int
    lib.kernl_probe_rate.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_int, _vp, _vp, _i64, _vp, _vp, _vp]
    _lib = lib
    return lib


def host():
    """The CPython module over the library, loaded once; raises KernlLibraryError if it has not been built."""
    global _host
    if _host is None:
        load()
        try:
            module = importlib.import_module("kernl_amd._host")
        except ImportError as exc:
            raise KernlLibraryError(f"kernl_amd/_host.so cannot be loaded ({exc}): build it with `python -m kernl_amd.build`") from exc
        module.set_error_type(KernlLibraryError)
        _host = module
    return _host


def _arr(values: Sequence[int]):
    return (ctypes.c_int64 * len(values))(*values)


def _check(status: int, what: str) -> None:
    if status != 0:
        msg = load().kernl_last_error_string().decode("utf-8", "replace")
        raise KernlLibraryError(f"{what} failed with status {status}: {msg}")


def _stream(t: torch.Tensor) -> int:
    return torch.cuda.current_stream(t.device).cuda_stream


def _require_gpu(*tensors: torch.Tensor) -> None:
    for t in tensors:
        if t is not None and not t.is_cuda:
            raise KernlLibraryError("kernl_amd kernels need tensors on a GPU device (there is no CPU path)")


def attention_fwd(q, k, v, out, mask, sm_scale: float, is_causal: bool, mask_min_clamp: float) -> None:
    (_host or host()).attention_fwd(q, k, v, out, mask, sm_scale, is_causal, mask_min_clamp)


def attention_cached_fwd(q, k, v, out, mask, sm_scale: float, start_position: int, mask_min_clamp: float) -> None:
    """Causal attention of the rows of q, which sit at positions start_position.. of the sequence held in k / v."""
    (_host or host()).attention_cached_fwd(q, k, v, out, mask, sm_scale, start_position, mask_min_clamp)


def attention_kv8_fwd(q, k8, v8, out, mask, sm_scale: float, is_causal: bool, start_position: int, mask_min_clamp: float) -> None:
    """k8, v8 [B, H, N, D]: fp8 e5m2 bytes (int8 / uint8 / float8_e5m2); q and out fp16."""
    _require_gpu(q, k8, v8, out, mask)
    B, H, M, D = q.shape
    N = k8.shape[2]
    lib = load()
    if mask is not None:
        msizes, mstrides, mdtype, mptr = _arr(mask.shape), _arr(mask.stride()), DTYPE_CODE[mask.dtype], mask.data_ptr()
    else:
        msizes, mstrides, mdtype, mptr = None, None, KERNL_F32, None
    with torch.cuda.device(q.device):
        st = lib.kernl_attention_kv8_fwd(
            q.data_ptr(), k8.data_ptr(), v8.data_ptr(), out.data_ptr(), mptr,
            B, H, M, N, D,
            _arr(q.stride()), _arr(k8.stride()), _arr(v8.stride()), _arr(out.stride()),
            msizes, mstrides, mdtype,
            float(sm_scale), int(bool(is_causal)), int(start_position), float(mask_min_clamp), DTYPE_CODE[q.dtype], _stream(q),
        )
    _check(st, "kernl_attention_kv8_fwd")


def attention_skinny_workspace_bytes(B: int, H: int, M: int, N: int, D: int) -> int:
    return int(load().kernl_attention_skinny_workspace_bytes(B, H, M, N, D))


def attention_skinny_fwd(q, k, v, out, mask, workspace, sm_scale: float, is_causal: bool, mask_min_clamp: float) -> None:
    (_host or host()).attention_skinny_fwd(q, k, v, out, mask, workspace, sm_scale, is_causal, mask_min_clamp)


def attention_skinny_static_init(device=None) -> None:
    """Look up the static partial-result buffer of `device` (default: the current one): to be called outside graph
    capture before `attention_skinny_static_fwd` is captured for the first time on that device."""
    lib = load()
    with torch.cuda.device(device):
        st = lib.kernl_attention_skinny_static_init()
    _check(st, "kernl_attention_skinny_static_init")


def attention_skinny_static_fwd(q, k, v, out, mask, sm_scale: float, is_causal: bool, mask_min_clamp: float) -> None:
    """`attention_skinny_fwd` on the library's own static partial-result buffer: no workspace, no allocation."""
    _require_gpu(q, k, v, out, mask)
    B, H, M, D = q.shape
    N = k.shape[2]
    lib = load()
    if mask is not None:
        msizes, mstrides, mdtype, mptr = _arr(mask.shape), _arr(mask.stride()), DTYPE_CODE[mask.dtype], mask.data_ptr()
    else:
        msizes, mstrides, mdtype, mptr = None, None, KERNL_F32, None
    with torch.cuda.device(q.device):
        st = lib.kernl_attention_skinny_static_fwd(
            q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), mptr,
            B, H, M, N, D,
            _arr(q.stride()), _arr(k.stride()), _arr(v.stride()), _arr(out.stride()),
            msizes, mstrides, mdtype,
            float(sm_scale), int(bool(is_causal)), float(mask_min_clamp), DTYPE_CODE[q.dtype], _stream(q),
        )
    _check(st, "kernl_attention_skinny_static_fwd")


def rope_fwd(x, cos, sin, out) -> None:
    """x, out [B,H,S,D]; cos, sin [B|1,H|1,S,D] of the same dtype as each other."""
    _require_gpu(x, cos, sin, out)
    B, H, S, D = x.shape
    lib = load()
    with torch.cuda.device(x.device):
        st = lib.kernl_rope_fwd(
            x.data_ptr(), cos.data_ptr(), sin.data_ptr(), out.data_ptr(), B, H, S, D,
            _arr(x.stride()), _arr(out.stride()), _arr(cos.shape), _arr(cos.stride()), _arr(sin.stride()),
            DTYPE_CODE[cos.dtype], DTYPE_CODE[x.dtype], _stream(x),
        )
    _check(st, "kernl_rope_fwd")


def rope_tables(inv_freq, positions, cos, sin, scale: float) -> None:
    """inv_freq [B|1,half,1], positions [B|1,1,S] (int64 or float32); cos, sin [B,S,2*half] contiguous, of the same dtype as each other."""
    _require_gpu(inv_freq, positions, cos, sin)
    B, S, D = cos.shape
    lib = load()
    fs = _arr((0 if inv_freq.shape[0] == 1 else inv_freq.stride(0), inv_freq.stride(1)))
    ps = _arr((0 if positions.shape[0] == 1 else positions.stride(0), positions.stride(2)))
    with torch.cuda.device(cos.device):
        st = lib.kernl_rope_tables(
            inv_freq.data_ptr(), positions.data_ptr(), cos.data_ptr(), sin.data_ptr(), B, S, D // 2, fs, ps,
            DTYPE_CODE[inv_freq.dtype], int(positions.dtype == torch.int64), float(scale), DTYPE_CODE[cos.dtype], _stream(cos),
        )
    _check(st, "kernl_rope_tables")


def linear_small_kind(M: int, N: int, K: int) -> int:
    """Non-zero when `kernl_linear_fwd` runs an M x N x K problem on one of its small-problem kernels."""
    return int(load().kernl_linear_small_kind(int(M), int(N), int(K)))


def linear_mid_kind(M: int, N: int, K: int, gated: bool = False) -> int:
    """Non-zero when `kernl_linear_fwd` (`kernl_linear_glu_fwd`) runs the problem on one of its middling tiles: such shapes are not
    handed to the stream-K or split-K entry points."""
    return int(load().kernl_linear_mid_kind(int(M), int(N), int(K), int(bool(gated))))


def linear_wide_kind(M: int, N: int, K: int) -> int:
    """Non-zero when `kernl_linear_fwd` runs a plain 16-bit M x N x K problem on one of its wide tile kernels."""
    return int(load().kernl_linear_wide_kind(int(M), int(N), int(K)))


def linear_fwd(x2d, weight, bias, out2d, act_in2d, activation: int) -> None:
    (_host or host()).linear_fwd(x2d, weight, bias, out2d, act_in2d, activation)


def linear_norm_kind(M: int, N: int, K: int) -> int:
    """Non-zero when both deferred-norm entry points take an M x N x K problem."""
    return int(load().kernl_linear_norm_kind(int(M), int(N), int(K)))


NORM_GROUP = 16  # columns per statistics pair of a deferred norm


def _norm_checks(x2d, weight, out2d, statistics, parameters, width: int) -> None:
    """Layouts of the deferred-norm entry points: what their pointers are taken to mean."""
    if any(t is not None and (t.dtype != torch.float32 or t.numel() != x2d.shape[0] * width // NORM_GROUP * 2 or not t.is_contiguous()) for t in statistics):
        raise ValueError("statistics are contiguous fp32 [rows, columns / 16, 2]")
    if any(p is not None and (p.dtype != weight.dtype or p.shape != (n,) or not p.is_contiguous()) for p, n in parameters):
        raise ValueError("bias and norm parameters are contiguous vectors of the weight's type")
    if x2d.stride(1) != 1 or out2d.stride(1) != 1 or not weight.is_contiguous() or x2d.shape[1] != weight.shape[1] or out2d.shape != (x2d.shape[0], weight.shape[0]):
        raise ValueError("unit feature strides, a contiguous weight and matching sizes")


def linear_norm_add_fwd(x2d, weight, bias, residual2d, residual_stats, gamma, beta, eps: float, out2d, out_stats) -> None:
    """out = x @ w^T + bias + residual in fp32 with the statistics of its rows; with `residual_stats` the residual is the fp32
    rows of a deferred LayerNorm (gamma, beta, eps)."""
    _require_gpu(x2d, weight, bias, residual2d, residual_stats, gamma, beta, out2d, out_stats)
    M, K = x2d.shape
    N = weight.shape[0]
    _norm_checks(x2d, weight, out2d, (residual_stats, out_stats), ((bias, N), (gamma, N), (beta, N)), N)
    if out2d.dtype != torch.float32 or residual2d.dtype != (weight.dtype if residual_stats is None else torch.float32) or residual2d.shape != (M, N) \
            or residual2d.stride(1) != 1 or x2d.dtype != weight.dtype:
        raise ValueError("fp32 rows out, a residual of x's type (fp32 rows where it has statistics)")
    with torch.cuda.device(x2d.device):
        st = load().kernl_linear_norm_add_fwd(
            x2d.data_ptr(), weight.data_ptr(), None if bias is None else bias.data_ptr(), residual2d.data_ptr(),
            None if residual_stats is None else residual_stats.data_ptr(), None if gamma is None else gamma.data_ptr(),
            None if beta is None else beta.data_ptr(), float(eps), out2d.data_ptr(), out_stats.data_ptr(), M, N, K, x2d.stride(0),
            out2d.stride(0), residual2d.stride(0), DTYPE_CODE[weight.dtype], _stream(x2d),
        )
    _check(st, "kernl_linear_norm_add_fwd")


def linear_norm_apply_fwd(x2d, x_stats, gamma, beta, eps: float, weight, bias, out2d, activation: int) -> None:
    """out = act(LN(x) @ w^T + bias) of fp32 rows x with their statistics, LN(x) rounded to the weight's type."""
    _require_gpu(x2d, x_stats, gamma, beta, weight, bias, out2d)
    M, K = x2d.shape
    N = weight.shape[0]
    _norm_checks(x2d, weight, out2d, (x_stats,), ((bias, N), (gamma, K), (beta, K)), K)
    if x2d.dtype != torch.float32 or out2d.dtype != weight.dtype:
        raise ValueError("fp32 rows in, rows of the weight's type out")
    with torch.cuda.device(x2d.device):
        st = load().kernl_linear_norm_apply_fwd(
            x2d.data_ptr(), x_stats.data_ptr(), gamma.data_ptr(), None if beta is None else beta.data_ptr(), float(eps), weight.data_ptr(),
            None if bias is None else bias.data_ptr(), out2d.data_ptr(), M, N, K, x2d.stride(0), out2d.stride(0), int(activation),
            DTYPE_CODE[weight.dtype], _stream(x2d),
        )
    _check(st, "kernl_linear_norm_apply_fwd")


def layernorm_rows32_fwd(x2d, weight, bias, out2d, eps: float) -> None:
    """out = LN(x) of fp32 rows x in the weight's 16-bit type."""
    _require_gpu(x2d, weight, bias, out2d)
    M, N = x2d.shape
    if x2d.dtype != torch.float32 or out2d.dtype != weight.dtype or out2d.shape != x2d.shape or x2d.stride(1) != 1 or out2d.stride(1) != 1 \
            or any(p is not None and (p.dtype != weight.dtype or p.shape != (N,) or not p.is_contiguous()) for p in (weight, bias)):
        raise ValueError("fp32 rows in, rows of the weight's type out, contiguous parameters")
    with torch.cuda.device(x2d.device):
        st = load().kernl_layernorm_rows32_fwd(x2d.data_ptr(), weight.data_ptr(), None if bias is None else bias.data_ptr(), out2d.data_ptr(), M, N,
                                               x2d.stride(0), out2d.stride(0), float(eps), DTYPE_CODE[weight.dtype], _stream(x2d))
    _check(st, "kernl_layernorm_rows32_fwd")


def linear_w8_supported(x2d, weight8) -> bool:
    """What `kernl_linear_w8_fwd` takes: fp16 rows with unit feature stride, 16-byte aligned, K a multiple of 8."""
    M, K = x2d.shape
    return (
        x2d.dtype == torch.float16 and K % 8 == 0 and K < (1 << 22) and x2d.stride(1) == 1 and x2d.stride(0) % 8 == 0
        and x2d.stride(0) < (1 << 22)
        and x2d.data_ptr() % 16 == 0 and weight8.is_contiguous() and weight8.data_ptr() % 16 == 0
    )


def linear_w8_fwd(x2d, weight8, bias, out2d, act_in2d, activation: int) -> None:
    """weight8 [N, K]: fp8 e5m2 bytes (int8 / uint8 / float8_e5m2)."""
    _require_gpu(x2d, weight8, bias, out2d, act_in2d)
    M, K = x2d.shape
    N = weight8.shape[0]
    lib = load()
    with torch.cuda.device(x2d.device):
        st = lib.kernl_linear_w8_fwd(
            x2d.data_ptr(), weight8.data_ptr(), None if bias is None else bias.data_ptr(), out2d.data_ptr(),
            None if act_in2d is None else act_in2d.data_ptr(),
            M, N, K,
            _arr(x2d.stride()), _arr(out2d.stride()), None if act_in2d is None else _arr(act_in2d.stride()),
            int(activation), DTYPE_CODE[x2d.dtype], _stream(x2d),
        )
    _check(st, "kernl_linear_w8_fwd")


def linear_rms_supported(x2d) -> bool:
    """What `kernl_linear_rms_fwd` takes: 16-bit rows, at most 64 of them, K a multiple of 64."""
    M, K = x2d.shape
    return (
        x2d.dtype in (torch.float16, torch.bfloat16) and M <= 64 and K % 64 == 0 and x2d.stride(1) == 1
        and x2d.stride(0) % 8 == 0 and x2d.data_ptr() % 16 == 0
    )


def linear_rms_fwd(x2d, rms_weight, eps: float, weight, bias, out2d, activation: int, gated: bool) -> None:
    (_host or host()).linear_rms_fwd(x2d, rms_weight, eps, weight, bias, out2d, activation, gated)


def linear_scaled_supported(x2d, weight) -> bool:
    """What `kernl_linear_scaled_fwd` takes: 16-bit rows with unit feature stride, 16-byte aligned, K a multiple of 8."""
    M, K = x2d.shape
    return (
        x2d.dtype in (torch.float16, torch.bfloat16) and weight.dtype == x2d.dtype and K % 8 == 0 and x2d.stride(1) == 1
        and x2d.stride(0) % 8 == 0 and x2d.stride(0) < (1 << 22) and K < (1 << 22) and x2d.data_ptr() % 16 == 0
        and weight.is_contiguous() and weight.data_ptr() % 16 == 0
    )


def linear_scaled_fwd(x2d, weight, bias, row_scale, out2d, activation: int, gated: bool) -> None:
    """out = act((x @ w^T) * row_scale[:, None] + bias); gated: w and bias interleaved as for `linear_glu_fwd`."""
    _require_gpu(x2d, weight, bias, row_scale, out2d)
    M, K = x2d.shape
    N = out2d.shape[1]
    if row_scale.dtype != torch.float32 or row_scale.numel() != M or not row_scale.is_contiguous():
        raise ValueError("row_scale must be a contiguous fp32 vector with one entry per row of x")
    lib = load()
    with torch.cuda.device(x2d.device):
        st = lib.kernl_linear_scaled_fwd(
            x2d.data_ptr(), weight.data_ptr(), None if bias is None else bias.data_ptr(), row_scale.data_ptr(),
            out2d.data_ptr(), M, N, K, _arr(x2d.stride()), _arr(out2d.stride()), int(activation), int(bool(gated)),
            DTYPE_CODE[x2d.dtype], _stream(x2d),
        )
    _check(st, "kernl_linear_scaled_fwd")


def linear_residual_fwd(x2d, weight, bias, residual2d, out2d) -> None:
    """out = round(x @ w^T + bias) + residual in the epilogue of the wide tile kernels (`linear_scaled_supported` says
    which x and w they take; residual and out are [M, N] of x's dtype and must not overlap)."""
    _require_gpu(x2d, weight, bias, residual2d, out2d)
    M, K = x2d.shape
    N = out2d.shape[1]
    if residual2d.shape != out2d.shape or residual2d.dtype != x2d.dtype or out2d.dtype != x2d.dtype:
        raise ValueError("residual and out must have shape [M, N] and the dtype of x")
    lib = load()
    with torch.cuda.device(x2d.device):
        st = lib.kernl_linear_residual_fwd(
            x2d.data_ptr(), weight.data_ptr(), None if bias is None else bias.data_ptr(), residual2d.data_ptr(),
            out2d.data_ptr(), M, N, K, _arr(x2d.stride()), _arr(out2d.stride()), _arr(residual2d.stride()),
            DTYPE_CODE[x2d.dtype], _stream(x2d),
        )
    _check(st, "kernl_linear_residual_fwd")


def embedding_layernorm_fwd(tables, ids, weight, bias, out, eps: float) -> None:
    """out[b, s] = LayerNorm(sum of tables[i][ids[i][b, s]]) (rows added one after the other in the tables' dtype).
    tables: 1 to 3 contiguous [rows, N] matrices; ids: int64 [batch, seq] views (stride 0 allowed); out [batch, seq, N]."""
    _require_gpu(*tables, *ids, weight, bias, out)
    batch, seq, n = out.shape
    if not 1 <= len(tables) <= 3 or len(ids) != len(tables):
        raise ValueError("one to three tables, each with its ids")
    if not out.is_contiguous() or any(not t.is_contiguous() or t.shape[1] != n or t.dtype != out.dtype for t in tables):
        raise ValueError("tables and out must be contiguous, of one dtype and one width")
    if any(i.dtype != torch.int64 or tuple(i.shape) != (batch, seq) for i in ids):
        raise ValueError("ids must be int64 [batch, seq] (expanded views are fine)")
    args = []
    for k in range(3):
        if k < len(tables):
            args += [tables[k].data_ptr(), ids[k].data_ptr(), ids[k].stride(0), ids[k].stride(1), tables[k].shape[0]]
        else:
            args += [None, None, 0, 0, 0]
    lib = load()
    with torch.cuda.device(out.device):
        st = lib.kernl_embedding_layernorm_fwd(*args, weight.data_ptr(), None if bias is None else bias.data_ptr(), out.data_ptr(),
                                               batch, seq, n, float(eps), DTYPE_CODE[out.dtype], _stream(out))
    _check(st, "kernl_embedding_layernorm_fwd")


def select_mask_fwd(mask, on: float, off: float, out) -> None:
    """out = where(mask != 0, on, off) of a contiguous integer or boolean mask."""
    _require_gpu(mask, out)
    if not mask.is_contiguous() or not out.is_contiguous() or mask.numel() != out.numel() or mask.is_floating_point():
        raise ValueError("a contiguous integer mask and an output of its size")
    with torch.cuda.device(mask.device):
        st = load().kernl_select_mask_fwd(mask.data_ptr(), mask.element_size(), float(on), float(off), out.data_ptr(), mask.numel(),
                                          DTYPE_CODE[out.dtype], _stream(mask))
    _check(st, "kernl_select_mask_fwd")


def add_rms_stats_fwd(a2d, b2d, sum2d, rstd, eps: float) -> None:
    """sum = a + b (b and sum may be None: statistics of `a` alone), rstd[m] = 1 / sqrt(mean(sum[m]^2) + eps)."""
    _require_gpu(a2d, b2d, sum2d, rstd)
    M, N = a2d.shape
    if rstd.dtype != torch.float32 or rstd.numel() != M or not rstd.is_contiguous():
        raise ValueError("rstd must be a contiguous fp32 vector with one entry per row")
    if a2d.stride(1) != 1 or (b2d is not None and (b2d.stride(1) != 1 or sum2d.stride(1) != 1)):
        raise ValueError("add_rms_stats needs unit feature strides")
    lib = load()
    with torch.cuda.device(a2d.device):
        st = lib.kernl_add_rms_stats_fwd(
            a2d.data_ptr(), None if b2d is None else b2d.data_ptr(), None if sum2d is None else sum2d.data_ptr(),
            rstd.data_ptr(), M, N, a2d.stride(0), 0 if b2d is None else b2d.stride(0),
            0 if sum2d is None else sum2d.stride(0), float(eps), DTYPE_CODE[a2d.dtype], _stream(a2d),
        )
    _check(st, "kernl_add_rms_stats_fwd")


def linear_decode_supported(x2d, weight) -> bool:
    """What `kernl_linear_decode_fwd` takes: 16-bit rows, at most 64 of them, K a multiple of 64, a 16-bit weight."""
    M, K = x2d.shape
    return (
        x2d.dtype in (torch.float16, torch.bfloat16) and weight.dtype == x2d.dtype and M <= 64 and K % 64 == 0
        and x2d.stride(1) == 1 and x2d.stride(0) % 8 == 0 and x2d.data_ptr() % 16 == 0
        and weight.is_contiguous() and weight.data_ptr() % 16 == 0
    )


def linear_decode_fwd(x2d, rms_weight, eps: float, weight, bias, residual2d, out2d, cos=None, sin=None, head_dim: int = 0,
                      rope_cols: int = 0, rows_per_batch: int = 1) -> None:
    """cos / sin: [batch | 1, positions, head_dim] tables (unit feature stride) or None; row m of x2d is position
    m % rows_per_batch of batch entry m / rows_per_batch."""
    (_host or host()).linear_decode_fwd(x2d, rms_weight, eps, weight, bias, residual2d, out2d, cos, sin, head_dim, rope_cols, rows_per_batch)


def linear_splitk_workspace_bytes(x2d, weight) -> int:
    """Bytes of workspace `linear_splitk_fwd` wants for this product; 0: splitting K does not pay (or the input is not
    what the kernel takes) and `linear_fwd` is the call to make."""
    M, K = x2d.shape
    if not (
        x2d.dtype in (torch.float16, torch.bfloat16) and weight.dtype == x2d.dtype and K % 64 == 0 and K < (1 << 22)
        and x2d.stride(1) == 1 and x2d.stride(0) % 8 == 0 and x2d.stride(0) < (1 << 22) and x2d.data_ptr() % 16 == 0
        and weight.is_contiguous() and weight.data_ptr() % 16 == 0
    ):
        return 0
    return int(load().kernl_linear_splitk_workspace_bytes(M, weight.shape[0], K))


def linear_splitk_fwd(x2d, weight, bias, out2d, act_in2d, activation: int, workspace) -> None:
    _require_gpu(x2d, weight, bias, out2d, act_in2d, workspace)
    M, K = x2d.shape
    N = out2d.shape[1]
    lib = load()
    with torch.cuda.device(x2d.device):
        st = lib.kernl_linear_splitk_fwd(
            x2d.data_ptr(), weight.data_ptr(), None if bias is None else bias.data_ptr(), out2d.data_ptr(),
            None if act_in2d is None else act_in2d.data_ptr(), workspace.data_ptr(),
            workspace.numel() * workspace.element_size(), M, N, K, _arr(x2d.stride()), _arr(out2d.stride()),
            None if act_in2d is None else _arr(act_in2d.stride()), int(activation), DTYPE_CODE[x2d.dtype], _stream(x2d),
        )
    _check(st, "kernl_linear_splitk_fwd")


FINISH_PLAIN, FINISH_RESIDUAL, FINISH_RMS_STATS, FINISH_LAYER_NORM = range(4)


def linear_split_workspace_bytes(M: int, N: int, K: int, finish: int = FINISH_PLAIN) -> int:
    """Bytes of workspace where splitting K beats one pass over it (65 to 4096 rows); 0 where it does not."""
    return int(load().kernl_linear_split_workspace_bytes(M, N, K, finish))


def linear_split_fwd(x2d, weight, bias, residual2d, gamma, beta, eps: float, out2d, rstd, workspace, finish: int) -> None:
    """`kernl_linear_split_fwd`: the product with K split, its rows finished (residual, row statistics or LayerNorm)."""
    _require_gpu(x2d, weight, bias, residual2d, gamma, beta, out2d, rstd, workspace)
    ptr = lambda t: None if t is None else t.data_ptr()  # noqa: E731
    lib = load()
    with torch.cuda.device(x2d.device):
        st = lib.kernl_linear_split_fwd(
            x2d.data_ptr(), weight.data_ptr(), ptr(bias), residual2d.data_ptr(), ptr(gamma), ptr(beta), float(eps), out2d.data_ptr(), ptr(rstd),
            workspace.data_ptr(), workspace.numel() * workspace.element_size(), x2d.shape[0], out2d.shape[1], x2d.shape[1], x2d.stride(0),
            residual2d.stride(0), out2d.stride(0), int(finish), DTYPE_CODE[x2d.dtype], _stream(x2d),
        )
    _check(st, "kernl_linear_split_fwd")


def linear_exchange_bytes(M: int, N: int, K: int) -> int:
    """Bytes of a region of `linear_add_norm_fwd`; 0 where other routes are faster."""
    return int(load().kernl_linear_exchange_bytes(M, N, K))


def linear_add_norm_fwd(x2d, weight, bias, residual2d, gamma, beta, eps: float, out2d, sums, region, next_region, patience: int = -1) -> None:
    """`kernl_linear_add_norm_fwd`: product, addition and LayerNorm in one launch; `region` is all zeros, `next_region` is left so."""
    _require_gpu(x2d, weight, bias, residual2d, gamma, beta, out2d, sums, region, next_region)
    ptr = lambda t: None if t is None else t.data_ptr()  # noqa: E731
    lib = load()
    with torch.cuda.device(x2d.device):
        st = lib.kernl_linear_add_norm_fwd(
            x2d.data_ptr(), weight.data_ptr(), ptr(bias), residual2d.data_ptr(), gamma.data_ptr(), ptr(beta), float(eps), out2d.data_ptr(),
            sums.data_ptr(), region.data_ptr(), next_region.data_ptr(), min(region.numel(), next_region.numel()) * 8, int(patience), x2d.shape[0],
            out2d.shape[1], x2d.shape[1], x2d.stride(0), residual2d.stride(0), out2d.stride(0), DTYPE_CODE[x2d.dtype], _stream(x2d),
        )
    _check(st, "kernl_linear_add_norm_fwd")


def linear_fewrow_supported(x2d, weight) -> bool:
    """What `kernl_linear_fewrow_fwd` / `_w8_fwd` take: 16-bit rows, at most 128 of them, K a multiple of 64 from 256 on,
    a weight of the same type or — fp16 rows only — fp8 e5m2 bytes."""
    M, K = x2d.shape
    one_byte = weight.dtype in (torch.int8, torch.uint8, torch.float8_e5m2)
    return (
        x2d.dtype in (torch.float16, torch.bfloat16) and 0 < M <= 128
        and (weight.dtype == x2d.dtype or (one_byte and x2d.dtype == torch.float16))
        and K % 64 == 0 and K >= 256 and x2d.stride(1) == 1 and x2d.stride(0) % 8 == 0 and x2d.data_ptr() % 16 == 0
        and weight.is_contiguous() and weight.data_ptr() % 16 == 0
    )


def linear_fewrow_workspace_bytes(M: int, N: int, K: int, gated: bool = False, rotated: bool = False) -> int:
    """N: output width (the gated form's weight has twice as many rows)."""
    return int(load().kernl_linear_fewrow_workspace_bytes(M, N, K, int(bool(gated)), int(bool(rotated))))


def linear_fewrow_fwd(x2d, weight, bias, residual2d, out2d, activation: int, workspace=None, rms_weight=None,
                      eps: float = 0.0, gated: bool = False, cos=None, sin=None, head_dim: int = 0, rope_cols: int = 0,
                      rows_per_batch: int = 1) -> None:
    """`workspace`: device tensor of at least `linear_fewrow_workspace_bytes` bytes; allocated in the call when None (a
    fresh allocation per call: stream-ordered, so calls on different streams never share one).  cos / sin as for
    `linear_decode_fwd`; `gated`: weight and bias interleaved as for `linear_glu_fwd`, out2d half as wide."""
    (_host or host()).linear_fewrow_fwd(x2d, weight, bias, residual2d, out2d, activation, workspace, rms_weight, eps, gated, cos, sin,
                                        head_dim, rope_cols, rows_per_batch)


def linear_glu_fwd(x2d, weight_interleaved, bias_interleaved, out2d, activation: int) -> None:
    _require_gpu(x2d, weight_interleaved, bias_interleaved, out2d)
    M, K = x2d.shape
    N = weight_interleaved.shape[0] // 2
    lib = load()
    with torch.cuda.device(x2d.device):
        st = lib.kernl_linear_glu_fwd(
            x2d.data_ptr(), weight_interleaved.data_ptr(),
            None if bias_interleaved is None else bias_interleaved.data_ptr(), out2d.data_ptr(),
            M, N, K, _arr(x2d.stride()), _arr(out2d.stride()), int(activation), DTYPE_CODE[x2d.dtype], _stream(x2d),
        )
    _check(st, "kernl_linear_glu_fwd")


def layernorm_fwd(x2d, weight, bias, out2d, mean, rstd, eps: float, is_rms: bool, residual2d=None) -> None:
    (_host or host()).layernorm_fwd(x2d, weight, bias, out2d, mean, rstd, eps, is_rms, residual2d)
