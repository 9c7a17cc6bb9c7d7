"""Rotary position embedding — host side of `kernl_rope_fwd`.

out = x·cos + rotate_half(x)·sin in the half-split convention of Hugging Face decoders.  The reference fuses the
same rotation, in Meta's interleaved-pair convention, into its query/key projection kernel
(experimental/llama-v2/kernel/fused_kernel_proj_qkv.py:69-100; eager form experimental/llama-v2/llama/model.py:78-88).
"""
import torch

from kernl_amd import _lib


def rotary_forward(x: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor) -> torch.Tensor:
    """x [B,H,S,D]; cos, sin broadcastable to it with sizes [B|1, H|1, S, D].  The result has the dtype PyTorch's
    type promotion gives `x * cos` and the strides of x."""
    assert x.dim() == 4, f"expected [batch, heads, positions, features], got {tuple(x.shape)}"
    assert cos.shape == sin.shape and cos.dtype == sin.dtype, "cos and sin must agree in shape and dtype"
    while cos.dim() < 4:
        cos, sin = cos.unsqueeze(0), sin.unsqueeze(0)
    assert x.shape[-1] % 2 == 0, "feature size must be even"
    assert cos.dtype in _lib.DTYPE_CODE, f"Unsupported table dtype {cos.dtype}"
    out_dtype = torch.result_type(x, cos)
    assert out_dtype in _lib.DTYPE_CODE, f"Unsupported dtype {out_dtype}"
    if x.dtype != out_dtype:
        x = x.to(out_dtype)
    out = torch.empty_like(x)
    _lib.rope_fwd(x, cos, sin, out)
    return out


def rotary_tables(inv_freq: torch.Tensor, positions: torch.Tensor, scale: float, dtype: torch.dtype):
    """(cos, sin) [B,S,2*half] of `cat((a, a), -1)` with a = (inv_freq @ positions).transpose(1, 2), times scale, in dtype.
    inv_freq [B|1,half,1] floating, positions [B|1,1,S]: float32, or int64 to be rounded to it."""
    batch = max(inv_freq.shape[0], positions.shape[0])
    taken = (inv_freq.is_cuda and inv_freq.device == positions.device and inv_freq.dim() == 3 and positions.dim() == 3
             and inv_freq.shape[2] == 1 and positions.shape[1] == 1 and inv_freq.shape[0] in (1, batch) and positions.shape[0] in (1, batch)
             and inv_freq.dtype in _lib.DTYPE_CODE and positions.dtype in (torch.int64, torch.float32) and dtype in _lib.DTYPE_CODE
             and inv_freq.shape[1] > 0 and not torch.is_autocast_enabled("cuda"))
    if not taken:
        angles = (inv_freq.to(torch.float32) @ positions.to(torch.float32)).transpose(1, 2)
        both = torch.cat((angles, angles), dim=-1)
        return (both.cos() * scale).to(dtype), (both.sin() * scale).to(dtype)
    cos = torch.empty((batch, positions.shape[2], 2 * inv_freq.shape[1]), dtype=dtype, device=inv_freq.device)
    sin = torch.empty_like(cos)
    _lib.rope_tables(inv_freq, positions, cos, sin, scale)
    return cos, sin
