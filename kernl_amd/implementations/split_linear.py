"""Linear layers with K split over several workgroups a tile, whose second launch finishes the rows: the residual, the row statistics of
the RMSNorm behind it, or the whole add + LayerNorm (`kernl_linear_split_fwd`).  No counterpart in the reference, whose models add and
normalise in kernels of their own behind its linear kernel (implementations/linear_layer.py:213-292)."""
import torch
from torch.autograd import forward_ad

from kernl_amd import _lib
from kernl_amd.implementations.deferred_norm import row_stride, rows_of

FINISH_RESIDUAL, FINISH_RMS_STATS, FINISH_LAYER_NORM = _lib.FINISH_RESIDUAL, _lib.FINISH_RMS_STATS, _lib.FINISH_LAYER_NORM


def split_finish_bytes(x: torch.Tensor, weight: torch.Tensor, bias, residual: torch.Tensor, finish: int, gamma=None, beta=None) -> int:
    """Bytes of workspace for `split_finish_linear` on these operands; 0 where another route is faster or they are not plain 16-bit GPU
    tensors with nothing to record about them."""
    return finishing_bytes(lambda m, n, k: _lib.linear_split_workspace_bytes(m, n, k, finish), x, weight, bias, residual, finish, gamma, beta)


def finishing_bytes(bytes_of, x: torch.Tensor, weight: torch.Tensor, bias, residual: torch.Tensor, finish: int, gamma=None, beta=None) -> int:
    """What `bytes_of(rows, out features, in features)` says if the operands are plain 16-bit GPU tensors with nothing to record about
    them, of the layouts that the finishing kernels take; else 0."""
    n, k = weight.shape
    if not (isinstance(residual, torch.Tensor) and x.is_cuda and x.dtype in (torch.float16, torch.bfloat16) and x.dim() >= 2 and x.numel() > 0):
        return 0
    if residual.dtype != x.dtype or residual.device != x.device or residual.shape != (*x.shape[:-1], n) or x.shape[-1] != k:
        return 0
    params = [p for p in (weight, bias, gamma, beta) if p is not None]
    if any(p.dtype != x.dtype or p.device != x.device or not p.is_contiguous() or p.data_ptr() % 16 != 0 for p in params):
        return 0
    if any(p.shape != (n,) for p in (bias, gamma, beta) if p is not None) or (finish == FINISH_LAYER_NORM and gamma is None):
        return 0
    need = bytes_of(x.numel() // k, n, k)
    if need == 0 or not _lib.host().takes_call() or forward_ad._current_level >= 0:
        return 0
    if torch.is_grad_enabled() and any(t.requires_grad for t in (x, residual, *params)):
        return 0
    stride = row_stride(x)
    return need if stride is not None and k <= stride < (1 << 22) and row_stride(residual) is not None else 0


def split_finish_linear(need: int, x: torch.Tensor, weight: torch.Tensor, bias, residual: torch.Tensor, finish: int, gamma=None, beta=None,
                        eps: float = 0.0):
    """FINISH_RESIDUAL: round(linear(x)) + residual; FINISH_RMS_STATS: (that, rstd fp32 [rows]); FINISH_LAYER_NORM: layer_norm(linear(x) +
    residual), the sum in fp32.  `need`: what `split_finish_bytes` said; eps as it is used."""
    out = torch.empty(residual.shape, device=x.device, dtype=x.dtype)
    rows = x.numel() // x.shape[-1]
    rstd = torch.empty((rows,), device=x.device, dtype=torch.float32) if finish == FINISH_RMS_STATS else None
    workspace = torch.empty(need, dtype=torch.uint8, device=x.device)
    _lib.linear_split_fwd(rows_of(x), weight, bias, rows_of(residual), gamma, beta, eps, out.view(rows, -1), rstd, workspace, finish)
    return (out, rstd) if finish == FINISH_RMS_STATS else out
