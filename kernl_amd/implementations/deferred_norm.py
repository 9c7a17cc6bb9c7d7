"""A LayerNorm between linear layers without a kernel of its own — host side of `kernl_linear_norm_add_fwd` and
`kernl_linear_norm_apply_fwd` (csrc/norm_fold.h says what is computed where, and in how many bits).

The reference runs one Triton LayerNorm between its linear kernels (src/kernl/implementations/layer_norm.py:279-335); at
a few dozen rows such a launch is 2.7 us for a fraction of a microsecond of work, twice per encoder layer."""
from typing import Optional, Sequence, Tuple

import torch

from kernl_amd import _lib
from kernl_amd.implementations.linear_layer import ACTIVATIONS

MAX_WIDTH = 1024  # statistics of a row that the kernels stage


class DeferredNorm:
    """layer_norm(rows, gamma, beta, eps) that has not been carried out: fp32 rows and their statistics, standing for a tensor
    of gamma's 16-bit type."""

    def __init__(self, rows: torch.Tensor, stats: torch.Tensor, gamma: torch.Tensor, beta: Optional[torch.Tensor], eps: float):
        self.rows, self.stats, self.gamma, self.beta, self.eps = rows, stats, gamma, beta, eps
        self._normed = None

    @property
    def dtype(self) -> torch.dtype:
        return self.gamma.dtype

    @property
    def kernel_eps(self) -> float:
        return max(self.eps, 1.6e-5) if self.dtype == torch.float16 else self.eps  # the fp16 policy of the operator

    def normalised(self) -> torch.Tensor:
        """The tensor this stands for."""
        if self._normed is None:
            k = self.rows.shape[-1]
            out = torch.empty(self.rows.shape, device=self.rows.device, dtype=self.dtype)
            _lib.layernorm_rows32_fwd(self.rows.view(-1, k), self.gamma, self.beta, out.view(-1, k), self.kernel_eps)
            self._normed = out
        return self._normed

    def takes_linear(self, weight: torch.Tensor, bias: Optional[torch.Tensor], activation: str) -> bool:
        return activation in ACTIVATIONS and _takes(self.rows.numel() // self.rows.shape[-1], weight.shape[0], weight.shape[1]) and _plain(self.dtype, weight, bias)

    def linear(self, weight: torch.Tensor, bias: Optional[torch.Tensor], activation: str = "") -> torch.Tensor:
        """activation(linear(layer_norm(rows), weight, bias)), in one launch."""
        k, n = self.rows.shape[-1], weight.shape[0]
        out = torch.empty((*self.rows.shape[:-1], n), device=self.rows.device, dtype=self.dtype)
        _lib.linear_norm_apply_fwd(self.rows.view(-1, k), self.stats, self.gamma, self.beta, self.kernel_eps, weight, bias,
                                   out.view(-1, n), ACTIVATIONS[activation])
        return out


def _takes(rows: int, n: int, k: int) -> bool:
    return _lib.linear_norm_kind(rows, n, k) != 0


def _plain(dtype: torch.dtype, *params: Optional[torch.Tensor]) -> bool:
    return all(p is None or (p.dtype == dtype and p.is_contiguous() and p.data_ptr() % 16 == 0) for p in params)


def rows_of(t: torch.Tensor) -> torch.Tensor:
    """t as [rows, features]; a copy where its strides have no such view."""
    return t if t.dim() == 2 else t.reshape(-1, t.shape[-1])


def row_stride(t: torch.Tensor) -> Optional[int]:
    """The row stride of `rows_of(t)`, found without making it; None unless its features are contiguous and its 16-bit rows 16-byte aligned."""
    features, row, step = t.shape[-1], None, None
    for size, stride in zip(reversed(t.shape[:-1]), reversed(t.stride()[:-1])):
        if size == 1:
            continue
        if step is None:
            row, step = stride, stride * size
        elif stride == step:
            step *= size
        else:  # no view: the rows of the copy lie one behind the other
            return features if features % 8 == 0 else None
    if t.dim() == 2:  # as it lies, also with one row
        row = t.stride(0)
    elif row is None:  # one row: the view's rows lie one behind the other
        row = features
    return row if t.stride(-1) == 1 and row % 8 == 0 and t.data_ptr() % 16 == 0 else None


def deferrable(x: torch.Tensor, weight: torch.Tensor, bias, residual, gamma, beta, behind: Sequence[Tuple[torch.Tensor, ...]]) -> bool:
    """Whether layer_norm(linear(x, weight, bias) + residual, gamma, beta) can be left to the layers behind it, whose weights are
    `behind` (several for sibling projections, which run as one)."""
    n, k = weight.shape
    inner = residual.rows if isinstance(residual, DeferredNorm) else residual
    if not (x.is_cuda and x.dtype in (torch.float16, torch.bfloat16) and x.dim() >= 2 and x.numel() > 0 and gamma is not None):
        return False
    if torch.is_autocast_enabled("cuda") or not _plain(x.dtype, weight, bias, gamma, beta) or residual.dtype != x.dtype:
        return False
    if inner.shape != (*x.shape[:-1], n) or gamma.shape != (n,) or n % 32 != 0 or n > MAX_WIDTH:
        return False
    rows = x.numel() // k
    for weights in ((weight,), *behind):
        # (of siblings the rows are copied together, a single weight is read where and as it lies)
        if len(weights) == 1 and not _plain(x.dtype, weights[0]) or any(w.dtype != x.dtype for w in weights):
            return False
        if not _takes(rows, sum(w.shape[0] for w in weights), weights[0].shape[1]):
            return False
    stride = row_stride(x)  # (rows that lie over each other, as expanded ones do, are left to the other kernels)
    return stride is not None and k <= stride < (1 << 22) and row_stride(inner) is not None


def linear_add_deferred(x: torch.Tensor, weight: torch.Tensor, bias, residual, gamma, beta, eps: float) -> DeferredNorm:
    """linear(x, weight, bias) + residual in fp32 with its row statistics, in one launch; `residual` may be a deferred norm."""
    n = weight.shape[0]
    out = torch.empty((*x.shape[:-1], n), device=x.device, dtype=torch.float32)
    stats = torch.empty((x.numel() // x.shape[-1], n // _lib.NORM_GROUP, 2), device=x.device, dtype=torch.float32)
    if isinstance(residual, DeferredNorm):
        args = (rows_of(residual.rows), residual.stats, residual.gamma, residual.beta, residual.kernel_eps)
    else:
        args = (rows_of(residual), None, None, None, 0.0)
    _lib.linear_norm_add_fwd(rows_of(x), weight, bias, *args, out.view(-1, n), stats)
    return DeferredNorm(out, stats, gamma, beta, eps)
