"""A LayerNorm between linear layers without a kernel of its own — host side of `kernl_linear_norm_add_fwd` and
`kernl_linear_norm_apply_fwd` (csrc/norm_fold.h says what is computed where).

The reference runs one Triton LayerNorm between its linear kernels (src/kernl/implementations/layer_norm.py:279-335); at
a few hundred rows such a launch is 2.7 us for a microsecond of work, twice per encoder layer."""
from typing import NamedTuple, Optional

import torch

from kernl_amd import _lib
from kernl_amd.implementations.linear_layer import ACTIVATIONS

MAX_WIDTH = 1024  # statistics of a row that the kernels stage


class FoldedParams(NamedTuple):
    """A linear layer's parameters with the LayerNorm in front of it folded in."""

    weight: torch.Tensor  # w * gamma, rounded once to the storage type
    colsum: torch.Tensor  # fp32 sums of its rows: what a row's mean contributes
    bias: torch.Tensor  # fp32, bias + w @ beta

    @classmethod
    def of(cls, weight, bias, gamma, beta) -> "FoldedParams":
        w32 = weight.detach().float()
        folded = (w32 * gamma.detach().float()[None, :]).to(weight.dtype)
        b = torch.zeros(weight.shape[0], device=weight.device) if bias is None else bias.detach().float()
        if beta is not None:
            b = b + (w32 * beta.detach().float()[None, :]).sum(1)
        return cls(folded.contiguous(), folded.float().sum(1), b.contiguous())


class DeferredNorm:
    """layer_norm(rows, gamma, beta, eps) that has not been carried out: the rows and their statistics."""

    def __init__(self, rows: torch.Tensor, stats: torch.Tensor, gamma: torch.Tensor, beta: Optional[torch.Tensor], eps: float):
        self.rows, self.stats, self.gamma, self.beta, self.eps = rows, stats, gamma, beta, eps
        self._normed = None

    @property
    def kernel_eps(self) -> float:
        return max(self.eps, 1.6e-5) if self.rows.dtype == torch.float16 else self.eps  # the fp16 policy of the operator

    def normalised(self) -> torch.Tensor:
        """The tensor this stands for, by the LayerNorm kernel."""
        from kernl_amd.implementations.layer_norm import layer_norm

        if self._normed is None:
            self._normed = layer_norm(self.rows, self.gamma, self.beta, self.eps)
        return self._normed

    def takes_linear(self, out_features: int, activation: str) -> bool:
        k = self.rows.shape[-1]
        return activation in ACTIVATIONS and _lib.linear_norm_kind(self.rows.numel() // k, out_features, k) != 0

    def linear(self, params: FoldedParams, activation: str = "") -> torch.Tensor:
        """activation(linear(layer_norm(rows))) with the folded parameters, in one launch."""
        k, n = self.rows.shape[-1], params.weight.shape[0]
        out = torch.empty((*self.rows.shape[:-1], n), device=self.rows.device, dtype=self.rows.dtype)
        _lib.linear_norm_apply_fwd(self.rows.view(-1, k), self.stats, self.kernel_eps, params.weight, params.colsum, params.bias,
                                   out.view(-1, n), ACTIVATIONS[activation])
        return out


def _rows(t: torch.Tensor) -> Optional[torch.Tensor]:
    t = t if t.dim() == 2 else t.reshape(-1, t.shape[-1])
    return t if t.stride(-1) == 1 and t.stride(0) % 8 == 0 and t.data_ptr() % 16 == 0 else None


def deferrable(x: torch.Tensor, weight: torch.Tensor, bias, residual, gamma, beta) -> bool:
    """Whether layer_norm(linear(x, weight, bias) + residual, gamma, beta) can be left to the layers behind it."""
    n, k = weight.shape
    inner = residual.rows if isinstance(residual, DeferredNorm) else residual
    params = [p for p in (weight, bias, gamma, beta) if p is not None]
    if not (x.is_cuda and x.dtype in (torch.float16, torch.bfloat16) and x.dim() >= 2 and x.numel() > 0 and gamma is not None):
        return False
    if torch.is_autocast_enabled("cuda") or any(p.dtype != x.dtype or not p.is_contiguous() or p.data_ptr() % 16 for p in params):
        return False
    if inner.dtype != x.dtype or inner.shape != (*x.shape[:-1], n) or gamma.shape != (n,) or n % 32 != 0 or n > MAX_WIDTH:
        return False
    rows = x.numel() // k
    # ... and the layers an encoder has behind its norms (three and four times as wide) take what is left to them
    if any(_lib.linear_norm_kind(rows, a, b) == 0 for a, b in ((n, k), (3 * n, n), (4 * n, n))):
        return False
    return _rows(x) is not None and _rows(inner) is not None


def linear_add_deferred(x: torch.Tensor, weight: torch.Tensor, bias, residual, gamma, beta, eps: float) -> DeferredNorm:
    """linear(x, weight, bias) + residual with its row statistics, in one launch; `residual` may be a deferred norm."""
    n = weight.shape[0]
    out = torch.empty((*x.shape[:-1], n), device=x.device, dtype=x.dtype)
    rows = x.numel() // x.shape[-1]
    stats = torch.empty((rows, n // _lib.linear_norm_group(rows), 2), device=x.device, dtype=torch.float32)
    if isinstance(residual, DeferredNorm):
        args = (_rows(residual.rows), residual.stats, residual.gamma, residual.beta, residual.kernel_eps)
    else:
        args = (_rows(residual), None, None, None, 0.0)
    _lib.linear_norm_add_fwd(_rows(x), weight, bias, *args, out.view(-1, n), stats)
    return DeferredNorm(out, stats, gamma, beta, eps)
