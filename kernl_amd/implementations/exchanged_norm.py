"""linear + residual + LayerNorm in one launch for more than 64 rows (`kernl_linear_add_norm_fwd`; csrc/norm_exchange.h says how the workgroups
of a row agree on its statistics).  No counterpart in the reference, whose models add and normalise in kernels of their own behind its linear
kernel (implementations/linear_layer.py:213-292, layer_norm.py:279-335)."""
from typing import Optional, Tuple

import torch

from kernl_amd import _lib
from kernl_amd.implementations.deferred_norm import rows_of
from kernl_amd.implementations.split_linear import FINISH_LAYER_NORM, finishing_bytes


class ExchangeRegions:
    """The pair of regions that the launches of ONE pass over a graph take by turns: a launch finds zeros in the first and leaves them in
    the second.  Made anew for every pass (a captured pass keeps its own), so that nothing is shared between passes, streams or threads."""

    def __init__(self):
        self._pair = None
        self._of: Optional[Tuple[torch.device, int]] = None

    def take(self, need: int, device: torch.device) -> Tuple[torch.Tensor, torch.Tensor]:
        """(region, region of the next launch), of at least `need` bytes each, for one launch on the current stream."""
        of = (device, torch.cuda.current_stream(device).cuda_stream)
        if self._pair is None or self._of != of or self._pair[0].numel() * 8 < need:
            words = (need + 7) // 8 * 2  # (the layers of a model differ in their tiles: room for twice as many words)
            self._pair = (torch.zeros(words, dtype=torch.int64, device=device), torch.empty(words, dtype=torch.int64, device=device))
            self._of = of
        pair = self._pair
        self._pair = pair[::-1]
        return pair


def exchange_bytes(x: torch.Tensor, weight: torch.Tensor, bias, residual: torch.Tensor, gamma, beta) -> int:
    """Bytes of a region for `linear_add_norm` on these operands; 0 where another route is faster or they are not plain 16-bit GPU tensors
    with nothing to record about them."""
    return finishing_bytes(_lib.linear_exchange_bytes, x, weight, bias, residual, FINISH_LAYER_NORM, gamma, beta)


def linear_add_norm(need: int, regions: ExchangeRegions, x: torch.Tensor, weight: torch.Tensor, bias, residual: torch.Tensor, gamma, beta,
                    eps: float, patience: int = -1) -> torch.Tensor:
    """layer_norm(linear(x) + residual), the sum in fp32.  `need`: what `exchange_bytes` said; eps as it is used."""
    out = torch.empty(residual.shape, device=x.device, dtype=x.dtype)
    n = out.shape[-1]
    rows = out.numel() // n
    sums = torch.empty((rows, n), dtype=torch.float32, device=x.device)
    region, behind = regions.take(need, x.device)
    _lib.linear_add_norm_fwd(rows_of(x), weight, bias, rows_of(residual), gamma, beta, eps, out.view(rows, n), sums, region, behind, patience)
    return out
