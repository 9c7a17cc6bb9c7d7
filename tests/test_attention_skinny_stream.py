"""Single-query attention over keys and values larger than the memory-side cache (loaded without a place in it)."""
import pytest
import torch

from kernl_amd import _lib
from kernl_amd.implementations.attention_skinny import skinny_attention_forward

pytestmark = pytest.mark.gpu


# just above the border and just below it, a ragged number of keys
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("shape", [(8, 32, 1, 2051, 128), (8, 32, 1, 2045, 128), (16, 32, 1, 2051, 64)], ids=str)
def test_streamed_keys_and_values(shape, dtype):
    B, H, M, N, D = shape
    gen = torch.Generator("cuda").manual_seed(N)
    q = torch.randn((B, H, M, D), generator=gen, device="cuda").to(dtype)
    k, v = (torch.randn((B, H, N, D), generator=gen, device="cuda").to(dtype) for _ in range(2))
    out = torch.empty_like(q)
    skinny_attention_forward(q, k, v, out, D ** -0.5)
    # in fp32, one head at a time
    for b, h in ((0, 0), (B - 1, H - 1), (B // 2, 3)):
        p = torch.softmax(q[b, h].float() @ k[b, h].float().T * D ** -0.5, -1)
        ref = p @ v[b, h].float()
        # one rounding of the result: |result| <= 0.5, 2^-11 (2^-8) of it, and as much again for 16-bit products of q
        assert (out[b, h].float() - ref).abs().max().item() <= (2.0 ** -10 if dtype == torch.float16 else 2.0 ** -8)
