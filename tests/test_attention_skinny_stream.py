"""Single-query attention over keys and values larger than the memory-side cache (loaded without a place in it)."""
import pytest
import torch

from kernl_amd.implementations.attention_skinny import skinny_attention_forward

pytestmark = pytest.mark.gpu


# just above the border and just below it, a ragged number of keys
@pytest.mark.parametrize("masked", [False, True], ids=["whole", "masked"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("shape", [(8, 32, 1, 2051, 128), (8, 32, 1, 2045, 128), (16, 32, 1, 2051, 64)], ids=str)
def test_streamed_keys_and_values(shape, dtype, masked):
    B, H, M, N, D = shape
    gen = torch.Generator("cuda").manual_seed(N)
    q = torch.randn((B, H, M, D), generator=gen, device="cuda").to(dtype)
    k, v = (torch.randn((B, H, N, D), generator=gen, device="cuda").to(dtype) for _ in range(2))
    # Some 40 keys hold nearly all of the weight, 2 % each, and values of 3 or -3: the last eight, the first, and both sides of every
    # multiple of 128.  Leaving one of them out, or taking it twice, moves the result by 0.05.
    heavy = sorted({0, *range(N - 8, N), *range(127, N, 128), *range(128, N, 128)})
    scale = D ** -0.5
    k[:, :, heavy] = (q.float() * (8.0 / scale) / q.float().square().sum(-1, keepdim=True)).to(dtype)
    v[:, :, heavy] = (6 * torch.randint(0, 2, (B, H, len(heavy), D), generator=gen, device="cuda") - 3).to(dtype)
    mask = None
    if masked:  # the last keys of some entries, heavy ones among them, and a slope over the others
        mask = torch.linspace(0, -0.5, N, device="cuda").expand(B, 1, 1, N).contiguous()
        mask[1::2, ..., -5:] = float("-inf")
        mask[::3, ..., 100:300] = float("-inf")
    out = torch.empty_like(q)
    skinny_attention_forward(q, k, v, out, scale, False, mask)
    unit = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -9
    for b in range(B):  # in fp32, all heads
        s = (q[b].float() * k[b].float()).sum(-1) * scale
        if masked:
            s = s + mask[b, 0]
        p, vb = torch.softmax(s, -1)[..., None], v[b].float()
        expect, size = (p * vb).sum(-2), (p * vb.abs()).sum(-2)
        # weights rounded to 16 bits above and below the line, the result once more, fp32 sums of 128 + N terms: unit each of sum(p |v|)
        assert ((out[b, :, 0].float() - expect).abs() <= (3 * unit + 1e-4) * size).all(), b
