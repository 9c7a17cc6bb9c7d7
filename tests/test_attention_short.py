"""The attention kernel for short key sequences (csrc/attention_short.hip) at the edges of its key blocks and row tiles."""
import pytest
import torch

from kernl_amd import _lib
from kernl_amd.implementations.attention import attention_forward
from oracle import attention_oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def short_kernel():
    lib = _lib.load()
    lib.kernl_attention_set_variant(6)
    yield
    lib.kernl_attention_set_variant(0)


# (rows, keys): blocks of 16 keys in steps of 2 / 4 / 6 / 8 / 12 / 16, rows around 16 and 64
SIZES = [(1, 1), (16, 16), (17, 31), (32, 32), (15, 33), (63, 64), (65, 65), (77, 77), (96, 96), (5, 97), (128, 128), (129, 129), (3, 192),
         (193, 193), (64, 255), (256, 256)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("head", [64, 128])
@pytest.mark.parametrize("kind", ["none", "padding", "min", "causal", "cached"])
@pytest.mark.parametrize("m, n", SIZES, ids=lambda v: str(v))
def test_short_key_sequences(m, n, kind, head, dtype, close):
    if kind == "cached" and n < m:
        pytest.skip("new rows sit at the end of the keys")
    gen = torch.Generator().manual_seed(m * 300 + n)
    b, h = 2, 3
    # heads interleaved in one buffer, as a fused projection leaves them
    q = torch.randn((b, m, h, head), generator=gen).to(dtype).transpose(1, 2)
    k, v = torch.randn((2, b, n, h, head), generator=gen).to(dtype).transpose(2, 3)
    mask, causal, start = None, kind in ("causal", "cached"), n - m if kind == "cached" else 0
    if kind in ("padding", "min"):
        lengths = torch.randint(0 if kind == "min" else (n + 1) // 2, n + 1, (b, 1), generator=gen)  # (0: a fully masked row)
        fill = torch.finfo(dtype).min if kind == "min" else float("-inf")
        mask = torch.zeros((b, n)).masked_fill_(torch.arange(n)[None, :] >= lengths, fill)[:, None, None, :].to(dtype if kind == "min" else torch.float32)
    out = torch.full((b, m, h, head), float("nan"), dtype=dtype, device="cuda").transpose(1, 2)
    attention_forward(q.cuda(), k.cuda(), v.cuda(), out, head ** -0.5, causal, None if mask is None else mask.cuda(), start)
    torch.cuda.synchronize()
    expected = attention_oracle(q, k, v, head ** -0.5, causal, mask, start_position=start)
    close(out, expected, dtype, what=f"{m}x{n} {kind} {head}")


# (batch, heads, rows, keys, head size): many rows over few keys, on both sides of the lines of `attention_short_pays`
CROSS = [(2, 3, 1000, 32, 128), (2, 3, 1000, 33, 64), (2, 3, 4096, 64, 128), (2, 3, 4160, 64, 128), (9, 16, 190, 40, 128), (7, 64, 64, 64, 128)]


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("b, h, m, n, head", CROSS, ids=str)
def test_many_rows_over_few_keys(b, h, m, n, head, masked, close):
    _lib.load().kernl_attention_set_variant(0)  # the kernel the rule takes
    gen = torch.Generator().manual_seed(m + n)
    q, (k, v) = torch.randn((b, h, m, head), generator=gen).half(), torch.randn((2, b, h, n, head), generator=gen).half()
    mask = None
    if masked:
        mask = torch.zeros((b, n)).masked_fill_(torch.arange(n)[None, :] >= torch.randint(1, n + 1, (b, 1), generator=gen), float("-inf"))[:, None, None, :]
    out = torch.full_like(q, float("nan"), device="cuda")
    attention_forward(q.cuda(), k.cuda(), v.cuda(), out, head ** -0.5, False, None if mask is None else mask.cuda())
    torch.cuda.synchronize()
    close(out, attention_oracle(q, k, v, head ** -0.5, False, mask), what=f"{m} rows over {n} keys")
