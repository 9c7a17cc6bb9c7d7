"""Linear layer for up to four rows of x on the kernel that streams the weight in whole lines (csrc/linear_stream.h)."""
import pytest
import torch

from kernl_amd.implementations.linear_layer import decode_linear_layer, interleave_glu_rows, linear_layer, rms_linear_layer
from oracle import linear_oracle, rotary_oracle

pytestmark = pytest.mark.gpu

DTYPES = pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
ROWS = pytest.mark.parametrize("rows", [1, 2, 3, 4])


def _operands(rows, n, k, dtype):
    gen = torch.Generator().manual_seed(rows + n + k)
    x, w = torch.randn((rows, k), generator=gen).to(dtype), (torch.randn((n, k), generator=gen) * k ** -0.5).to(dtype)
    return x, w, (0.3 * torch.randn((n,), generator=gen)).to(dtype), (1 + 0.1 * torch.randn((k,), generator=gen)).to(dtype), gen


def _normed(x, g, w, b=None):
    """The kernel's own order: x times the norm's weight in 16 bits, the row's factor on the sums."""
    r = torch.rsqrt(x.float().pow(2).mean(-1, keepdim=True) + 1.6e-5)
    y = linear_oracle((x * g).float(), w.float(), None, "") * r
    return y + b.float() if b is not None else y


# units of four and eight columns, whole and cut; one batch of k-steps a wave and fewer than there are waves; a last batch that is not whole; the most LDS
@DTYPES
@ROWS
@pytest.mark.parametrize("n, k", [(345, 1536), (513, 1664), (1024, 2048), (2050, 5120), (4096, 2176), (8196, 1536)])
@pytest.mark.parametrize("activation", ["", "gelu"])
def test_linear_layer(rows, n, k, activation, dtype, close):
    x, w, b, _, _ = _operands(rows, n, k, dtype)
    saved = torch.full((rows, n), float("nan"), dtype=dtype, device="cuda")
    wide = torch.full((rows, k + 8), float("nan"), dtype=dtype, device="cuda")
    wide[:, :k] = x.cuda()
    out = linear_layer(wide[:, :k], w.cuda(), b.cuda(), activation, saved)
    torch.cuda.synchronize()
    expect, pre = linear_oracle(x, w, b, activation, return_act_inputs=True)
    close(out, expect, dtype, what=f"{rows} x {n} x {k} {activation!r}")
    close(saved, pre, dtype, what="pre-activation")


@DTYPES
@ROWS
@pytest.mark.parametrize("n, k", [(352, 1536), (2752, 2048), (5504, 1664)])
def test_gates_behind_a_norm(rows, n, k, dtype, close):
    x, gate, b, g, gen = _operands(rows, n, k, dtype)
    value = (torch.randn((n, k), generator=gen) * k ** -0.5).to(dtype)
    out = rms_linear_layer(x.cuda().view(rows, 1, k), g.cuda(), 1.6e-5, interleave_glu_rows(gate.cuda(), value.cuda()), None, "silu", gated=True)
    torch.cuda.synchronize()
    expect = torch.nn.functional.silu(_normed(x, g, gate)) * _normed(x, g, value)
    close(out.view(rows, n), expect.to(dtype), dtype, what=f"gated {rows} x {n} x {k}")
    plain = rms_linear_layer(x.cuda().view(rows, 1, k), g.cuda(), 1.6e-5, gate.cuda(), b.cuda(), "")
    close(plain.view(rows, n), _normed(x, g, gate, b).to(dtype), dtype, what=f"norm {rows} x {n} x {k}")


@DTYPES
@ROWS
@pytest.mark.parametrize("table", [torch.float32, torch.float16, torch.bfloat16], ids=["t32", "t16", "tb16"])
@pytest.mark.parametrize("head, heads, turned, k, batches", [(64, 9, 6, 1536, 1), (128, 32, 32, 2048, 2), (32, 21, 0, 1664, 1)])
def test_rotated_columns(rows, head, heads, turned, k, batches, table, dtype, close):
    """Rows that are positions of one sequence, or of two; tables whose rows start at odd places."""
    if rows % batches:
        pytest.skip("rows do not divide over the sequences")
    n, seq = head * heads, rows // batches
    x, w, b, g, gen = _operands(rows, n, k, dtype)
    angle = torch.rand((batches, seq, head // 2), generator=gen) * 6
    tables = [f(torch.cat((angle, angle), -1)).to(table) for f in (torch.cos, torch.sin)]
    placed = []
    for t in tables:
        wide = torch.zeros((batches, seq, head + 3), dtype=table, device="cuda")
        wide[..., 1:head + 1] = t.cuda()
        placed.append(wide[..., 1:head + 1])
    res = torch.randn((rows, n), generator=gen).to(dtype)
    out = decode_linear_layer(x.cuda().view(batches, seq, k), w.cuda(), b.cuda(), g.cuda(), 1.6e-5, res.cuda().view(batches, seq, n), *placed,
                              head_dim=head, rope_cols=turned * head)
    torch.cuda.synchronize()
    y = _normed(x, g, w, b).view(batches, seq, heads, head).transpose(1, 2)
    y = torch.cat((rotary_oracle(y[:, :turned], *(t.float()[:, None] for t in tables)), y[:, turned:]), 1) if turned else y
    expect = y.transpose(1, 2).reshape(rows, n) + res.float()
    close(out.reshape(rows, n), expect.to(dtype), dtype, what=f"{rows} rows, {heads} heads of {head}")


@DTYPES
@ROWS
def test_residual(rows, dtype, close):
    x, w, b, _, gen = _operands(rows, 1021, 1792, dtype)
    res = torch.randn((1021, rows), generator=gen).to(dtype).t()  # its columns one after the other
    out = decode_linear_layer(x.cuda().view(rows, 1, -1), w.cuda(), b.cuda(), residual=res.cuda().view(rows, 1, -1))
    torch.cuda.synchronize()
    close(out.view(rows, -1), (linear_oracle(x, w, b, "").float() + res.float()).to(dtype), dtype, what="residual")


@DTYPES
@ROWS
def test_error_against_64_bits(rows, dtype):
    """Each result is within half a unit of its last place, plus the rounding of fp32 sums, of the result in 64 bits."""
    n, k = 2048, 4096
    x, w, b, _, _ = _operands(rows, n, k, dtype)
    out = linear_layer(x.cuda(), w.cuda(), b.cuda()).double().cpu()
    exact = x.double() @ w.double().t() + b.double()
    size = x.double().abs() @ w.double().abs().t() + b.double().abs()
    half_ulp = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    bound = exact.abs() * half_ulp * 1.001 + 2.0 ** -25 + size * 2.0 ** -23 * 8  # products are exact in fp32; some eight of the sums' partial results are as large
    assert ((out - exact).abs() <= bound).all()
