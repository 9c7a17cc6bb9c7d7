"""Where split K is what runs: `linear_layer` by both its routes, and the wrappers that finish the rows in the launch behind it."""
import pytest
import torch

from kernl_amd import _lib
from kernl_amd.implementations.linear_layer import LinearLayer, linear_layer
from kernl_amd.optimizer import linear as wrappers
from oracle import effective_eps, layer_norm_oracle, linear_oracle

pytestmark = pytest.mark.gpu

DTYPES = pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])


def _operands(M, N, K, dtype, seed):
    gen = torch.Generator().manual_seed(seed)
    x, w = torch.randn((M, K), generator=gen).to(dtype), (torch.randn((N, K), generator=gen) * K ** -0.5).to(dtype)
    return x, w, (0.3 * torch.randn((N,), generator=gen)).to(dtype), gen


@DTYPES
@pytest.mark.parametrize("activation, code", [("", _lib.ACT_NONE), ("fast_gelu", _lib.ACT_GELU_TANH)], ids=["plain", "gelu"])
@pytest.mark.parametrize("route", ["host", "python"])
def test_linear_layer(route, activation, code, dtype, close):
    M, N, K = 200, 4096, 11008
    x, w, b, _ = _operands(M, N, K, dtype, 3)
    xd, wd, bd = x.cuda(), w.cuda(), b.cuda()
    need = _lib.linear_split_workspace_bytes(M, N, K)
    assert need > 0
    split, one_pass, saved, saved_split = (torch.full((M, N), float("nan"), dtype=dtype, device="cuda") for _ in range(4))
    _lib.linear_splitk_fwd(xd, wd, bd, split, saved_split, code, torch.full((need // 4,), float("nan"), device="cuda"))
    _lib.linear_fwd(xd, wd, bd, one_pass, None, code)
    run = LinearLayer.apply if route == "python" else linear_layer
    out = run(xd.view(2, M // 2, K), wd, bd, activation, saved)
    torch.cuda.synchronize()
    # the sums of the ranges in another order than one pass over K: the bits say which ran
    assert torch.equal(out.view(M, N), split) and torch.equal(saved, saved_split) and not torch.equal(split, one_pass)
    expect, pre = linear_oracle(x, w, b, activation, return_act_inputs=True)
    close(out.view(M, N), expect, dtype, what=f"{route} {activation!r}")
    close(saved, pre, dtype, what=f"{route} pre-activation")


@pytest.fixture
def finished(monkeypatch):
    """The (eps, finish, row strides of x and residual) of every launch that finishes rows."""
    calls, real = [], _lib.linear_split_fwd

    def spy(x2d, weight, bias, residual2d, gamma, beta, eps, out2d, rstd, workspace, finish):
        calls.append((eps, finish, x2d.stride(0), residual2d.stride(0)))
        return real(x2d, weight, bias, residual2d, gamma, beta, eps, out2d, rstd, workspace, finish)

    monkeypatch.setattr(_lib, "linear_split_fwd", spy)
    return calls


def _cut(t, extra):
    """t [rows, features] as three dimensions whose rows lie `extra` elements further apart than they are long."""
    rows, features = t.shape
    wide = torch.full((3, rows // 3, features + extra), float("nan"), dtype=t.dtype, device="cuda")
    wide[..., :features] = t.view(3, rows // 3, features).cuda()
    return wide[..., :features]


# eps below what fp16 takes (clamped to 1.6e-5 there) and one that rows of small values feel
@pytest.mark.parametrize("dtype, eps", [(torch.float16, 1e-12), (torch.bfloat16, 1e-3)], ids=["fp16", "bf16"])
@pytest.mark.parametrize("finish", [_lib.FINISH_RESIDUAL, _lib.FINISH_RMS_STATS, _lib.FINISH_LAYER_NORM], ids=["residual", "stats", "norm"])
def test_wrappers_with_rows_cut_out_of_wider_ones(finish, dtype, eps, finished, close):
    M, N, K = (150, 4096, 11008) if finish == _lib.FINISH_RESIDUAL else (300, 1024, 4096)
    x, w, b, gen = _operands(M, N, K, dtype, 5)
    x, b, res = x * 0.05, b * 0.05, (0.05 * torch.randn((M, N), generator=gen)).to(dtype)
    gamma, beta = (1 + 0.1 * torch.randn((N,), generator=gen)).to(dtype), (0.1 * torch.randn((N,), generator=gen)).to(dtype)
    xd, rd, wd, bd = _cut(x, 16), _cut(res, 8), w.cuda(), b.cuda()
    rstd = None
    with torch.no_grad():
        if finish == _lib.FINISH_RESIDUAL:
            out = wrappers.linear_residual_wrapper(xd, wd, bd, rd)
        elif finish == _lib.FINISH_RMS_STATS:
            out, rstd = wrappers.linear_residual_stats_wrapper(xd, wd, bd, rd, eps)
        else:
            out = wrappers.linear_add_layer_norm_wrapper(xd, wd, bd, rd, (N,), gamma.cuda(), beta.cuda(), eps)
    used = 0.0 if finish == _lib.FINISH_RESIDUAL else effective_eps(eps, dtype)
    assert finished == [(used, finish, K + 16, N + 8)]
    assert out.shape == rd.shape
    y, out = linear_oracle(x, w, b, "").float(), out.reshape(M, N)
    if finish == _lib.FINISH_LAYER_NORM:
        close(out, layer_norm_oracle(y + res.float(), gamma.float(), beta.float(), used), dtype, what="norm")
        return
    close(out, y + res.float(), dtype, what="sum")
    if rstd is not None:
        expect = torch.rsqrt(out.float().square().mean(-1) + used)
        assert (rstd - expect).abs().max().item() <= 1e-5 * expect.max().item()  # fp32 sums of N squares in another order, N 2^-24 at worst
