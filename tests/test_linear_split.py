"""Products with K split over several workgroups a tile and the launch that finishes their rows (csrc/linear_mid.hip, linear_finish.hip)."""
import pytest
import torch

from kernl_amd import _lib
from kernl_amd.implementations.split_linear import split_finish_bytes, split_finish_linear
from oracle import layer_norm_oracle, linear_oracle

pytestmark = pytest.mark.gpu


def _case(M, N, K, dtype, seed=0):
    gen = torch.Generator().manual_seed(seed)
    x, w = torch.randn((M, K), generator=gen).to(dtype), (torch.randn((N, K), generator=gen) * K ** -0.5).to(dtype)
    return x, w, (0.3 * torch.randn((N,), generator=gen)).to(dtype), torch.randn((M, N), generator=gen).to(dtype), gen


# a workgroup a row of up to 1024 columns (231, 500, 130 rows), of up to 4096, of up to 8192; a wave a row beyond 1024 rows of up to 768 and of
# up to 1024 columns; ragged rows, a K that ends inside a k-tile, ranges of unequal length; two to eight ranges, on each of the tiles
SHAPES = [(231, 768, 3072), (500, 772, 3080), (130, 1024, 4096), (333, 4096, 4096), (200, 4100, 11008), (140, 8192, 4104),
          (100, 768, 3072), (150, 4096, 11008), (1500, 768, 4096), (1400, 1024, 4096), (3000, 768, 8192), (2000, 512, 8192)]
# where the residual alone pays for a split: long K
RESIDUAL_SHAPES = [(100, 4096, 11008), (150, 4096, 11008), (200, 4100, 11008), (700, 1024, 11008), (1500, 1024, 8192), (2000, 512, 8192), (2079, 1024, 11008)]
FINISHES = ([(_lib.FINISH_RESIDUAL, shape) for shape in RESIDUAL_SHAPES] + [(_lib.FINISH_RMS_STATS, shape) for shape in SHAPES]
            + [(_lib.FINISH_LAYER_NORM, shape) for shape in SHAPES])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("finish, shape", FINISHES, ids=lambda v: ("residual", "stats", "norm")[v - 1] if isinstance(v, int) else "x".join(map(str, v)))
def test_finished_rows(finish, shape, dtype, close):
    M, N, K = shape
    x, w, b, res, gen = _case(M, N, K, dtype, M)
    gamma, beta = (1 + 0.1 * torch.randn((N,), generator=gen)).to(dtype), (0.1 * torch.randn((N,), generator=gen)).to(dtype)
    need = _lib.linear_split_workspace_bytes(M, N, K, finish)
    assert need > 0, "the shape lists are meant for the split form"
    out = torch.full((M, N + 4), float("nan"), dtype=dtype, device="cuda")[:, :N]
    rstd = torch.full((M,), float("nan"), device="cuda")
    ws = torch.full((need // 4,), float("nan"), device="cuda")
    _lib.linear_split_fwd(x.cuda(), w.cuda(), b.cuda(), res.cuda(), gamma.cuda(), beta.cuda(), 1.6e-5, out, rstd, ws, finish)
    torch.cuda.synchronize()
    y = linear_oracle(x, w, b, "").float()
    if finish == _lib.FINISH_LAYER_NORM:
        close(out, layer_norm_oracle(y + res.float(), gamma.float(), beta.float(), 1.6e-5), dtype, what=f"{shape}")
        return
    close(out, y + res.float(), dtype, scale="magnitude", what=f"{shape}")
    if finish == _lib.FINISH_RMS_STATS:
        ref = torch.rsqrt(out.float().square().mean(-1) + 1.6e-5)
        assert (rstd - ref).abs().max().item() <= 1e-5 * ref.max().item()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("shape", [(140, 12288, 4096), (150, 4096, 11008)], ids=str)  # 192 x 96 and 192 x 128 tiles, two and eight ranges
def test_plain_sums(shape, dtype, close):
    M, N, K = shape
    x, w, b, _, _ = _case(M, N, K, dtype, M)
    need = _lib.linear_split_workspace_bytes(M, N, K)
    assert need > 0
    out, saved = torch.full((2, M, N), float("nan"), dtype=dtype, device="cuda")
    _lib.linear_splitk_fwd(x.cuda(), w.cuda(), b.cuda(), out, saved, _lib.ACT_SILU, torch.full((need // 4,), float("nan"), device="cuda"))
    torch.cuda.synchronize()
    close(out, linear_oracle(x, w, b, "silu"), dtype, scale="magnitude", what=f"{shape}")
    close(saved, linear_oracle(x, w, b, ""), dtype, what=f"{shape} pre-activation")


def test_the_operands_it_leaves_to_other_routes():
    x, w, b, res, _ = _case(231, 768, 3072, torch.float16)
    x, w, b, res = x.cuda(), w.cuda(), b.cuda(), res.cuda()
    stats = _lib.FINISH_RMS_STATS
    assert split_finish_bytes(x, w, b, res, stats) > 0
    assert split_finish_bytes(x, w, b, res[:, :1], stats) == 0                       # a residual that broadcasts
    assert split_finish_bytes(x, w, b, res.float(), stats) == 0
    assert split_finish_bytes(x, w.t().contiguous().t(), b, res, stats) == 0         # a weight that is not contiguous
    assert split_finish_bytes(x.t().contiguous().t(), w, b, res, stats) == 0
    assert split_finish_bytes(x, w, b, res, _lib.FINISH_LAYER_NORM) == 0             # no gamma
    assert split_finish_bytes(x[:60], w, b, res[:60], stats) == 0                    # few rows
    w.requires_grad_()
    assert split_finish_bytes(x, w, b, res, stats) == 0
    with torch.no_grad():
        assert split_finish_bytes(x, w, b, res, stats) > 0
    with torch.autocast("cuda"):
        assert split_finish_bytes(x, w.detach(), b, res, stats) == 0


def test_error_against_64_bits():
    """The split add + LayerNorm is no further from the 64-bit result than the linear kernel followed by the add + LayerNorm kernel."""
    from kernl_amd.implementations.layer_norm import add_layer_norm
    from kernl_amd.implementations.linear_layer import linear_layer

    for M, N, K in ((231, 768, 3072), (500, 768, 3072)):
        x, w, b, res, gen = _case(M, N, K, torch.float16, 9)
        gamma, beta = (1 + 0.1 * torch.randn((N,), generator=gen)).half().cuda(), (0.1 * torch.randn((N,), generator=gen)).half().cuda()
        x, w, b, res = x.cuda(), w.cuda(), b.cuda(), res.cuda()
        s = x.double() @ w.double().T + b.double() + res.double()
        ref = torch.nn.functional.layer_norm(s, (N,), gamma.double(), beta.double(), 1.6e-5)
        need = split_finish_bytes(x, w, b, res, _lib.FINISH_LAYER_NORM, gamma, beta)
        assert need > 0
        fused = split_finish_linear(need, x, w, b, res, _lib.FINISH_LAYER_NORM, gamma, beta, 1.6e-5)
        two = add_layer_norm(linear_layer(x, w, b, ""), res, gamma, beta, 1e-12)
        err = lambda t: ((t.double() - ref).norm() / ref.norm()).item()  # noqa: E731
        assert err(fused) <= err(two)
