"""The 8-wave tiles over the whole K (csrc/linear_mid.hip) and the narrow dealt tiles: every tile forced at its edges, and the
epilogues — gated, row factors, residual, saved pre-activation — at shapes the rule gives to them."""
import pytest
import torch

from kernl_amd import _lib
from oracle import glu_oracle, linear_oracle

TILES = [11, 15, 16, 17, 18, 19, 20, 21]  # 64x64, 128x64, dealt 16x16, 128x128, 192x128, 192x192, 128x256, 256x128


def _case(M, N, K, dtype, seed=0):
    gen = torch.Generator().manual_seed(seed)
    x = torch.randn((M, K), generator=gen).to(dtype)
    w = (torch.randn((N, K), generator=gen) * K ** -0.5).to(dtype)
    return x, w, (0.3 * torch.randn((N,), generator=gen)).to(dtype), gen


@pytest.fixture
def force():
    lib = _lib.load()
    yield lib.kernl_linear_force_tile
    lib.kernl_linear_force_tile(0)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("tile", TILES)
# ragged rows and columns, fewer k-tiles than ring stages, ragged last k-tile, one tile exactly, unaligned output rows
@pytest.mark.parametrize("shape", [(65, 70, 8), (129, 136, 64), (193, 257, 136), (256, 256, 192), (300, 200, 776), (17, 40, 1544), (500, 390, 520)], ids=str)
def test_every_tile_at_its_edges(shape, tile, dtype, force, close):
    M, N, K = shape
    x, w, b, _ = _case(M, N, K, dtype, M)
    xd, wd, bd = x.cuda(), w.cuda(), b.cuda()
    out, saved = torch.full((2, M, N), float("nan"), dtype=dtype, device="cuda")
    force(tile)
    _lib.linear_fwd(xd, wd, bd, out, saved, _lib.ACT_GELU_TANH)
    torch.cuda.synchronize()
    close(out, linear_oracle(x, w, b, "fast_gelu"), dtype, what=f"tile {tile} {shape}")
    close(saved, linear_oracle(x, w, b, ""), dtype, what=f"tile {tile} {shape} pre-activation")
    wide = torch.zeros((M, N + 24), dtype=dtype, device="cuda")
    _lib.linear_fwd(xd, wd, None, wide[:, 8:8 + N], None, _lib.ACT_NONE)
    torch.cuda.synchronize()
    close(wide[:, 8:8 + N], linear_oracle(x, w, None, ""), dtype, what=f"tile {tile} {shape} strided")
    assert (wide[:, :8] == 0).all() and (wide[:, 8 + N:] == 0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("tile", [t for t in TILES if t != 16])
@pytest.mark.parametrize("shape", [(70, 32, 72), (300, 96, 200), (257, 160, 520), (193, 288, 64)], ids=str)
def test_every_gated_tile_at_its_edges(shape, tile, force, close):
    from kernl_amd.implementations.linear_layer import interleave_glu_rows

    M, N, K = shape
    x, wg, bg, gen = _case(M, N, K, torch.float16, tile)
    _, wv, bv, _ = _case(M, N, K, torch.float16, tile + 50)
    out = torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda")
    force(tile)
    _lib.linear_glu_fwd(x.cuda(), interleave_glu_rows(wg, wv).cuda(), interleave_glu_rows(bg, bv).cuda(), out, _lib.ACT_SILU)
    torch.cuda.synchronize()
    close(out, glu_oracle(x, wg, bg, wv, bv, "silu"), scale="magnitude", what=f"gated tile {tile} {shape}")


def test_rule():
    mid = _lib.linear_mid_kind
    assert mid(64, 3072, 768, 0) == 0 and mid(128, 4608, 2048, 0) == 0 and mid(16384, 3072, 768, 0) == 0 and mid(200, 4096, 4100, 0) == 0
    assert mid(768, 3072, 768, 0) == 15 and mid(1024, 2304, 768, 0) == 15 and mid(3072, 768, 768, 0) == 17  # short K
    assert mid(100, 4096, 4096, 0) == 14 and mid(768, 4096, 4096, 0) == 17 and mid(256, 4096, 4096, 0) == 11
    assert mid(130, 22016, 4096, 1) == 18 and mid(256, 22016, 4096, 1) == 21 and mid(333, 22016, 4096, 1) == 19
    assert mid(2048, 22016, 4096, 1) == 0 and mid(2048, 12288, 4096, 0) == 0  # the wide tiles


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("shape", [(1000, 2048, 1536), (700, 4096, 2048), (190, 4096, 4096)], ids=str)
def test_residual_and_row_factors(shape, dtype, close):
    M, N, K = shape
    assert _lib.linear_mid_kind(M, N, K) >= 11 and _lib.linear_small_kind(M, N, K) == 0
    x, w, b, gen = _case(M, N, K, dtype, 3)
    xd, wd, bd = x.cuda(), w.cuda(), b.cuda()
    res = torch.randn((M, N + 8), generator=gen).to(dtype)[:, :N].cuda()
    out = torch.empty((M, N), dtype=dtype, device="cuda")
    plain = torch.empty_like(out)
    _lib.linear_residual_fwd(xd, wd, bd, res, out)
    _lib.linear_fwd(xd, wd, bd, plain, None, _lib.ACT_NONE)
    torch.cuda.synchronize()
    assert torch.equal(out, plain + res)
    factor = torch.rand((M,), generator=gen) + 0.5
    _lib.linear_scaled_fwd(xd, wd, bd, factor.cuda(), out, _lib.ACT_NONE, False)
    torch.cuda.synchronize()
    close(out, linear_oracle(x, w, None, "") * factor[:, None] + b.float(), dtype, what=f"row factors {shape}")


@pytest.mark.gpu
def test_gated_row_factors_and_the_operators_route(close, monkeypatch):
    """A short prompt's gated projection with the norm folded in runs the 8-wave tiles (row factors in their epilogue)."""
    from kernl_amd.implementations import linear_layer as ll

    gen = torch.Generator().manual_seed(4)
    M, N, K = 150, 11008, 2048
    assert _lib.linear_mid_kind(M, 2 * N, K, True) != 0
    x = torch.randn((M, K), generator=gen).half()
    wg, wv = ((torch.randn((N, K), generator=gen) * K ** -0.5).half() for _ in range(2))
    w = ll.interleave_glu_rows(wg, wv).cuda()
    calls = []
    real = _lib.linear_scaled_fwd
    monkeypatch.setattr(_lib, "linear_scaled_fwd", lambda *a, **k: (calls.append(1), real(*a, **k))[1])
    out = ll.rms_linear_layer(x.cuda(), torch.ones(K).half().cuda(), 1e-5, w, None, "silu", gated=True, folded_weight=w)
    torch.cuda.synchronize()
    assert calls == [1]
    normed = x.float() * torch.rsqrt(x.float().square().mean(-1, keepdim=True) + 1.6e-5)
    close(out, glu_oracle(normed.half(), wg, None, wv, None, "silu"), scale="magnitude", what="gated prompt")
