"""The tiles of csrc/linear_mid.hip with loading waves: k-tiles dealt among the workgroups that share a weight tile (weights of more
than 8 M elements), and the 192 x 96 tile."""
import pytest
import torch

from kernl_amd import _lib
from oracle import glu_oracle, linear_oracle

pytestmark = pytest.mark.gpu


@pytest.fixture
def force():
    lib = _lib.load()
    yield lib.kernl_linear_force_tile
    lib.kernl_linear_force_tile(0)


@pytest.mark.parametrize("tile", [11, 15, 17, 18, 19, 20, 21, 22])
# one row tile up to many, k-tiles that are no multiple of a dealt group, a ragged last k-tile, groups longer than K
@pytest.mark.parametrize("shape", [(66, 4200, 2056), (333, 4096, 2112), (700, 8200, 1096)], ids=str)
def test_dealt_k_tiles(shape, tile, force, close):
    M, N, K = shape
    gen = torch.Generator().manual_seed(M + tile)
    x, w = torch.randn((M, K), generator=gen).half(), (torch.randn((N, K), generator=gen) * K ** -0.5).half()
    out = torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda")
    force(tile)
    _lib.linear_fwd(x.cuda(), w.cuda(), None, out, None, _lib.ACT_NONE)
    torch.cuda.synchronize()
    close(out, linear_oracle(x, w, None, ""), what=f"tile {tile} {shape}")


@pytest.mark.parametrize("shape", [(65, 70, 8), (193, 97, 64), (385, 390, 520)], ids=str)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
def test_192_x_96_at_its_edges(shape, dtype, force, close):
    M, N, K = shape
    gen = torch.Generator().manual_seed(M)
    x, w = torch.randn((M, K), generator=gen).to(dtype), (torch.randn((N, K), generator=gen) * K ** -0.5).to(dtype)
    b = torch.randn((N,), generator=gen).to(dtype)
    out, saved = torch.full((2, M, N), float("nan"), dtype=dtype, device="cuda")
    force(22)
    _lib.linear_fwd(x.cuda(), w.cuda(), b.cuda(), out, saved, _lib.ACT_GELU_ERF)
    torch.cuda.synchronize()
    close(out, linear_oracle(x, w, b, "gelu"), dtype, what=f"{shape}")
    close(saved, linear_oracle(x, w, b, ""), dtype, what=f"{shape} pre-activation")


def test_gates_with_dealt_k_tiles(force, close):
    from kernl_amd.implementations.linear_layer import interleave_glu_rows

    gen = torch.Generator().manual_seed(5)
    M, N, K = 300, 2112, 2120
    x = torch.randn((M, K), generator=gen).half()
    wg, wv = ((torch.randn((N, K), generator=gen) * K ** -0.5).half() for _ in range(2))
    out = torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda")
    force(19)
    _lib.linear_glu_fwd(x.cuda(), interleave_glu_rows(wg, wv).cuda(), None, out, _lib.ACT_SILU)
    torch.cuda.synchronize()
    close(out, glu_oracle(x, wg, None, wv, None, "silu"), scale="magnitude", what="gated")


@pytest.mark.parametrize("tile", [5, 6, 7, 8])
# whole groups of four k-tiles (dealt), an odd number of groups, and a K that leaves the order as it is
@pytest.mark.parametrize("shape", [(600, 8300, 1024), (300, 4200, 2304), (1100, 4096, 2112)], ids=str)
def test_dealt_k_tiles_of_the_wide_kernels(shape, tile, force, close):
    M, N, K = shape
    gen = torch.Generator().manual_seed(M + tile)
    x, w = torch.randn((M, K), generator=gen).half(), (torch.randn((N, K), generator=gen) * K ** -0.5).half()
    out = torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda")
    force(tile)
    _lib.linear_fwd(x.cuda(), w.cuda(), None, out, None, _lib.ACT_NONE)
    torch.cuda.synchronize()
    close(out, linear_oracle(x, w, None, ""), what=f"tile {tile} {shape}")


@pytest.mark.parametrize("tile", [11, 15, 17, 18, 19, 20, 21, 22])
@pytest.mark.parametrize("K", [8, 64, 128, 192, 200, 256, 264, 320])  # fewer k-tiles than the ring is deep, as many, one and two more
@pytest.mark.parametrize("layout", ["rows", "odd rows", "columns"])   # whole vectors; row strides that no vector has; column-major
def test_short_rings_and_the_epilogues_forms(layout, K, tile, force, close):
    M, N = 200, 208
    gen = torch.Generator().manual_seed(K + tile)
    x, w = torch.randn((M, K), generator=gen).half(), (torch.randn((N, K), generator=gen) * K ** -0.5).half()
    b = torch.randn((N,), generator=gen).half()

    def tensor():
        if layout == "columns":
            return torch.full((N, M), float("nan"), dtype=torch.float16, device="cuda").t()
        return torch.full((M, N + (3 if layout == "odd rows" else 8)), float("nan"), dtype=torch.float16, device="cuda")[:, :N]

    out, saved, plain = tensor(), tensor(), tensor()
    force(tile)
    _lib.linear_fwd(x.cuda(), w.cuda(), b.cuda(), out, saved, _lib.ACT_SILU)
    _lib.linear_fwd(x.cuda(), w.cuda(), b.cuda(), plain, None, _lib.ACT_NONE)
    torch.cuda.synchronize()
    close(out, linear_oracle(x, w, b, "silu"), scale="magnitude", what=f"tile {tile}")
    close(saved, linear_oracle(x, w, b, ""), what=f"tile {tile} pre-activation")
    assert torch.equal(saved, plain)


def _laid(layout, M, N, dtype=torch.float16):
    """[M, N] of NaNs: row strides that no vector has, or column-major."""
    if layout == "columns":
        return torch.full((N, M), float("nan"), dtype=dtype, device="cuda").t()
    return torch.full((M, N + 3), float("nan"), dtype=dtype, device="cuda")[:, :N]


# what the rule gives to 128 x 64, 128 x 128, 192 x 96, 192 x 128 and 192 x 192 tiles, rows and columns ragged
@pytest.mark.parametrize("tile, shape", [(15, (200, 4104, 1536)), (17, (200, 8200, 1536)), (22, (903, 4104, 1536)), (18, (903, 6152, 1536)), (19, (903, 8200, 1536))],
                         ids=str)
@pytest.mark.parametrize("layout", ["odd rows", "columns"])
def test_a_residual_and_results_that_no_vector_takes(layout, tile, shape, close):
    M, N, K = shape
    assert _lib.linear_mid_kind(M, N, K) == tile
    gen = torch.Generator().manual_seed(tile)
    x, w = torch.randn((M, K), generator=gen).half(), (torch.randn((N, K), generator=gen) * K ** -0.5).half()
    b, res = torch.randn((N,), generator=gen).half(), torch.randn((M, N), generator=gen).half()
    out, resd = _laid(layout, M, N), _laid(layout, M, N)
    resd.copy_(res)
    _lib.linear_residual_fwd(x.cuda(), w.cuda(), b.cuda(), resd, out)
    torch.cuda.synchronize()
    close(out, linear_oracle(x, w, b, "").half().float() + res.float(), scale="magnitude", what=f"tile {tile} {layout}")


@pytest.mark.parametrize("tile", [11, 15, 17, 18, 19, 20, 21])
@pytest.mark.parametrize("layout", ["odd rows", "columns"])
def test_gated_results_that_no_vector_takes(layout, tile, force, close):
    from kernl_amd.implementations.linear_layer import interleave_glu_rows

    gen = torch.Generator().manual_seed(tile)
    M, N, K = 201, 224, 264
    x = torch.randn((M, K), generator=gen).half()
    wg, wv = ((torch.randn((N, K), generator=gen) * K ** -0.5).half() for _ in range(2))
    out = _laid(layout, M, N)
    force(tile)
    _lib.linear_glu_fwd(x.cuda(), interleave_glu_rows(wg, wv).cuda(), None, out, _lib.ACT_SILU)
    torch.cuda.synchronize()
    close(out, glu_oracle(x, wg, None, wv, None, "silu"), scale="magnitude", what=f"tile {tile} {layout}")


# (gates run on 256 x 256 tiles only)
@pytest.mark.parametrize("epilogue, tile", [(epilogue, tile) for epilogue in ("residual", "row factors") for tile in (5, 6, 7, 8)] + [("gates", 5)])
def test_dealt_k_tiles_of_the_wide_kernels_with_their_epilogues(epilogue, tile, force, close):
    from kernl_amd.implementations.linear_layer import interleave_glu_rows

    M, N, K = 300, 8256, 1024  # whole groups of four k-tiles, a weight of more than 8 M elements, ragged tiles
    gen = torch.Generator().manual_seed(tile)
    x, w = torch.randn((M, K), generator=gen).half(), (torch.randn((N, K), generator=gen) * K ** -0.5).half()
    b, res, factor = torch.randn((N,), generator=gen).half(), torch.randn((M, N), generator=gen).half(), 0.5 + torch.rand((M,), generator=gen)
    force(tile)
    if epilogue == "gates":
        out = torch.full((M, N // 2), float("nan"), dtype=torch.float16, device="cuda")
        _lib.linear_glu_fwd(x.cuda(), interleave_glu_rows(w[: N // 2], w[N // 2:]).cuda(), None, out, _lib.ACT_SILU)
        expect = glu_oracle(x, w[: N // 2], None, w[N // 2:], None, "silu")
    else:
        out = torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda")
        if epilogue == "residual":
            _lib.linear_residual_fwd(x.cuda(), w.cuda(), b.cuda(), res.cuda(), out)
            expect = linear_oracle(x, w, b, "").half().float() + res.float()
        else:
            _lib.linear_scaled_fwd(x.cuda(), w.cuda(), b.cuda(), factor.cuda(), out, _lib.ACT_NONE, False)
            expect = linear_oracle(x, w, None, "") * factor[:, None] + b.float()
    torch.cuda.synchronize()
    close(out, expect, scale="magnitude", what=f"tile {tile} {epilogue}")


@pytest.mark.parametrize("tile", [17, 18, 7])
def test_equal_rows_in_other_row_tiles(tile, force):
    """The order of the k-tiles, and with it that of the fp32 sums, depends on the row tile: the same row at another place of a batch may
    round to the other neighbour.  The same call gives the same bits."""
    M, N, K = 384, 4160, 2048
    gen = torch.Generator().manual_seed(tile)
    x, w = torch.randn((M, K), generator=gen).half().cuda(), (torch.randn((N, K), generator=gen) * K ** -0.5).half().cuda()
    outs = [torch.full((2 * M, N), float("nan"), dtype=torch.float16, device="cuda") for _ in range(2)]
    force(tile)
    for out in outs:
        _lib.linear_fwd(torch.cat((x, x)), w, None, out, None, _lib.ACT_NONE)
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1])
    first, second = outs[0][:M].float(), outs[0][M:].float()
    # two sums of K products of deviation K^-1/2 in fp32: K 2^-24 = 1.2e-4 of their size at worst, then a rounding to the next value at most
    spacing = 2.0 ** (torch.maximum(first.abs(), second.abs()).clamp_min(2.0 ** -14).log2().floor() - 10)
    assert ((first - second).abs() <= spacing + 1.2e-4 * 4).all()
