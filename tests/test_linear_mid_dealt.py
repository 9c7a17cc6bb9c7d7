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
