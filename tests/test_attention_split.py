"""The attention kernel whose waves split every key tile (csrc/attention_split.hip), forced and on the route that takes it."""
import pytest
import torch

from kernl_amd import _lib
from kernl_amd.implementations.attention import attention_forward
from oracle import attention_oracle

pytestmark = pytest.mark.gpu


@pytest.fixture
def variant():
    lib = _lib.load()
    yield lib.kernl_attention_set_variant
    lib.kernl_attention_set_variant(0)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("which", [0, 7], ids=["route", "forced"])
@pytest.mark.parametrize("head", [64, 128])
# one ragged tile; keys that end inside a key group; rows that see no key of some groups; new rows over a cache; more keys than rows
@pytest.mark.parametrize("rows, keys, start", [(1, 1, 0), (70, 70, 0), (129, 300, 171), (333, 333, 0), (40, 515, 475), (257, 700, 100), (640, 640, 0)], ids=str)
def test_against_the_oracle(rows, keys, start, head, which, dtype, variant, close):
    gen = torch.Generator().manual_seed(rows + head)
    q = torch.randn((2, 3, rows, head), generator=gen).to(dtype)
    k, v = (torch.randn((2, 3, keys, head), generator=gen).to(dtype) for _ in range(2))
    out = torch.full((2, 3, rows, head), float("nan"), dtype=dtype, device="cuda")
    variant(which)
    attention_forward(q.cuda(), k.cuda(), v.cuda(), out, head ** -0.5, True, None, start_position=start)
    torch.cuda.synchronize()
    close(out, attention_oracle(q, k, v, head ** -0.5, True, None, start_position=start), dtype, what=f"{which} {rows}x{keys}")


def test_references_that_move_and_strided_operands(variant, close):
    """Scores that grow along the keys move the rows' references again and again; heads interleaved with positions, as projections leave them."""
    gen = torch.Generator().manual_seed(3)
    packed = torch.randn((2, 400, 3, 4, 64), generator=gen)
    packed[:, :, 1] *= torch.linspace(0.1, 6.0, 400)[None, :, None, None]
    packed = packed.half()
    q, k, v = (packed[:, :, i].transpose(1, 2) for i in range(3))
    dev = packed.cuda()
    dq, dk, dv = (dev[:, :, i].transpose(1, 2) for i in range(3))
    out = torch.empty((2, 400, 4, 64), dtype=torch.float16, device="cuda").transpose(1, 2)
    variant(7)
    attention_forward(dq, dk, dv, out, 0.125, True, None)
    torch.cuda.synchronize()
    close(out, attention_oracle(q, k, v, 0.125, True, None), what="growing scores")


@pytest.mark.parametrize("which", [3, 4], ids=["streaming", "pipelined"])
@pytest.mark.parametrize("heads, rows", [(3, 260), (128, 130), (131, 140), (265, 257)], ids=str)  # one head an XCD; 16; 17 (a short group); 34
def test_every_query_tile_of_ranked_grids(heads, rows, which, variant, close):
    """The longest-first orders of the causal kernels: every (head, query tile) once, whatever the heads of an XCD and of its last group."""
    gen = torch.Generator().manual_seed(heads)
    q, k, v = (torch.randn((1, heads, rows, 64), generator=gen).half() for _ in range(3))
    out = torch.full((1, heads, rows, 64), float("nan"), dtype=torch.float16, device="cuda")
    variant(which)
    attention_forward(q.cuda(), k.cuda(), v.cuda(), out, 0.125, True, None)
    torch.cuda.synchronize()
    close(out, attention_oracle(q, k, v, 0.125, True, None), what=f"{which} {heads}x{rows}")
