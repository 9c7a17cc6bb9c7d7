"""Tables of the rotary position embedding in one launch: the graph pass and `kernl_rope_tables` against the operations they replace."""
import pytest
import torch

from kernl_amd.implementations.rotary import rotary_tables
from kernl_amd.optimizer.rotary import fuse_rotary_tables


def _eager(inv_freq, positions, scale, dtype):
    a = (inv_freq.float() @ positions.float()).transpose(1, 2)
    e = torch.cat((a, a), dim=-1)
    return (e.cos() * scale).to(dtype), (e.sin() * scale).to(dtype)


def _graph(fn, *inputs):
    """The traced graph with the example values that TorchDynamo leaves on its nodes."""
    gm = torch.fx.symbolic_trace(fn)

    class Recorder(torch.fx.Interpreter):
        def run_node(self, n):
            n.meta["example_value"] = super().run_node(n)
            return n.meta["example_value"]

    Recorder(gm).run(*inputs)
    return gm


def _other_reader(inv, pos):
    a = (inv.float() @ pos.float()).transpose(1, 2)
    e = torch.cat((a, a), dim=-1)
    return e.cos(), e.sin(), e + 1


def _unlike_halves(inv, pos):
    a = (inv.float() @ pos.float()).transpose(1, 2)
    e = torch.cat((a, a + 1), dim=-1)
    return e.cos(), e.sin()


def _unlike_scales(inv, pos):
    a = (inv.float() @ pos.float()).transpose(1, 2)
    e = torch.cat((a, a), dim=-1)
    return e.cos() * 2.0, e.sin()


@pytest.mark.parametrize("fn, fused", [
    (lambda inv, pos: _eager(inv, pos, 1.0, torch.float16), True), (lambda inv, pos: _eager(inv, pos, 0.5, torch.float32), True),
    (_other_reader, False), (_unlike_halves, False), (_unlike_scales, False)], ids=["fp16", "fp32", "other reader", "halves", "scales"])
def test_pass(fn, fused):
    inv, pos = torch.rand(1, 8, 1).half(), torch.arange(9)[None, None]
    gm = _graph(fn, inv, pos)
    expect = gm(inv, pos)
    fuse_rotary_tables(gm)
    names = [getattr(n.target, "__name__", n.target) for n in gm.graph.nodes]
    assert ("rotary_tables_wrapper" in names) == fused and ("cat" in names) != fused and ("float" in names) != fused
    assert all(torch.equal(a, b) for a, b in zip(gm(inv, pos), expect))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32], ids=["fp16", "bf16", "fp32"])
@pytest.mark.parametrize("inv_dtype", [torch.float16, torch.float32], ids=["inv16", "inv32"])
# one frequency; an odd number; one row of either for all; positions far out, where the argument reduction is the long one
@pytest.mark.parametrize("batch, positions, half, start", [((1, 1), 1, 1, 0), ((3, 1), 77, 5, 1 << 20), ((1, 2), 333, 64, 0), ((2, 2), 2048, 64, 5)], ids=str)
def test_kernel(batch, positions, half, start, inv_dtype, dtype):
    inv = (10000.0 ** -(torch.arange(half).float() / half))[None, :, None].expand(batch[0], half, 1).to(inv_dtype).cuda()
    pos = (start + torch.arange(positions))[None, None].repeat(batch[1], 1, 1).cuda()
    # the same operations on the device: the angle is one rounded product on both sides and the functions are the same ones, so the
    # results are equal; the strided operands (an expanded batch, positions of every other column) must not change that
    wide = torch.stack((pos, pos), dim=-1).flatten(-2)[..., ::2]
    for p in (pos, wide, pos.float()):
        got, want = rotary_tables(inv, p, 0.75, dtype), _eager(inv, p, 0.75, dtype)
        assert all(torch.equal(g, w) and g.shape == w.shape for g, w in zip(got, want))
