"""linear + residual + LayerNorm in one launch, the rows' statistics exchanged between workgroups (csrc/norm_exchange.h)."""
import pytest
import torch

from kernl_amd import _lib
from kernl_amd.implementations.exchanged_norm import ExchangeRegions, exchange_bytes, linear_add_norm
from kernl_amd.optimizer import linear as wrappers
from oracle import effective_eps, layer_norm_oracle, linear_oracle

DTYPES = pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
# for each tile the fewest rows that take it, the most of one round, and an odd number between; K that ends inside a k-tile; one workgroup a row
# tile's columns and 24 of them
SHAPES = [(65, 768, 768), (170, 768, 3072), (171, 768, 776), (341, 768, 768), (128, 1024, 4096), (600, 512, 2048), (342, 768, 768), (1365, 768, 768),
          (682, 768, 3072), (1366, 768, 768), (2730, 768, 768), (2731, 768, 776), (5461, 768, 768), (5462, 768, 768), (8192, 768, 768),
          (8193, 768, 768), (10922, 768, 768), (10923, 768, 768), (12288, 768, 768), (16384, 384, 768), (300, 128, 64),
          # the wide kernel: 256 x 192 tiles, then 256 x 256
          (12289, 768, 136), (16384, 768, 64), (16385, 768, 200), (21760, 768, 64), (8193, 1024, 136), (16384, 1024, 64), (32768, 512, 64)]


def _operands(M, N, K, dtype):
    gen = torch.Generator().manual_seed(M + K)
    x, w = torch.randn((M, K), generator=gen).to(dtype), (torch.randn((N, K), generator=gen) * K ** -0.5).to(dtype)
    b, res = (0.3 * torch.randn((N,), generator=gen)).to(dtype), torch.randn((M, N), generator=gen).to(dtype)
    return x, w, b, res, (1 + 0.1 * torch.randn((N,), generator=gen)).to(dtype), (0.1 * torch.randn((N,), generator=gen)).to(dtype)


def _expected(x, w, b, res, gamma, beta, eps=1.6e-5):
    beta = beta.float() if beta is not None else torch.zeros_like(gamma.float())
    return layer_norm_oracle(linear_oracle(x, w, b, "").float() + res.float(), gamma.float(), beta, eps)


@pytest.mark.gpu
@DTYPES
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_rows(shape, dtype, close):
    M, N, K = shape
    ops = _operands(M, N, K, dtype)
    need = _lib.linear_exchange_bytes(M, N, K)
    assert need > 0, "the shape list is meant for this launch"
    dev = [t.cuda() for t in ops]
    expected, sums = _expected(*ops), torch.empty((M, N), device="cuda")
    # 0: every workgroup that does not find all words at its first look leaves, and the last ones finish the tiles of the others
    first = None
    for patience in (-1, 0, 1):
        regions = [torch.zeros(need // 8, dtype=torch.int64, device="cuda"), torch.full((need // 8,), -1, dtype=torch.int64, device="cuda")]
        for _ in range(3):
            out = torch.full((M, N + 8), float("nan"), dtype=dtype, device="cuda")[:, :N]
            sums.fill_(float("nan"))
            _lib.linear_add_norm_fwd(*dev[:4], *dev[4:], 1.6e-5, out, sums, *regions, patience)
            regions.reverse()
            torch.cuda.synchronize()
            assert (regions[0] == 0).all(), "the region of the next launch"
            if first is None:
                close(out, expected, dtype, what=f"{shape}")
                first = out
            assert torch.equal(out, first), f"patience {patience}: the same rows whoever finishes them"


@pytest.mark.gpu
@DTYPES
def test_wrapper_with_rows_cut_out_of_wider_ones(dtype, close):
    x, w, b, res, gamma, beta = _operands(300, 768, 768, dtype)

    def cut(t, extra):
        wide = torch.full((3, 100, t.shape[1] + extra), float("nan"), dtype=dtype, device="cuda")
        wide[..., :t.shape[1]] = t.view(3, 100, -1).cuda()
        return wide[..., :t.shape[1]]

    regions = ExchangeRegions()
    for bias, shift in ((b.cuda(), beta.cuda()), (None, None)):
        out = wrappers.linear_add_layer_norm_wrapper(cut(x, 8), w.cuda(), bias, cut(res, 16), (768,), gamma.cuda(), shift, 1e-12, regions=regions)
        torch.cuda.synchronize()
        expected = _expected(x, w, b if bias is not None else None, res, gamma, beta if bias is not None else None, effective_eps(1e-12, dtype))
        close(out.reshape(300, 768), expected, dtype, what="cut rows")
    assert regions._pair is not None, "the launch this test is about"


@pytest.mark.gpu
def test_a_captured_chain_replays():
    """Layers of different tiles take the regions by turns, and every replay starts from zeros of its own."""
    ops = [_operands(M, 768, K, torch.float16) for M, K in ((300, 768), (300, 3072), (300, 768))]
    dev = [[t.cuda() for t in o] for o in ops]
    x = dev[0][0].clone()

    def chain():
        regions, h = ExchangeRegions(), []
        for o in dev:
            inp = x if o[0].shape[1] == 768 else o[0]
            h.append(linear_add_norm(exchange_bytes(inp, *o[1:]), regions, inp, *o[1:], 1.6e-5))
        return h

    chain()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = chain()
    for seed in range(4):
        x.copy_(torch.randn((300, 768), generator=torch.Generator().manual_seed(seed)))
        graph.replay()
        torch.cuda.synchronize()
        replayed = [t.clone() for t in captured]
        assert all(torch.equal(a, b) for a, b in zip(replayed, chain())), f"replay {seed}"


@pytest.mark.gpu
def test_the_operands_it_leaves_to_other_routes():
    x, w, b, res, gamma, beta = (t.cuda() for t in _operands(300, 768, 768, torch.float16))
    assert exchange_bytes(x, w, b, res, gamma, beta) > 0
    assert exchange_bytes(x[:64], w, b, res[:64], gamma, beta) == 0
    assert exchange_bytes(x, w, b, res.float(), gamma, beta) == 0
    assert exchange_bytes(x, w, b, res[:, :1], gamma, beta) == 0
    assert exchange_bytes(x, w, b, res, None, None) == 0
    assert exchange_bytes(x.t().contiguous().t(), w, b, res, gamma, beta) == 0
    assert exchange_bytes(x, w, b, res.t().contiguous().t(), gamma, beta) == 0
    assert exchange_bytes(x, w.requires_grad_(), b, res, gamma, beta) == 0
    with pytest.raises(RuntimeError, match="region"):
        few = torch.zeros(8, dtype=torch.int64, device="cuda")
        _lib.linear_add_norm_fwd(x, w, b, res, gamma, beta, 1e-5, torch.empty_like(res), torch.empty((300, 768), device="cuda"), few, few.clone())


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(300, 768, 768), (1024, 768, 3072), (4096, 768, 768)], ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("mean", [0.0, 10.0])
def test_error_against_64_bits(shape, mean):
    """No further from the result in 64 bits than product and LayerNorm as two launches, also where the rows' mean is far from zero."""
    x, w, b, res, gamma, beta = _operands(*shape, torch.float16)
    res = (res.float() + mean).half()
    dev = [t.cuda() for t in (x, w, b, res, gamma, beta)]
    exact = torch.nn.functional.layer_norm(dev[0].double() @ dev[1].double().t() + dev[2].double() + dev[3].double(), (shape[1],),
                                           dev[4].double(), dev[5].double(), 1.6e-5)
    error = lambda t: ((t.double() - exact).norm() / exact.norm()).item()  # noqa: E731
    one = linear_add_norm(exchange_bytes(*dev), ExchangeRegions(), *dev, 1.6e-5)
    two = wrappers.linear_add_layer_norm_wrapper(*dev[:4], (shape[1],), *dev[4:], 1e-12)
    assert error(one) <= 1.02 * error(two)  # (both round the result to 16 bits: half an ulp is what they share)


def test_every_order_of_events_normalises_every_tile():
    """The protocol of three workgroups of a row, each with no patience, in every order of their steps: publish, look; then either finish and
    read the notes, or store the sums, leave a note and look once more."""
    memo = set()

    def walk(state):
        if state in memo:
            return
        memo.add(state)
        steps, found, published, notes, written = state
        if all(s == 5 for s in steps):
            assert written == frozenset({0, 1, 2}), state
            return
        for who in range(3):
            s = steps[who]
            if s == 5:
                continue
            f, p, n, w = list(found), published, notes, written
            if s == 0:
                p = p | {who}
            elif s in (1, 3) and not f[who]:
                f[who] = len(p) == 3
            elif s == 2 and not f[who]:
                n = n | {who}
            elif s == 4 and f[who]:
                w = w | {who} | n
            walk((steps[:who] + (s + 1,) + steps[who + 1:], tuple(f), p, n, w))

    walk(((0, 0, 0), (False,) * 3, frozenset(), frozenset(), frozenset()))
    assert len(memo) > 100
