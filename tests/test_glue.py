"""What surrounds the kernels of a captured encoder (csrc/glue.hip): the copies of its inputs, its mask and its token types."""
import pytest
import torch

from kernl_amd import _lib


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [[1], [15, 16, 17], [16384, 16383, 16385, 3], [40000, 1, 0, 4096, 5, 6, 7, 70001]], ids=str)
def test_copies_of_all_inputs_in_one_launch(sizes):
    src = [torch.randint(0, 255, (n,), dtype=torch.uint8, device="cuda") for n in sizes]
    dst = [torch.zeros(n + 16, dtype=torch.uint8, device="cuda")[:n] for n in sizes]
    assert _lib.host().copy_many(dst, src) is True
    for d, s, n in zip(dst, src, sizes):
        assert torch.equal(d, s)
        assert not d.as_strided((16,), (1,), n).any()


@pytest.mark.gpu
def test_inputs_that_need_more_than_a_plain_copy_are_left_to_torch():
    x = torch.arange(64, device="cuda")
    for dst, src in (([x.clone()], [x.int()]), ([x.clone()], [x.cpu()]), ([x.clone()[:32]], [x[::2]]), ([x[:32], x[32:]], [x[32:], x[:32]]),
                     ([x.clone()[1:]], [x[1:]]), ([torch.empty_like(x)] * 9, [x] * 9)):
        before = [d.clone() for d in dst]
        assert _lib.host().copy_many(dst, src) is None
        assert all(torch.equal(d, b) for d, b in zip(dst, before))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32], ids=str)
@pytest.mark.parametrize("mask_dtype", [torch.bool, torch.uint8, torch.int32, torch.int64], ids=str)
@pytest.mark.parametrize("shape", [(1, 1), (3, 85), (2, 128), (0, 4), (7, 513)], ids=str)
def test_mask_selection(shape, mask_dtype, dtype):
    from kernl_amd.optimizer.mask import select_mask

    mask = torch.randint(0, 2, shape).to(mask_dtype)
    if mask_dtype == torch.int64:
        mask = mask << 32  # no look at the low half only
    for off in (float("-inf"), torch.finfo(dtype).min):
        out = select_mask(mask.cuda(), 0.0, off, dtype)
        want = torch.where(mask.bool(), torch.zeros((), dtype=dtype), torch.full((), off, dtype=dtype))
        assert out.dtype == dtype and torch.equal(out.cpu(), want)
        assert torch.equal(select_mask(mask, 0.0, off, dtype), want)


def test_token_types_gathered_at_the_position_ids_stay_gathered():
    """A position id outside the token-type buffer is torch.gather's to refuse: the lookups that follow it must not replace it."""
    from kernl_amd.optimizer.dynamo_backend import dynamo_backend_ofi
    from kernl_amd.optimizer.layer_norm import embedding_layer_norm_wrapper

    class Embeddings(torch.nn.Module):
        def __init__(self):
            super().__init__()
            self.words, self.types, self.places = (torch.nn.Parameter(torch.randn(n, 32)) for n in (50, 2, 16))
            self.weight, self.bias = torch.nn.Parameter(torch.ones(32)), torch.nn.Parameter(torch.zeros(32))
            self.register_buffer("type_ids", torch.zeros(1, 16, dtype=torch.long))

        def forward(self, ids, position_ids):
            types = torch.gather(self.type_ids.expand(1, -1), dim=1, index=position_ids).expand(3, 7)
            lookup = torch.nn.functional.embedding
            total = lookup(ids, self.words) + lookup(types, self.types) + lookup(position_ids, self.places)
            return torch.nn.functional.layer_norm(total, (32,), self.weight, self.bias, 1e-5)

    gm = torch.fx.symbolic_trace(Embeddings())
    dynamo_backend_ofi(gm)
    targets = [n.target for n in gm.graph.nodes if n.op == "call_function"]
    assert embedding_layer_norm_wrapper in targets and torch.gather in targets


def test_mask_selection_pass_leaves_other_readers_alone():
    from kernl_amd.optimizer.mask import fuse_mask_selection, select_mask

    class Model(torch.nn.Module):
        def __init__(self, shared):
            super().__init__()
            self.shared = shared

        def forward(self, mask):
            keep = mask.to(torch.bool)
            additive = torch.where(keep.reshape(2, 1, 1, 5), 0.0, -65504.0)
            return (additive, keep) if self.shared else additive

    mask = torch.tensor([[1, 1, 0, 1, 0], [0, 1, 1, 1, 3]])
    for shared in (False, True):
        model = Model(shared)
        gm = torch.fx.symbolic_trace(model)
        next(n for n in gm.graph.nodes if n.op == "placeholder").meta["example_value"] = mask
        fuse_mask_selection(gm)
        assert any(n.target is select_mask for n in gm.graph.nodes) == (not shared)
        got, want = gm(mask), model(mask)
        for g, w in zip((got if shared else (got,)), (want if shared else (want,))):
            assert g.dtype == w.dtype and torch.equal(g, w)


def _fused_selection(forward, mask):
    """The graph of `forward` after the pass, and whether the pass took the selection."""
    from kernl_amd.optimizer.mask import fuse_mask_selection, select_mask

    class Model(torch.nn.Module):
        def forward(self, mask):
            return forward(mask)

    gm = torch.fx.symbolic_trace(Model())
    next(n for n in gm.graph.nodes if n.op == "placeholder").meta["example_value"] = mask
    fuse_mask_selection(gm)
    return gm, any(n.target is select_mask for n in gm.graph.nodes)


@pytest.mark.parametrize("on, off, fused", [(0.0, -65504.0, True), (1, 0, False), (16777217, 0, False), (0, -65504.0, False),
                                            (True, False, False)], ids=str)
def test_only_selections_between_floats_are_fused(on, off, fused):
    """A selection between integers keeps its integer type (positions are counted with such masks) and all their bits."""
    mask = torch.tensor([[1, 1, 0, 1, 0], [0, 1, 1, 1, 3]])
    gm, taken = _fused_selection(lambda m: torch.where(m.to(torch.bool), on, off), mask)
    want = torch.where(mask.to(torch.bool), on, off)
    assert taken == fused and gm(mask).dtype == want.dtype and torch.equal(gm(mask), want)


@pytest.mark.parametrize("convert, fused", [
    (lambda m: m.to(torch.bool), True),
    (lambda m: m.to(dtype=torch.bool), True),
    (lambda m: m.to(device=torch.device("cpu"), dtype=torch.bool), True),
    (lambda m: m.to("cpu", torch.bool), True),
    (lambda m: m.to(device=torch.device("meta"), dtype=torch.bool), False),
    (lambda m: m.to("meta", torch.bool), False),
    (lambda m: m.to(torch.bool, False), False),
    (lambda m: m.to(torch.bool, copy=True), False),
], ids=str)
def test_conversions_that_move_the_mask_are_left_alone(convert, fused):
    mask = torch.tensor([[1, 1, 0, 1, 0], [0, 1, 1, 1, 3]])
    gm, taken = _fused_selection(lambda m: torch.where(convert(m).reshape(2, 1, 1, 5), 0.0, -65504.0), mask)
    want = torch.where(convert(mask).reshape(2, 1, 1, 5), 0.0, -65504.0)
    got = gm(mask)
    assert taken == fused and got.device == want.device and got.dtype == want.dtype and got.shape == want.shape
    assert want.is_meta or torch.equal(got, want)


# masks that are not contiguous: sliced out of a longer one, columns and rows; every other column; transposed
LAYOUTS = {"columns": lambda m: m[:, :7], "rows": lambda m: m[1:3, 2:], "steps": lambda m: m[:, ::2], "transposed": lambda m: m.t(),
           "expanded": lambda m: m[:, :1].expand(4, 5), "four": lambda m: m[:, None, None, :5]}


def _check_selection_of_a_layout(layout, device, dtype):
    from kernl_amd.optimizer.mask import select_mask

    mask = LAYOUTS[layout](torch.tensor([[1, 0, 3, 0, 1, 1, 0, 1 << 33, 0]] * 3 + [[0] * 9], device=device))
    assert not mask.is_contiguous()
    want = torch.where(mask.to(torch.bool), *(torch.full((), v, dtype=dtype, device=device) for v in (0.0, -1e4)))
    got = select_mask(mask, 0.0, -1e4, dtype)
    assert got.dtype == dtype and torch.equal(got, want) and got.stride() == want.stride()


@pytest.mark.parametrize("layout", LAYOUTS)
def test_selection_of_masks_that_are_not_contiguous(layout, monkeypatch):
    def host_tensor(*args, **kwargs):
        raise AssertionError("a copy from the host, which stream capture refuses")

    with monkeypatch.context() as patch:
        patch.setattr("kernl_amd.optimizer.mask.torch.tensor", host_tensor)
        from kernl_amd.optimizer.mask import select_mask

        select_mask(torch.ones(4, 9, dtype=torch.long)[:, :7], 0.0, -1.0, torch.float16)
    for dtype in (torch.float16, torch.float32, torch.float64):
        _check_selection_of_a_layout(layout, "cpu", dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32, torch.float64], ids=str)
@pytest.mark.parametrize("layout", LAYOUTS)
def test_selection_of_masks_that_are_not_contiguous_on_the_gpu(layout, dtype):
    _check_selection_of_a_layout(layout, "cuda", dtype)


def test_selections_outside_the_kernels_types_are_left_alone():
    mask = torch.tensor([[1, 0, 1]])
    before = torch.get_default_dtype()
    torch.set_default_dtype(torch.float64)
    try:
        gm, taken = _fused_selection(lambda m: torch.where(m.to(torch.bool), 0.0, -1e300), mask)
        assert not taken and torch.equal(gm(mask), torch.tensor([[0.0, -1e300, 0.0]]))
    finally:
        torch.set_default_dtype(before)
    gm, taken = _fused_selection(lambda m: torch.where(m.to(torch.bool).view(torch.int8) == 1, 0.0, -1.0), mask)
    assert not taken and torch.equal(gm(mask), torch.tensor([[0.0, -1.0, 0.0]]))


@pytest.mark.gpu
@pytest.mark.parametrize("batch, seq", [(1, 33), (3, 77)], ids=str)
def test_encoder_with_a_mask_sliced_out_of_a_longer_one(batch, seq):
    """What a loop over batches of a tokenizer with a fixed length hands over; captured, so nothing may synchronise."""
    from transformers import BertConfig, BertModel

    from kernl_amd.model_optimization import optimize_model

    torch._dynamo.reset()
    cfg = BertConfig(num_hidden_layers=1)
    cfg._attn_implementation = "eager"
    torch.manual_seed(0)
    model = BertModel(cfg).eval().half().cuda()
    ids = torch.randint(0, 30522, (batch, 128), device="cuda")
    full = (torch.arange(128, device="cuda")[None, :] < torch.randint(seq // 2, seq + 1, (batch, 1), device="cuda")).long()
    with torch.inference_mode():
        optimize_model(model)
        want = model(input_ids=ids[:, :seq].contiguous(), attention_mask=full[:, :seq].contiguous()).last_hidden_state.clone()
        for _ in range(2):
            got = model(input_ids=ids[:, :seq], attention_mask=full[:, :seq]).last_hidden_state
            assert torch.equal(got, want)
