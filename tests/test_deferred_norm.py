"""LayerNorms left to the linear layers behind them (csrc/norm_fold.h): both kernels' forms against 64 bits at the edges of their
tiles, the error of the route against that of the kernels it replaces, and the graph pass."""
import pytest
import torch

from kernl_amd import _lib


def _make(rows, n, k, dtype, seed, scale=1.0, offset=0.0):
    gen = torch.Generator().manual_seed(seed)

    def t(*shape, std=1.0, mean=0.0):
        return (torch.randn(shape, generator=gen) * std + mean).to(dtype).cuda()

    x, w, b = t(rows, k, std=0.5), t(n, k, std=0.03), t(n, std=0.1)
    res, gamma, beta = t(rows, n, std=scale, mean=offset), t(n, std=0.2, mean=1.0), t(n, std=0.2)
    return x, w, b, res, gamma, beta


def _ln(rows, gamma, beta, eps):
    return torch.nn.functional.layer_norm(rows.double(), (rows.shape[-1],), gamma.double(), None if beta is None else beta.double(), eps)


def _error(a, ref):
    return ((a.double() - ref).norm() / ref.norm()).item()


# rows around the tile heights, widths around the groups and the k-tiles: (rows, width, k) of the layer in front of the norm
SHAPES = [(8, 768, 768), (9, 32, 264), (16, 768, 3072), (16, 96, 72), (17, 768, 3072), (31, 416, 768), (33, 1024, 1024), (47, 160, 1536),
          (64, 768, 768), (64, 1024, 4096)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("offset", [0.0, 30.0])
@pytest.mark.parametrize("rows, n, k", SHAPES, ids=str)
def test_both_sides_of_a_deferred_norm(rows, n, k, offset, dtype):
    from kernl_amd.implementations.deferred_norm import linear_add_deferred

    assert _lib.linear_norm_kind(rows, n, k) != 0
    x, w, b, res, gamma, beta = _make(rows, n, k, dtype, rows + n, offset=offset)
    # one rounding to the 16-bit type is at most `unit` of a value, and 1/sqrt(3) of that in the 2-norm
    unit = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    # fp32 sums of k products and a residual: 2^-24 of the largest partial sum per addition, far inside k * 2^-24
    fp32 = 2.0 ** -24 * max(k, n)
    norm = linear_add_deferred(x, w, b, res, gamma, beta, 1e-12)
    s = x.double() @ w.double().T + b.double() + res.double()
    assert norm.rows.dtype == torch.float32 and _error(norm.rows, s) <= fp32
    groups = norm.rows.double().view(rows, n // 16, 16)
    assert torch.allclose(norm.stats[..., 0].double(), groups.sum(-1), rtol=1e-5, atol=1e-3)
    assert torch.allclose(norm.stats[..., 1].double(), groups.var(-1, unbiased=False) * 16, rtol=1e-4, atol=1e-4)
    # a second addition on top of the deferred residual: nothing on the way is rounded to 16 bits
    # (a mean of 30 takes 30 * 2^-24 of the deviations in fp32)
    fp32 *= 1 + offset
    eps = norm.kernel_eps
    h = _ln(s, gamma, beta, eps)
    again = linear_add_deferred(x, w, None, norm, gamma, None, 1e-12)
    assert _error(again.rows, x.double() @ w.double().T + h) <= fp32
    # as a tensor: one rounding
    assert _error(norm.normalised(), h) <= 0.6 * unit + fp32
    # the layers behind: every activation's branch, with and without parameters.  The normalised operand and the result are
    # rounded once each; an activation passes an error of its input on at most 1.13-fold (gelu), and may cut the result's norm (relu, gelu
    # of values around zero) to some 0.6 of its input's.  3072 columns are tiles of 16 x 16, 16 x 32 or 32 x 32, by the rows.
    for width, bias, activation in ((64, None, ""), (96, True, "gelu"), (32, True, "relu"), (256, True, "tanh"), (3072, True, "fast_gelu"), (160, None, "silu")):
        w2, b2 = _make(1, width, n, dtype, 7)[1], (_make(1, width, n, dtype, 7)[2] if bias else None)
        if not norm.takes_linear(w2, b2, activation):
            continue
        ref = h @ w2.double().T + (0 if b2 is None else b2.double())
        act = {"": lambda t: t, "gelu": torch.nn.functional.gelu, "relu": torch.relu, "tanh": torch.tanh, "silu": torch.nn.functional.silu,
               "fast_gelu": lambda t: torch.nn.functional.gelu(t, approximate="tanh")}[activation]
        assert _error(norm.linear(w2, b2, activation), act(ref)) <= (1.2 if activation == "" else 2.5) * unit + fp32, (width, activation)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("offset", [0.0, 3.0, 10.0])
@pytest.mark.parametrize("spread", [0.0, 0.2, 1.0])
def test_no_less_precise_than_the_norm_kernel(offset, spread, dtype):
    """Norm and next projection against 64 bits, rows with a mean and norms with parameters: the deferred route against the linear
    kernel, the add + LayerNorm kernel and the linear kernel.  (5 %: both errors are roundings, equal up to their luck.)"""
    from kernl_amd.implementations.deferred_norm import linear_add_deferred
    from kernl_amd.implementations.layer_norm import add_layer_norm
    from kernl_amd.implementations.linear_layer import linear_layer

    rows, n, k = 48, 768, 768
    x, w, b, res, _, _ = _make(rows, n, k, dtype, 11, offset=offset)
    gen = torch.Generator().manual_seed(5)
    gamma, beta = ((m + spread * torch.randn(n, generator=gen)).to(dtype).cuda() for m in (1.0, 0.0))
    w2 = _make(1, 2304, n, dtype, 7)[1]
    eps = 1.6e-5
    h = _ln(x.double() @ w.double().T + b.double() + res.double(), gamma, beta, eps)
    norm = linear_add_deferred(x, w, b, res, gamma, beta, eps)
    normed = add_layer_norm(linear_layer(x, w, b), res, gamma, beta, eps)
    for ours, theirs, want in ((norm.linear(w2, None), linear_layer(normed, w2, None), h @ w2.double().T), (norm.normalised(), normed, h)):
        assert _error(ours, want) <= 1.05 * _error(theirs, want)


def test_bad_arguments_are_rejected():
    lib, f = _lib.load(), 64  # never dereferenced
    kind, add, apply, rows32 = (getattr(lib, "kernl_" + n) for n in ("linear_norm_kind", "linear_norm_add_fwd", "linear_norm_apply_fwd", "layernorm_rows32_fwd"))
    assert kind(16, 768, 768) != 0 and kind(64, 768, 768) != 0
    assert kind(16, 776, 768) == 0 and kind(65, 768, 768) == 0 and kind(7, 768, 768) == 0
    assert apply(f, None, f, f, 1e-5, f, f, f, 16, 768, 768, 768, 768, 0, 0, None) == -1
    assert apply(f, f, None, f, 1e-5, f, f, f, 16, 768, 768, 768, 768, 0, 0, None) == -1
    assert apply(f, f, f, f, 1e-5, f, f, f, 16, 768, 768, 768, 768, 9, 0, None) == -1
    assert apply(f, f, f, f, 1e-5, f, f, f, 16, 768, 3072, 3072, 768, 0, 0, None) == -2
    assert apply(f, f, f, f, 1e-5, f, f, f, 16, 768, 40, 40, 768, 0, 0, None) == -2
    assert apply(f, f, f, f, 1e-5, f, f, f, 16, 768, 768, 770, 768, 0, 0, None) == -2
    assert apply(f + 8, f, f, f, 1e-5, f, f, f, 16, 768, 768, 768, 768, 0, 0, None) == -2
    assert apply(f, f, f, f, 1e-5, f, f, f, 65, 768, 768, 768, 768, 0, 0, None) == -2
    assert add(f, f, None, None, None, None, None, 1e-5, f, f, 16, 768, 768, 768, 768, 768, 0, None) == -1
    assert add(f, f, None, f, f, None, None, 1e-5, f, f, 16, 768, 768, 768, 768, 768, 0, None) == -1
    assert add(f, f, None, f, None, None, None, 1e-5, f, f, 16, 768, 768, 768, 768, 772, 0, None) == -1
    assert add(f, f, None, f, None, None, None, 1e-5, f, f, 16, 2048, 768, 768, 2048, 2048, 0, None) == -2
    assert add(f, f, None, f, None, None, None, 1e-5, f, f, 16, 768, 768, 768, 768, 768, 2, None) == -2
    assert rows32(None, f, f, f, 4, 768, 768, 768, 1e-5, 0, None) == -1
    for n, dtype in ((1028, 0), (766, 0), (768, 2)):
        assert rows32(f, f, f, f, 4, n, n, n, 1e-5, dtype, None) == -2


def _encoder(layers, seed=0, **config):
    """A model in fp32 whose norms do something, and its twin"""
    from transformers import BertConfig, BertModel

    torch.manual_seed(seed)
    ref = BertModel(BertConfig(num_hidden_layers=layers, **config)).eval()
    with torch.no_grad():
        for m in ref.modules():
            if isinstance(m, torch.nn.LayerNorm):
                m.weight.add_(torch.randn_like(m.weight) * 0.1), m.bias.add_(torch.randn_like(m.bias) * 0.1)
    model = BertModel(ref.config).eval()
    model.load_state_dict(ref.state_dict())
    return ref, model


def _count(monkeypatch, *names):
    calls = dict.fromkeys(names, 0)
    for name in names:
        real = getattr(_lib, name)
        monkeypatch.setattr(_lib, name, lambda *a, _k=name, _r=real, **k: (calls.__setitem__(_k, calls[_k] + 1), _r(*a, **k))[1])
    return calls


@pytest.mark.gpu
@pytest.mark.parametrize("shape, deferred", [((1, 16), True), ((2, 30), True), ((1, 5), False), ((3, 77), False)], ids=str)
def test_encoder_layers_run_without_a_norm_kernel_of_their_own(shape, deferred, monkeypatch):
    from kernl_amd.model_optimization import optimize_model

    torch._dynamo.reset()
    calls = _count(monkeypatch, "linear_norm_add_fwd", "linear_norm_apply_fwd", "layernorm_rows32_fwd")
    ref, model = _encoder(3)
    model = model.half().cuda()
    optimize_model(model)
    ids = torch.randint(0, 30522, shape)
    mask = (torch.arange(shape[1])[None, :] < torch.randint(shape[1] // 2, shape[1] + 1, (shape[0], 1))).long()
    with torch.inference_mode():
        expected = ref(input_ids=ids, attention_mask=mask).last_hidden_state
        for _ in range(2):
            out = model(input_ids=ids.cuda(), attention_mask=mask.cuda()).last_hidden_state
        torch.cuda.synchronize()
        valid = mask.bool()
        assert (out.cpu().float() - expected)[valid].abs().max() <= 3e-2
        # warm-up and capture run three layers each: two additions a layer, 2 + 2 x 2 - 1 projections behind a deferred norm, one
        # norm that leaves the encoder as a tensor
        assert list(calls.values()) == ([2 * 6, 2 * 5, 2] if deferred else [0, 0, 0]), calls
        # an updated norm is read where it is
        for m in (model, ref):
            m.encoder.layer[0].attention.output.LayerNorm.weight.mul_(1.5)
        expected = ref(input_ids=ids, attention_mask=mask).last_hidden_state
        out = model(input_ids=ids.cuda(), attention_mask=mask.cuda()).last_hidden_state
        torch.cuda.synchronize()
        assert (out.cpu().float() - expected)[valid].abs().max() <= 3e-2


@pytest.mark.gpu
def test_norms_whose_readers_do_not_take_them_are_carried_out(monkeypatch):
    """Feed-forward weights of more than 8 M elements are not the dealt tiles' to read: the norms around them are not deferred, and
    no row is written un-normalised for nothing, although the other projections of such a layer would take it."""
    from kernl_amd.model_optimization import optimize_model

    torch._dynamo.reset()
    calls = _count(monkeypatch, "linear_norm_add_fwd", "linear_norm_apply_fwd", "layernorm_rows32_fwd")
    ref, model = _encoder(2, hidden_size=1024, num_attention_heads=16, intermediate_size=8320)
    assert _lib.linear_norm_kind(20, 8320, 1024) == 0 and _lib.linear_norm_kind(20, 3072, 1024) != 0
    model = model.half().cuda()
    optimize_model(model)
    ids = torch.randint(0, 30522, (1, 20))
    with torch.inference_mode():
        expected = ref(input_ids=ids).last_hidden_state
        out = model(input_ids=ids.cuda()).last_hidden_state
        torch.cuda.synchronize()
    assert (out.cpu().float() - expected).abs().max() <= 3e-2
    assert list(calls.values()) == [0, 0, 0], calls


@pytest.mark.gpu
@pytest.mark.parametrize("readers, deferred", [
    ([["plain"]], True), ([["plain", "plain"], ["plain"]], True), ([["large"]], False), ([["large", "plain"]], False),
    ([["plain"], ["transposed"]], False), ([["other type"]], False), ([["narrow"]], False),
], ids=str)
def test_a_norm_is_deferred_by_the_weights_that_read_it(readers, deferred):
    from kernl_amd.implementations.deferred_norm import DeferredNorm
    from kernl_amd.implementations.layer_norm import add_layer_norm
    from kernl_amd.implementations.linear_layer import linear_layer
    from kernl_amd.optimizer.linear import linear_add_layer_norm_wrapper

    x, w, b, res, gamma, beta = _make(20, 768, 768, torch.float16, 1)
    weights = {"plain": _make(1, 3072, 768, torch.float16, 2)[1], "large": torch.zeros(11008, 768, device="cuda").half(),
               "transposed": torch.zeros(768, 768, device="cuda").half().t(), "other type": torch.zeros(768, 768, device="cuda").bfloat16(),
               "narrow": torch.zeros(40, 768, device="cuda").half()}
    behind = tuple(tuple(weights[name] for name in names) for names in readers)
    out = linear_add_layer_norm_wrapper(x, w, b, res, (768,), gamma, beta, 1e-5, behind=behind)
    assert isinstance(out, DeferredNorm) == deferred
    want = add_layer_norm(linear_layer(x, w, b), res, gamma, beta, 1e-5)
    if deferred:
        assert (out.normalised() - want).abs().max() <= 2e-2  # (two roundings fewer)
    else:
        assert torch.equal(out, want)


def test_only_norms_of_known_readers_are_marked():
    from kernl_amd.optimizer import linear

    class Layer(torch.nn.Module):
        def __init__(self, leak):
            super().__init__()
            self.leak = leak

        def forward(self, x, res, w, w2, g):
            a = linear.linear_add_layer_norm_wrapper(x, w, None, res, (32,), g, None, 1e-5)
            q = linear.fused_linear_wrapper(a, [w, w2], [None, None])[0]
            b = linear.linear_add_layer_norm_wrapper(linear.linear_wrapper_functional(q, w2, None), w, None, a, (32,), g, None, 1e-5)
            return (b, a) if self.leak else b

    for leak in (False, True):
        gm = torch.fx.symbolic_trace(Layer(leak))
        linear.defer_layer_norms(gm)
        norms = [n for n in gm.graph.nodes if n.target is linear.linear_add_layer_norm_wrapper]
        names = [[[w.name for w in weights] for weights in n.kwargs.get("behind", ())] for n in norms]
        assert names == ([[], []] if leak else [[["w", "w2"], ["w"]], []])


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["expanded", "one odd row"])
def test_rows_the_kernel_does_not_take_are_left_to_the_others(form):
    from kernl_amd.implementations.deferred_norm import DeferredNorm
    from kernl_amd.implementations.layer_norm import add_layer_norm
    from kernl_amd.implementations.linear_layer import linear_layer
    from kernl_amd.optimizer.linear import linear_add_layer_norm_wrapper

    x, w, b, res, gamma, beta = _make(20, 768, 768, torch.float16, 1)
    if form == "expanded":
        x = x[:1].expand(20, 768)
    else:
        x, res = torch.nn.functional.pad(x[:1], (0, 4))[:, :768], res[:1]
    behind = ((_make(1, 3072, 768, torch.float16, 2)[1],),)
    out = linear_add_layer_norm_wrapper(x, w, b, res, (768,), gamma, beta, 1e-5, behind=behind)
    assert not isinstance(out, DeferredNorm)
    assert torch.equal(out, add_layer_norm(linear_layer(x, w, b), res, gamma, beta, 1e-5))
