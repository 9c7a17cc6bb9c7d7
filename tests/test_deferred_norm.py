"""LayerNorms left to the linear layers behind them (csrc/norm_fold.h): both kernels' forms against fp32 PyTorch at the edges
of their tiles, and the graph pass."""
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


# rows around the tile heights, widths around the groups: (rows, width, k) of the layer in front of the norm
SHAPES = [(1, 96, 72), (8, 768, 768), (16, 768, 3072), (17, 768, 3072), (33, 1024, 1024), (65, 32, 264), (231, 768, 768),
          (320, 768, 3072), (500, 768, 768), (640, 768, 768)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("offset", [0.0, 30.0])
@pytest.mark.parametrize("rows, n, k", SHAPES, ids=str)
def test_both_sides_of_a_deferred_norm(rows, n, k, offset, dtype):
    from kernl_amd.implementations.deferred_norm import DeferredNorm, FoldedParams, linear_add_deferred

    if _lib.linear_norm_kind(rows, n, k) == 0:
        pytest.skip("not a small problem")
    x, w, b, res, gamma, beta = _make(rows, n, k, dtype, rows + n, offset=offset)
    unit = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    norm = linear_add_deferred(x, w, b, res, gamma, beta, 1e-12)
    s = x.double() @ w.double().T + b.double() + res.double()
    assert _error(norm.rows, s) <= unit
    # statistics of the stored rows, group by group
    group = _lib.linear_norm_group(rows)
    groups = norm.rows.double().view(rows, n // group, group)
    assert torch.allclose(norm.stats[..., 0].double(), groups.sum(-1), rtol=1e-5, atol=1e-3)
    assert torch.allclose(norm.stats[..., 1].double(), groups.var(-1, unbiased=False) * group, rtol=1e-4, atol=1e-4)
    # a second addition on top of the deferred residual
    eps = norm.kernel_eps
    h = _ln(norm.rows, gamma, beta, eps)
    again = linear_add_deferred(x, w, None, norm, gamma, None, 1e-12)
    assert _error(again.rows, x.double() @ w.double().T + h) <= 1.5 * unit
    # the layers behind: every activation's branch, with and without parameters
    for width, bias, activation in ((64, None, ""), (96, True, "gelu"), (32, True, "relu")):
        if not norm.takes_linear(width, activation):
            continue
        w2, b2 = _make(1, width, n, dtype, 7)[1], (_make(1, width, n, dtype, 7)[2] if bias else None)
        ref = h @ w2.double().T + (0 if b2 is None else b2.double())
        ref = torch.nn.functional.gelu(ref) if activation == "gelu" else torch.relu(ref) if activation == "relu" else ref
        out = norm.linear(FoldedParams.of(w2, b2, gamma, beta), activation)
        assert _error(out, ref) <= 4 * unit * (1 + offset / 4), (width, activation)
    assert isinstance(norm, DeferredNorm) and _error(norm.normalised(), h) <= 2 * unit


@pytest.mark.gpu
@pytest.mark.parametrize("force, rows", [(10, 70), (11, 70), (15, 70), (12, 21), (13, 45), (14, 70), (16, 40), (17, 130)], ids=str)
def test_every_tile_form_takes_both_modes(force, rows):
    from kernl_amd.implementations.deferred_norm import FoldedParams, linear_add_deferred

    x, w, b, res, gamma, beta = _make(rows, 160, 200, torch.float16, force)
    w2, b2 = _make(1, 160, 160, torch.float16, 3)[1:3]
    lib = _lib.load()
    lib.kernl_linear_force_tile(force)
    try:
        norm = linear_add_deferred(x, w, b, res, gamma, beta, 1e-5)
        out = norm.linear(FoldedParams.of(w2, b2, gamma, beta), "")
        torch.cuda.synchronize()
    finally:
        lib.kernl_linear_force_tile(0)
    assert _error(norm.rows, x.double() @ w.double().T + b.double() + res.double()) <= 2.0 ** -11
    assert _error(out, _ln(norm.rows, gamma, beta, norm.kernel_eps) @ w2.double().T + b2.double()) <= 2.0 ** -9


def test_bad_arguments_are_rejected():
    lib, f = _lib.load(), 64  # never dereferenced
    assert lib.kernl_linear_norm_kind(16, 768, 768) != 0 and lib.kernl_linear_norm_kind(16, 776, 768) == 0
    assert lib.kernl_linear_norm_apply_fwd(f, None, 1e-5, f, f, f, f, 16, 768, 768, 768, 768, 0, 0, None) == -1
    assert lib.kernl_linear_norm_apply_fwd(f, f, 1e-5, f, f, f, f, 16, 768, 3072, 3072, 768, 0, 0, None) == -2
    assert lib.kernl_linear_norm_apply_fwd(f, f, 1e-5, f, f, f, f, 16, 768, 768, 768, 768, 9, 0, None) == -1
    assert lib.kernl_linear_norm_add_fwd(f, f, None, None, None, None, None, 1e-5, f, f, 16, 768, 768, 768, 768, 768, 0, None) == -1
    assert lib.kernl_linear_norm_add_fwd(f, f, None, f, f, None, None, 1e-5, f, f, 16, 768, 768, 768, 768, 768, 0, None) == -1
    assert lib.kernl_linear_norm_add_fwd(f, f, None, f, None, None, None, 1e-5, f, f, 16, 2048, 768, 768, 2048, 2048, 0, None) == -2
    assert lib.kernl_linear_norm_add_fwd(f, f, None, f, None, None, None, 1e-5, f, f, 16, 768, 768, 768, 768, 768, 2, None) == -2


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(1, 16), (3, 77), (2, 250)], ids=str)
def test_encoder_layers_run_without_a_norm_kernel_of_their_own(shape, monkeypatch):
    from transformers import BertConfig, BertModel

    from kernl_amd.model_optimization import optimize_model

    torch._dynamo.reset()
    calls = {"add": 0, "apply": 0, "norm": 0}
    for key, name in (("add", "linear_norm_add_fwd"), ("apply", "linear_norm_apply_fwd")):
        real = getattr(_lib, name)
        monkeypatch.setattr(_lib, name, lambda *a, _k=key, _r=real: (calls.__setitem__(_k, calls[_k] + 1), _r(*a))[1])
    torch.manual_seed(0)
    ref = BertModel(BertConfig(num_hidden_layers=3)).eval()
    model = BertModel(ref.config).eval()
    model.load_state_dict(ref.state_dict())
    with torch.no_grad():  # norms that do something
        for a, b in zip(ref.modules(), model.modules()):
            if isinstance(a, torch.nn.LayerNorm):
                a.weight.add_(torch.randn_like(a.weight) * 0.1), a.bias.add_(torch.randn_like(a.bias) * 0.1)
                b.weight.copy_(a.weight), b.bias.copy_(a.bias)
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
        # warm-up and capture run three layers each: two additions a layer, 2 + 2 x 2 - 1 projections behind a deferred norm
        assert calls["add"] == 2 * 6 and calls["apply"] == 2 * 5, calls
        # an updated norm reaches the folded weights
        model.encoder.layer[0].attention.output.LayerNorm.weight.mul_(1.5)
        ref.encoder.layer[0].attention.output.LayerNorm.weight.mul_(1.5)
        expected = ref(input_ids=ids, attention_mask=mask).last_hidden_state
        out = model(input_ids=ids.cuda(), attention_mask=mask.cuda()).last_hidden_state
        torch.cuda.synchronize()
        assert (out.cpu().float() - expected)[valid].abs().max() <= 3e-2
