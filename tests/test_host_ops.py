"""The native host side of the operators (kernl_amd/csrc/host_ops.cpp): the calls it takes give bit for bit what the
Python route gives, the calls it does not take end up on that route."""
import pytest
import torch

from kernl_amd import _lib


def test_few_row_rule_is_the_python_one():
    from kernl_amd.implementations import linear_layer as m

    assert _lib.host().FEW_ROW_RULE == (m.FEW_ROW_MIN_ROWS, m.FEW_ROW_MAX_ROWS, m.FEW_ROW_MIN_WEIGHT, m.FEW_ROW_LONG_K, m.SPLIT_K_MAX_ROWS)


def test_cpu_tensors_and_wrong_arguments_are_refused():
    h = _lib.host()
    x = torch.zeros(2, 8)
    assert h.op_layer_norm(x, x[0], None, 1e-5, False, None) is None
    assert h.op_linear(x.half(), x.half(), None, 0, None, True) is None
    with pytest.raises(_lib.KernlLibraryError, match="GPU"):
        _lib.layernorm_fwd(x, x[0], None, x, None, None, 1e-5, False)
    with pytest.raises(TypeError):
        h.op_layer_norm(x)
    with pytest.raises(TypeError):
        h.linear_fwd(1, x, None, x, None, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(1, 8), (5, 3, 768), (70, 4096)], ids=str)
@pytest.mark.parametrize("rms", [False, True])
def test_layer_norm_routes_agree(shape, rms):
    from kernl_amd.implementations.layer_norm import LayerNorm, add_layer_norm, layer_norm

    x, res = torch.randn(2, *shape, device="cuda").half()
    w, b = torch.randn(2, shape[-1], device="cuda").half()
    b = None if rms else b
    assert torch.equal(layer_norm(x, w, b, 1e-12, use_rms_norm=rms), LayerNorm.apply(x, w, b, 1e-12, None, rms))
    assert torch.equal(add_layer_norm(x, res, w, b, 1e-12, rms), LayerNorm.apply(x, w, b, 1e-12, None, rms, res))
    strided = x.transpose(0, 1) if x.dim() == 2 else x[:, :1]
    if strided.shape[-1] == shape[-1]:
        assert torch.equal(layer_norm(strided, w, b, 1e-12, use_rms_norm=rms), layer_norm(strided.contiguous(), w, b, 1e-12, use_rms_norm=rms))


@pytest.mark.gpu
@pytest.mark.parametrize("rows, n, k", [(1, 768, 768), (40, 4096, 1024), (200, 4096, 4096), (300, 136, 200), (7, 33, 41)], ids=str)
def test_linear_routes_agree(rows, n, k):
    from kernl_amd.implementations.linear_layer import LinearLayer, linear_layer

    x, w, b = torch.randn(rows, k, device="cuda").half(), torch.randn(n, k, device="cuda").half() * 0.05, torch.randn(n, device="cuda").half()
    assert torch.equal(linear_layer(x, w, b, "gelu"), LinearLayer.apply(x, w, b, "gelu", None))
    assert torch.equal(linear_layer(x[None], w, None), LinearLayer.apply(x[None], w, None, "", None))
    saved = torch.empty(2, rows, n, device="cuda").half()
    assert torch.equal(linear_layer(x, w, b, "relu", saved[0]), LinearLayer.apply(x, w, b, "relu", saved[1])) and torch.equal(*saved)
    with pytest.raises(AssertionError):
        linear_layer(x, w.float(), b)


@pytest.mark.gpu
@pytest.mark.parametrize("rows, gated", [((3, 1), False), ((24, 1), False), ((2, 9), True), ((70, 1), True)], ids=str)
def test_few_row_projections_match_their_parts(rows, gated):
    """`plan_few_rows`: the calls it plans against the same product through the separate operators."""
    from kernl_amd.implementations.layer_norm import layer_norm
    from kernl_amd.implementations.linear_layer import decode_linear_layer, linear_glu_layer, linear_layer, rms_linear_layer

    x, g = torch.randn(*rows, 1024, device="cuda").half(), torch.randn(1024, device="cuda").half()
    w, res = torch.randn(8192, 1024, device="cuda").half() * 0.03, torch.randn(*rows, 8192, device="cuda").half()
    normed = layer_norm(x, g, None, 1e-5, use_rms_norm=True)
    ref = linear_glu_layer(normed, w, None, "silu") if gated else linear_layer(normed, w, None)
    out = rms_linear_layer(x, g, 1e-5, w, None, "silu" if gated else "", gated=gated)
    assert out.shape == ref.shape and (out - ref).float().norm() <= 3e-3 * ref.float().norm()
    if rows[0] * rows[1] <= 64:
        out, ref = decode_linear_layer(x, w, residual=res), linear_layer(x, w, None) + res
        assert out.shape == ref.shape and (out - ref).float().norm() <= 2e-3 * ref.float().norm()
        flat = decode_linear_layer(x.flatten(0, 1), w, residual=res.flatten(0, 1))
        assert torch.equal(flat, out.flatten(0, 1))


@pytest.mark.gpu
@pytest.mark.parametrize("causal, masked, start", [(False, True, 0), (True, False, 0), (True, False, 9)], ids=str)
def test_attention_routes_agree(causal, masked, start):
    from kernl_amd.implementations.attention import Attention, attention_forward
    from kernl_amd.implementations.attention_skinny import SkinnyAttention, skinny_attention_forward

    q = torch.randn(2, 3, 33, 64, device="cuda").half()
    k, v = torch.randn(2, 2, 3, 42, 64, device="cuda").half()
    mask = torch.randn(2, 1, 1, 42, device="cuda") if masked else None
    out = [torch.empty_like(q) for _ in range(2)]
    assert attention_forward(q, k, v, out[0], 0.125, causal, mask, start) is out[0]
    Attention.apply(q, k, v, out[1], 0.125, causal, mask, start)
    assert torch.equal(*out)
    one = [torch.empty_like(q[:, :, :1]) for _ in range(2)]
    skinny_attention_forward(q[:, :, :1], k, v, one[0], 0.125, False, mask)
    SkinnyAttention.apply(q[:, :, :1], k, v, one[1], 0.125, False, mask)
    assert torch.equal(*one)
    with pytest.raises(AssertionError):
        attention_forward(q, k.bfloat16(), v, out[0], 0.125, causal, mask, start)


@pytest.mark.gpu
def test_autocast_and_recorded_calls_take_the_python_route():
    from kernl_amd.implementations.layer_norm import layer_norm

    x, w = torch.randn(4, 64, device="cuda"), torch.ones(64, device="cuda")
    with torch.autocast("cuda", dtype=torch.float16):
        assert layer_norm(x, w, None, 1e-5).dtype == torch.float16
    assert layer_norm(x, w.requires_grad_(), None, 1e-5).requires_grad
    with torch.no_grad():
        assert not layer_norm(x, w, None, 1e-5).requires_grad
