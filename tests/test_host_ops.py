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


def _operators():
    """Every operator with a native route, as (name, function of its first tensor, that tensor)."""
    from kernl_amd.implementations.attention import attention_forward
    from kernl_amd.implementations.attention_skinny import skinny_attention_forward
    from kernl_amd.implementations.layer_norm import add_layer_norm, layer_norm
    from kernl_amd.implementations.linear_layer import linear_layer

    x, w = torch.randn(4, 64, device="cuda").half(), torch.randn(64, 64, device="cuda").half()
    q, k, v = torch.randn(3, 1, 2, 8, 64, device="cuda").half()
    return [
        ("layer_norm", lambda t: layer_norm(t, w[0], None, 1e-5), x),
        ("add_layer_norm", lambda t: add_layer_norm(t, x, w[0], None, 1e-5), x),
        ("linear_layer", lambda t: linear_layer(t, w, None), x),
        ("linear_layer (weight)", lambda t: linear_layer(x, t, None), w),
        ("attention_forward", lambda t: attention_forward(t, k, v, torch.empty_like(q), 0.125), q),
        ("skinny_attention_forward", lambda t: skinny_attention_forward(t, k[:, :, :1], v[:, :, :1], torch.empty_like(k[:, :, :1]), 0.125), q[:, :, :1].contiguous()),
    ]


@pytest.mark.gpu
def test_forward_mode_is_refused():
    """The autograd functions have no jvp: a tangent is an error, not a result without it."""
    import torch.autograd.forward_ad as fwAD

    for name, op, x in _operators():
        for grad in (False, True):
            with fwAD.dual_level(), torch.set_grad_enabled(grad):
                with pytest.raises(NotImplementedError):
                    op(fwAD.make_dual(x, torch.ones_like(x)))
                    pytest.fail(f"{name}: a tangent went lost")


@pytest.mark.gpu
def test_traced_calls_are_recorded():
    """What torch.jit.trace keeps is the autograd function, not an allocation that nothing fills."""
    from kernl_amd.implementations.layer_norm import layer_norm

    x, w = torch.randn(4, 64, device="cuda").half(), torch.randn(64, device="cuda").half()
    traced = torch.jit.trace(lambda t: layer_norm(t, w, None, 1e-5), x, check_trace=False)
    assert "LayerNorm" in str(traced.graph) and "aten::empty" not in str(traced.graph)


@pytest.mark.gpu
def test_transforms_are_refused():
    for name, op, x in _operators():
        for transformed in (lambda t: torch.vmap(op)(t), lambda t: torch.func.jvp(op, (t,), (torch.ones_like(t),)),
                            lambda t: torch.vmap(lambda i: op(x) + i)(torch.zeros(3, device="cuda"))):
            with pytest.raises(RuntimeError):  # (NotImplementedError among them)
                transformed(torch.stack((x, x)))
                pytest.fail(f"{name}: carried out inside a transform")


def test_calls_that_someone_watches_are_declined():
    """Under a transform, a tracer or a dispatch mode the native route declines before it looks at the tensors, and an
    operator goes to its autograd function."""
    from torch.utils._python_dispatch import TorchDispatchMode

    h, x = _lib.host(), torch.zeros(2, 8)
    seen = []

    def probe(t):
        seen.append([h.takes_call(), torch._C._are_functorch_transforms_active()])
        return t + 1

    probe(x)
    assert seen == [[True, False]]
    torch.vmap(probe)(x)
    torch.func.jvp(probe, (x,), (x,))
    assert seen[1:] == [[False, True]] * 2
    del seen[:]
    torch.jit.trace(probe, x, check_trace=False)
    with TorchDispatchMode():
        seen.append([h.takes_call(), False])
    assert seen == [[False, False]] * 2


@pytest.mark.gpu
def test_a_failed_allocation_is_pytorchs_error():
    """4 M x 128 K results are 1 TB: refused by the allocator before anything is launched."""
    from kernl_amd.implementations.linear_layer import LinearLayer, linear_layer

    x, w = torch.zeros(1 << 22, 8, dtype=torch.float16, device="cuda"), torch.zeros(1 << 17, 8, dtype=torch.float16, device="cuda")
    for call in (linear_layer, lambda *a: LinearLayer.apply(*a, "", None)):
        with pytest.raises(torch.OutOfMemoryError):
            call(x, w, None)


@pytest.mark.gpu
@pytest.mark.parametrize("causal, start, same_as", [(False, None, 0), (True, None, 0), (False, 5.0, 0), (True, 5.0, 5), (False, "x", 0)], ids=str)
def test_start_position_is_read_where_it_is_used(causal, start, same_as):
    from kernl_amd.implementations.attention import Attention, attention_forward

    q, k, v = torch.randn(3, 1, 2, 9, 64, device="cuda").half()
    out = [torch.empty_like(q) for _ in range(3)]
    attention_forward(q, k, v, out[0], 0.125, causal, None, start)
    Attention.apply(q, k, v, out[1], 0.125, causal, None, start)
    attention_forward(q, k, v, out[2], 0.125, causal, None, same_as)
    assert torch.equal(out[0], out[1]) and torch.equal(out[0], out[2])


@pytest.mark.gpu
def test_sizes_of_a_projection_may_be_floats():
    """int() is taken of them, as it always was."""
    from kernl_amd.implementations.linear_layer import decode_linear_layer

    x, w, g = torch.randn(3, 128, device="cuda").half(), torch.randn(256, 128, device="cuda").half(), torch.ones(128, device="cuda").half()
    cos, sin = torch.randn(2, 1, 3, 64, device="cuda").half()
    want = decode_linear_layer(x, w, None, g, 1e-5, None, cos, sin, 64, 128)
    assert torch.equal(decode_linear_layer(x, w, None, g, 1e-5, None, cos, sin, 64.0, 128.0), want)
