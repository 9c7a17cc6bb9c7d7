"""A half-precision projection in front of a residual stream and a LayerNorm that are kept in fp32, no autocast: the sum is fp32, and so stay
the parameters that meet it."""
import pytest
import torch

from kernl_amd.optimizer import layer_norm as norm_passes
from kernl_amd.optimizer import linear as linear_passes


def _operands(rows, device):
    gen = torch.Generator().manual_seed(rows)
    x, w = torch.randn((2, rows, 64), generator=gen).half(), (torch.randn((32, 64), generator=gen) * 0.125).half()
    b, residual = torch.randn((32,), generator=gen).half(), torch.randn((2, rows, 32), generator=gen)
    gamma, beta, behind = torch.rand((32,), generator=gen), torch.randn((32,), generator=gen), torch.randn((32, 32), generator=gen)
    return [t.to(device) for t in (x, w, b, residual, gamma, beta, behind)]


def _check(rows, marked, device):
    x, w, b, residual, gamma, beta, behind = _operands(rows, device)
    marks = {"behind": [[behind]]} if marked else {}
    out = linear_passes.linear_add_layer_norm_wrapper(x, w, b, residual, (32,), gamma, beta, 1e-5, **marks)
    assert gamma.dtype == beta.dtype == behind.dtype == out.dtype == torch.float32
    projected = torch.nn.functional.linear(x.double(), w.double(), b.double()).half().double()
    expect = torch.nn.functional.layer_norm(projected + residual.double(), (32,), gamma.double(), beta.double(), 1e-5)
    # the projection may round to the other neighbour: a spacing of 2^-8 for values below 8, over a deviation of 1 or more, times gamma below 1
    assert (out.double() - expect).abs().max() <= 4e-3


@pytest.mark.parametrize("marked", [False, True], ids=["plain", "marked"])
def test_parameters_of_an_fp32_sum(marked, monkeypatch):
    def linear_on_the_host(x, w, b, activation=""):
        return torch.nn.functional.linear(x.float(), w.float(), b.float()).to(x.dtype)

    def norm_on_the_host(x, w, b, eps):
        assert x.dtype == w.dtype == b.dtype  # as the operator asserts
        return torch.nn.functional.layer_norm(x, w.shape, w, b, eps)

    monkeypatch.setattr(linear_passes, "linear_layer", linear_on_the_host)
    monkeypatch.setattr(norm_passes, "layer_norm", norm_on_the_host)
    _check(5, marked, "cpu")


@pytest.mark.gpu
@pytest.mark.parametrize("marked", [False, True], ids=["plain", "marked"])
@pytest.mark.parametrize("rows", [5, 70, 700])
def test_parameters_of_an_fp32_sum_on_the_device(rows, marked):
    _check(rows, marked, "cuda")
