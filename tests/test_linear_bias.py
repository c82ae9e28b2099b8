"""A CiderLinear's bias reaches the kernels in every form a program can give it."""

import pytest
import torch

from cider_amd import nn, ops

N, K = 64, 256


def layer(group_size, device):
    g = torch.Generator().manual_seed(group_size)
    w = torch.randint(-127, 128, (N, K), dtype=torch.int8, generator=g)
    shape = (K // group_size, N) if group_size else (N,)
    s = torch.rand(shape, generator=g) * 1e-3 + 1e-4
    return nn.CiderLinear(w.to(device), s.to(device), group_size, K, N), g


@pytest.mark.parametrize("group_size", [0, 64])
@pytest.mark.parametrize("form", ["buffer", "parameter", "none"])
def test_native_call_gets_the_bias(monkeypatch, group_size, form):
    # without a GPU: which bias the native call would be given, if it is made
    lin, _ = layer(group_size, "cpu")
    b = torch.arange(N).half()
    lin.bias = {"buffer": b, "parameter": torch.nn.Parameter(b), "none": None}[form]
    given = []
    monkeypatch.setattr(ops, "_fast", lambda op, x, w, s, bias, *a: given.append(bias) or x)
    for general in ("perchannel_linear", "pergroup_linear"):
        monkeypatch.setattr(ops, general, lambda x, *a: x[:, :N])
    lin(torch.zeros(2, K).half())
    assert len(given) == (form != "none")
    assert all(t is lin.bias for t in given)


@pytest.mark.gpu
@pytest.mark.parametrize("group_size", [0, 64])
@pytest.mark.parametrize("M", [1, 5])
def test_parameter_bias(group_size, M):
    lin, g = layer(group_size, "cuda")
    x = torch.randn(M, K, generator=g).half().cuda()
    b = torch.randn(N, generator=g).half().cuda()
    without = lin(x)
    lin.bias = torch.nn.Parameter(b)
    y = lin(x)
    if group_size:
        e = ops.pergroup_linear(x, lin.w_int8, lin.scale_w, group_size, b)
    else:
        e = ops.perchannel_linear(x, lin.w_int8, lin.scale_w, b)
    assert torch.equal(y.view(torch.int16), e.view(torch.int16))
    assert not torch.equal(y, without)
