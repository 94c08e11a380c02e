"""Which projections go to a kernel by address (kernels/quantization.py), without a GPU: tensors that call themselves GPU tensors, and a library
that notes what it is asked for."""

import pytest
import torch
import torch.utils._python_dispatch
from torch import nn

from lite_llama_amd.kernels import quantization as Q


class OnGpu(torch.Tensor):
    is_cuda = True


def _gpu(*shape, dtype=torch.float16):
    return torch.zeros(*shape, dtype=dtype).as_subclass(OnGpu)


@pytest.fixture
def launches(monkeypatch):
    seen = []

    def entry(name):
        def call(*a):
            seen.append(name)
            return 0 if name.endswith("_matmul") else 1
        return call

    class Lib:
        def __getattr__(self, name):
            return entry(name)

    monkeypatch.setattr(Q.L, "lib", lambda: Lib())
    monkeypatch.setattr(Q.L, "has", lambda name: True)
    monkeypatch.setattr(Q.L, "stream_ptr", lambda: 0)
    monkeypatch.setattr(Q.L, "gemm_workspace", lambda *a: (torch.zeros(1), torch.zeros(1)))
    return lambda: [n for n in seen if n.endswith("_matmul")]


@pytest.mark.parametrize("linear", [Q.dense16_narrow_linear, Q.dense16_rows_linear, Q.dense16_linear])
@pytest.mark.parametrize("where", ["weight", "bias"])
def test_operands_on_another_device_are_left_to_the_library(launches, linear, where):
    x, weight, bias = _gpu(4, 896), _gpu(896, 896), _gpu(896)
    if where == "weight":
        weight = torch.empty(896, 896, dtype=torch.float16, device="meta")
    else:
        bias = torch.empty(896, dtype=torch.float16, device="meta")
    assert linear(x, weight, bias) is None and launches() == []
    if linear is not Q.dense16_narrow_linear:   # (where all of them are, the kernel runs; the narrow one takes no tensor types of others)
        linear(x, _gpu(896, 896), _gpu(896))
        assert len(launches()) == 1


def _plain(*shape, dtype=torch.float16):
    return torch.zeros(*shape, dtype=dtype)


@pytest.mark.parametrize("bias", [True, False])
def test_results_that_carry_more_than_values_are_left_to_the_library(launches, monkeypatch, bias):
    """The narrow projections replaced ``F.linear`` calls, which gradients, tangents, transforms, modes and autocast pass through."""
    monkeypatch.setattr(torch.Tensor, "is_cuda", True)
    x, weight, b = _plain(4, 896), _plain(896, 896), _plain(896) if bias else None
    ask = Q.dense16_narrow_linear

    def left(x=x, weight=weight, b=b):
        at = len(launches())
        out = ask(x, weight, b)
        assert (out is None) == (len(launches()) == at)
        return out is None

    assert not left() and not left(weight=nn.Parameter(weight, requires_grad=False))
    assert left(x=x.clone().requires_grad_()) and left(weight=nn.Parameter(weight))
    with torch.no_grad():
        assert not left(x=x.clone().requires_grad_()) and not left(weight=nn.Parameter(weight))
    if bias:
        assert left(b=nn.Parameter(b))
    assert left(weight=weight.as_subclass(OnGpu))
    with torch.autograd.forward_ad.dual_level():
        assert left(x=torch.autograd.forward_ad.make_dual(x, x)) and not left()
    seen = []
    torch.func.vmap(lambda row: (seen.append(left(x=row)), row)[1])(_plain(2, 4, 896))
    assert seen == [True]

    class Mode(torch.utils._python_dispatch.TorchDispatchMode):
        def __torch_dispatch__(self, func, kinds, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with Mode():
        assert left()
    monkeypatch.setattr(torch, "is_autocast_enabled", lambda *kind: True)
    assert left()
