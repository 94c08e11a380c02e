"""Which projections go to a kernel by address (kernels/quantization.py), without a GPU: tensors that call themselves GPU tensors, and a library
that notes what it is asked for."""

import types

import pytest
import torch
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
    linear(x, _gpu(896, 896), _gpu(896))
    assert len(launches()) == 1   # (where all of them are, the kernel runs)
