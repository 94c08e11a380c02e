"""The routes of a few rows over unquantised 16-bit weights: one rule, which the modules and the native layer call both ask."""

import os
import re

import pytest
import torch

from lite_llama_amd import _lib as L
from lite_llama_amd.kernels import quantization as Q

ROWS, NARROWER, SPLIT = 1, 2, 4


# both sides of every line of the rule
@pytest.mark.parametrize("m,n,k,route", [
    (1, 8192, 128, ROWS), (64, 8192, 128, ROWS), (65, 8192, 128, 0), (0, 8192, 128, 0), (1, 8192, 192, 0), (32, 32768, 1536, ROWS | SPLIT),
    (32, 151936, 4096, ROWS | SPLIT), (33, 151936, 4096, ROWS), (32, 1536, 8960, SPLIT), (33, 1536, 8960, 0), (32, 1536, 4032, 0), (32, 33000, 64, SPLIT),
    (32, 4096, 2048, NARROWER), (33, 4096, 2048, 0), (33, 5120, 2048, NARROWER), (48, 5120, 2048, NARROWER), (49, 5120, 2048, 0), (32, 4080, 2048, 0),
    (32, 4104, 2048, 0), (32, 6144, 2176, 0), (48, 7168, 3072, NARROWER), (48, 7152, 3072, 0), (32, 7168, 3200, 0), (48, 12080, 3072, NARROWER),
    # rows of 8192 columns lie 16 KB apart: above 32 rows the library's until there are outputs enough
    (48, 8208, 8192, 0), (33, 16368, 8192, 0), (32, 8208, 8192, NARROWER | SPLIT), (48, 16400, 8192, NARROWER), (48, 8208, 5120, NARROWER),
    (48, 8208, 14336, NARROWER), (48, 8224, 8192, ROWS)])
def test_the_rule(m, n, k, route):
    assert Q.dense16_route(m, n, k) == route
    assert (Q.dense16_rows_wins(m, n, k), Q.dense16_rows_narrower_wins(m, n, k), Q.dense16_wins(m, n, k)) == (
        bool(route & ROWS), bool(route & NARROWER), bool(route & SPLIT))


def test_nobody_writes_it_down_again():
    root = os.path.dirname(os.path.dirname(L.__file__))
    with open(os.path.join(root, "include", "lite_llama_amd.h")) as f:
        bits = dict(re.findall(r"(LL_ROUTE_\w+) = (\d+)", f.read()))
    assert [int(bits[f"LL_ROUTE_{name}"]) for name in ("ROWS", "ROWS_NARROWER", "SPLIT")] == [Q._ROUTE_ROWS, Q._ROUTE_ROWS_NARROWER, Q._ROUTE_SPLIT]
    with open(os.path.join(root, "lite_llama_amd", "csrc", "layered_decode.hip")) as f:
        text = f.read()
    asked = text[text.index("Route linear_route("):text.index("struct Walk")]
    assert "ll_dense16_route(m, n, k)" in asked and "ll_dense16_narrow_wins(m, n, k)" in asked
    assert not re.search(r"[mnk] [<>]=? *\d", asked)


def test_a_checkout_without_the_library_runs_on_the_host(monkeypatch):
    """Products of host tensors ask for no native code."""
    from lite_llama_amd.quantization.methods import UnquantizedLinearMethod

    def missing():
        raise RuntimeError("no library")

    monkeypatch.setattr(L, "lib", missing)
    layer = torch.nn.Module()
    layer.weight, layer.bias = torch.nn.Parameter(torch.randn(8192, 128), requires_grad=False), None
    x = torch.randn(3, 128)
    assert torch.equal(UnquantizedLinearMethod().apply(layer, x), x @ layer.weight.T)
    assert UnquantizedLinearMethod().apply_gate_up_swiglu(layer, x) is None
    assert Q.dense16_linear(x, layer.weight, policy="auto") is None
