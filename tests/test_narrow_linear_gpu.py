"""Projections of a few rows over narrow 16-bit weights (csrc/gemm_narrow.hip) against 64-bit products: contractions that end inside a unit and a
step, more waves than units, widths off the 16-row groups and off the 4-wide stores, column ranges of wider rows, a bias."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m", [1, 15, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("n,k", [(1, 8), (7, 16), (34, 120), (100, 136), (1024, 16), (896, 896), (1152, 1032), (2050, 2056), (4112, 392), (130, 5632)])
def test_like_the_product(dtype, m, n, k):
    from lite_llama_amd import _lib as L

    g = torch.Generator(device=DEV).manual_seed(m * n + k)
    wide = torch.randn(m, k + 24, generator=g, device=DEV).to(dtype)
    x = wide[:, 8:8 + k]
    w = (torch.randn(n, k, generator=g, device=DEV) * k ** -0.5).to(dtype)
    bias = torch.randn(n, generator=g, device=DEV).to(dtype) if n % 2 == 0 else None
    out = torch.empty(m, n, dtype=dtype, device=DEV)
    L.check(L.lib().ll_dense16_narrow_matmul(out.data_ptr(), x.data_ptr(), w.data_ptr(), L.ptr(bias), m, n, k, wide.stride(0), k,
                                             L.dtype_code(dtype), L.stream_ptr()), "narrow")
    want = x.double() @ w.double().T + (bias.double() if bias is not None else 0.0)
    # exact 16-bit products summed in fp32 (k 2^-24 of their magnitudes' sum, which stays below 40 deviations), rounded once
    unit = 2.0 ** (-11 if dtype == torch.float16 else -8)
    assert ((out.double() - want).abs() <= unit * want.abs() + k * 2.0 ** -24 * 40 + 2.0 ** -24).all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_which_calls_it_takes(dtype):
    from lite_llama_amd.kernels.quantization import dense16_narrow_linear

    w = torch.randn(896, 896, device=DEV).to(dtype)
    x = torch.randn(3, 5, 896, device=DEV).to(dtype)
    got = dense16_narrow_linear(x, w)
    assert got.shape == (3, 5, 896) and torch.equal(got.view(15, 896), dense16_narrow_linear(x.view(15, 896), w))
    assert dense16_narrow_linear(torch.randn(65, 896, device=DEV).to(dtype), w) is None
    assert dense16_narrow_linear(x.float(), w) is None
    rows = torch.randn(9, 928, device=DEV).to(dtype)
    part = rows[:, 16:912]     # rows 16-byte aligned: read in place; off by one: copied first
    assert torch.equal(dense16_narrow_linear(part, w), dense16_narrow_linear(part.contiguous(), w))
    odd = rows[:, 1:897]
    got = dense16_narrow_linear(odd, w)
    assert got is None or torch.equal(got, dense16_narrow_linear(odd.contiguous(), w))
