"""What a kernel stores as bf16 (common.h::f32_to_bf16_bits): round to nearest, ties to even, subnormals and infinities kept, NaN a NaN."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("low", [0x0000, 0x0001, 0x7fff, 0x8000, 0x8001, 0xffff])
def test_every_upper_half_beside_the_edges_of_a_rounding(low):
    from lite_llama_amd.kernels.norm_act import PartialSums, skip_rmsnorm_partials

    n = 4096
    bits = (torch.arange(1 << 16, dtype=torch.int64) << 16) + low
    values = (bits - (bits >> 31 << 32)).to(torch.int32).view(torch.float32).view(-1, n)
    # (one plane and a residual of zeros: the updated residual is the rounded value; -0 + 0 is 0 there)
    residual = torch.zeros(values.shape, dtype=torch.bfloat16, device=DEV)
    weight = torch.ones(n, dtype=torch.bfloat16, device=DEV)
    _, got = skip_rmsnorm_partials(PartialSums(values[None].to(DEV), values.shape, torch.bfloat16), residual, weight)
    got, want = got.cpu(), values.to(torch.bfloat16)
    assert torch.equal(got.isnan(), want.isnan())
    number = ~want.isnan()
    assert torch.equal(got[number], want[number])
