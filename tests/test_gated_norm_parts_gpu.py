"""The grouped norm over pieces of four channels (csrc/group_norm.hip) against 64-bit sums: every count of result rows at which another number of them
is requested ahead, groups at the edges of a thread's pieces, each optional input alone and together."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, F64 = "cuda", torch.float64


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("parts", [1, 2, 4, 5, 8, 9, 17])
@pytest.mark.parametrize("width,groups", [(4, 1), (1024, 1), (1028, 1), (2048, 2), (2052, 1), (4096, 1), (12288, 3)])
@pytest.mark.parametrize("given", ["", "shared", "gate", "bias", "shared gate bias"])
def test_rows_of_every_count_and_width(dtype, parts, width, groups, given):
    from lite_llama_amd.kernels.norm_act import GatedUpdate, gated_group_norm

    g = torch.Generator(device=DEV).manual_seed(width + parts)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV)  # noqa: E731
    n, eps = 3, 1e-5
    x, y = r(n, width) * 3, r(n, parts, width).to(dtype)
    pw, nw = (1 + 0.1 * r(width)).to(dtype), (1 + 0.1 * r(width)).to(dtype)
    shared, scale = (r(n, width).to(dtype), r(n).abs()) if "shared" in given else (None, None)
    gate = r(n, width + 8).to(dtype)[:, 4:4 + width] if "gate" in given else None
    gate_bias = r(width).to(dtype) if "gate bias" in given else None
    bias = r(width).to(dtype) if "bias" in given else None
    d = lambda t: t.to(F64)  # noqa: E731

    def norm(v, w):
        v = v.view(n, groups, -1)
        return (v / (v.square().mean(2, keepdim=True) + eps).sqrt()).reshape(n, width) * d(w)

    s = d(y).sum(1)
    s = s + d(bias) if bias is not None else s
    s = s + d(scale)[:, None] * d(shared) if shared is not None else s
    if gate is not None:
        s = s * torch.sigmoid(d(gate) + (d(gate_bias) if gate_bias is not None else 0))
    want_x = d(x) + norm(s, pw)
    want_h = norm(want_x, nw)
    got_x = x.clone()
    h = gated_group_norm(got_x, GatedUpdate(y, pw, gate, gate_bias, shared, scale, bias), nw, eps, groups)
    # fp32 throughout: a value's error is some units of the sums' terms (parts + 3 of them, each at most 5 deviations), and a norm over few channels
    # hands every channel's error on; the 16-bit forms take the hardware exponential (a few units of fp32)
    bar = 2.0 ** -20 * (parts + 8)
    assert ((d(got_x) - want_x).abs() <= bar * (want_x.abs() + 4)).all()
    unit = {torch.float32: 2.0 ** -23, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[dtype]
    assert ((d(h) - want_h).abs() <= unit * want_h.abs() + bar * (want_h.abs() + 4)).all()
