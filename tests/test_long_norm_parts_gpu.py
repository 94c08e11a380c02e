"""Read-out norms of long parts in 16-byte pieces (csrc/linear_mix.hip: a workgroup per part, every value read once) against 64 bits, at the
edges of a thread's pieces and of the form's range."""

import pytest
import torch

from oracle import nivotar as O

pytestmark = pytest.mark.gpu
DEV, F64 = "cuda", torch.float64


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("parts,ps,w_len", [(1, 512, 512), (3, 520, 520), (2, 2048, 4096), (1, 2056, 8), (1, 4096, 4096), (2, 4104, 4104),
                                          (1, 8192, 8192), (1, 8200, 8200)])
@pytest.mark.parametrize("gate,first", [("silu", True), ("sigmoid", False), (None, False)])
def test_long_parts(dtype, parts, ps, w_len, gate, first):
    from lite_llama_amd.kernels.recurrent import gated_out_norm

    g = torch.Generator(device=DEV).manual_seed(ps)
    n, width, eps, scale = 5, parts * ps, 1e-5, 0.7
    o = torch.randn(n, width, device=DEV, generator=g) * 3
    w = (1 + 0.2 * torch.randn(w_len, device=DEV, generator=g)).to(dtype)
    wide = torch.randn(n, width + 8, device=DEV, generator=g).to(dtype)
    out = torch.zeros(n, width + 8, device=DEV, dtype=dtype)
    gated_out_norm(o, w, eps, parts=parts, gate=wide[:, 8:] if gate else None, gate_kind=gate, gate_first=first, scale=scale, out=out[:, 8:])
    gv = wide[:, 8:].to(F64)
    gv = O.silu(gv) if gate == "silu" else torch.sigmoid(gv) if gate == "sigmoid" else torch.ones_like(gv)
    y = o.to(F64) * gv if first else o.to(F64)
    y = O.rms_norm(y.view(n, parts, ps), None, eps).view(n, width) * w.to(F64).repeat(width // w_len)
    y = (y if first else y * gv) * scale
    # fp32 until the last rounding: 32 units of it for the gate's exponential, the mean and four products, then half a unit of the storage type
    unit = {torch.float32: 0.0, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[dtype]
    assert ((out[:, 8:].to(F64) - y).abs() <= (32 * 2.0 ** -24 + unit) * y.abs() + 2.0 ** -24).all()
    assert out[:, :8].abs().max() == 0
    # one element off the 16-byte borders: the plain form, the same bits
    off = torch.zeros(n, width + 9, device=DEV, dtype=dtype)
    gated_out_norm(o, w, eps, parts=parts, gate=wide[:, 8:] if gate else None, gate_kind=gate, gate_first=first, scale=scale, out=off[:, 9:])
    assert torch.equal(off[:, 9:], out[:, 8:])
