"""Grouped expert products of a few rows per expert (csrc/moe_stream.hip) against 64-bit products of the same operands: contractions that end
inside a unit, widths off the row groups, experts without rows, with one, with more than a piece of a block, slots that no expert serves, one
token; 8-bit weights with every kind of code, scales per row and per block."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, F64 = "cuda", torch.float64


def _ids(tokens, experts, top, g, hot):
    """Random experts per token; ``hot``: every token's first slot goes to expert 1."""
    ids = torch.rand(tokens, experts, generator=g, device=DEV).topk(top).indices.to(torch.int32)
    if hot:
        ids = torch.where(ids == 1, ids[:, :1], ids)
        ids[:, 0] = 1
    return ids.contiguous()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("width,ff,experts,tokens,top", [(128, 16, 5, 1, 1), (136, 200, 9, 40, 2), (264, 128, 40, 33, 4), (2048, 704, 34, 32, 4),
                                                         (392, 1000, 300, 64, 8), (640, 136, 3, 20, 2), (264, 128, 3, 40, 2), (1032, 72, 5, 85, 2)])
@pytest.mark.parametrize("form", ["silu", "clamped", "square"])
def test_16_bit_experts(dtype, width, ff, experts, tokens, top, form):
    from lite_llama_amd.kernels.fused_moe import sparse_glu_experts, sparse_square_experts

    g = torch.Generator(device=DEV).manual_seed(width + ff)

    def r(*s, std=1.0):
        return (torch.randn(*s, generator=g, device=DEV) * std).to(dtype)

    ids = _ids(tokens, experts, top, g, tokens > 1)
    if form != "square" and tokens > 1:
        ids[::5, top - 1] = experts + 3          # slots that no expert serves
    h, weights = r(tokens, width), torch.rand(tokens, top, generator=g, device=DEV) + 0.1
    up = r(experts, ff if form == "square" else 2 * ff, width, std=width ** -0.5)
    down = r(experts, width, ff, std=ff ** -0.5)
    if form == "square":
        got = sparse_square_experts(h, up, down, ids, weights)
    else:
        got = sparse_glu_experts(h, up, down, ids, weights, limit=1.5 if form == "clamped" else None, skipped_ids=True)
    want, mid = torch.zeros(tokens, top, width, dtype=F64, device=DEV), torch.zeros(tokens, top, 1, dtype=F64, device=DEV)
    for e in ids.unique().tolist():
        if e >= experts:
            continue
        at = (ids == e).nonzero(as_tuple=True)
        x, wt = h[at[0]].to(F64), weights[at].to(F64)[:, None]
        if form == "square":
            act, wt = torch.relu(x @ up[e].to(F64).T * wt) ** 2, torch.ones_like(wt)
        else:
            gate, u = (x @ w.to(F64).T for w in (up[e, :ff], up[e, ff:]))
            if form == "clamped":
                gate, u = gate.clamp(max=1.5), u.clamp(-1.5, 1.5) + 1
                act = gate * torch.sigmoid(1.702 * gate) * u
            else:
                act = torch.nn.functional.silu(gate) * u
        want[at] = (act @ down[e].to(F64).T) * wt
        mid[at] = act.norm(dim=1, keepdim=True) * wt * ff ** -0.5
    # two roundings to 16 bits: the activations' (each a half unit, met by weights of std ff^-1/2: 6 deviations) and the result's own
    unit = 2.0 ** (-11 if dtype == torch.float16 else -8)
    assert ((got.to(F64) - want).abs() <= unit * (want.abs() + 6 * mid) + 2.0 ** -14 * unit).all()


@pytest.mark.parametrize("fmt", ["fp8", "int8"])
@pytest.mark.parametrize("width,ff,experts,tokens,top,group", [(128, 128, 4, 1, 2, 128), (144, 160, 6, 9, 2, 64), (384, 272, 30, 17, 3, 128),
                                                               (2048, 768, 128, 64, 8, 128), (512, 256, 20, 100, 2, 4096),
                                                               (400, 144, 8, 60, 2, 4096), (256, 272, 9, 130, 1, 64)])
@pytest.mark.parametrize("interleaved", [False, True])
def test_8_bit_experts(fmt, width, ff, experts, tokens, top, group, interleaved):
    from lite_llama_amd.kernels.fused_moe import fused_moe

    g = torch.Generator(device=DEV).manual_seed(width + ff)
    lo, hi = (0, 256) if fmt == "fp8" else (-127, 128)

    def codes(*shape):
        w = torch.randint(lo, hi, shape, generator=g, device=DEV)
        if fmt == "fp8":
            return torch.where(w & 127 == 127, w - 1, w).to(torch.uint8)
        return w.to(torch.int8)

    def wide(w, scale, rows, cols):
        v = (w.view(torch.float8_e4m3fn) if fmt == "fp8" else w).to(F64)
        s = scale.to(F64).repeat_interleave(rows, 1)[:, :w.shape[1]].repeat_interleave(cols, 2)[:, :, :w.shape[2]]
        return v * s

    rows = 1 if interleaved else 16
    spread = 80.0 if fmt == "fp8" else 73.0       # (deviation of the codes' values)
    w1, w2 = codes(experts, 2 * ff, width), codes(experts, width, ff)
    s1, s2 = ((torch.rand(experts, -(-n // r), -(-k // group), generator=g, device=DEV) + 0.5) * k ** -0.5 / spread
              for n, k, r in ((2 * ff, width, rows), (width, ff, 16)))
    x = torch.randn(tokens, width, generator=g, device=DEV).half()
    ids, weights = _ids(tokens, experts, top, g, tokens > 20), torch.rand(tokens, top, generator=g, device=DEV).half()
    got = fused_moe(x, w1, w2, weights, ids, w1_scale=s1, w2_scale=s2, w1_group=(rows, group), w2_group=(16, group), w1_interleaved=interleaved)
    d1, d2 = wide(w1, s1, rows, group), wide(w2, s2, 16, group)
    want, bound = torch.zeros(tokens, width, dtype=F64, device=DEV), torch.zeros(tokens, width, dtype=F64, device=DEV)
    for t in range(tokens):
        for k in range(top):
            e, wt = int(ids[t, k]), float(weights[t, k])
            y = d1[e] @ x[t].to(F64)
            gate, u = (y[0::2], y[1::2]) if interleaved else (y[:ff], y[ff:])
            act = torch.nn.functional.silu(gate) * u
            one = wt * (d2[e] @ act)
            want[t] += one
            # gate, up and their product are each rounded to fp16 (three half units, |silu'| <= 1.1), and so is the slot's result
            bound[t] += 2.0 ** -11 * (one.abs() + 6 * 3.3 * wt * ((d2[e] ** 2) @ act.abs().clamp(min=0.05) ** 2).sqrt())
    assert ((got.to(F64) - want).abs() <= bound + 2.0 ** -11 * want.abs() + 1e-6).all()


@pytest.mark.parametrize("width,ff,experts,tokens,top", [(128, 144, 4, 48, 2), (264, 200, 4, 100, 2), (392, 128, 20, 130, 4), (256, 72, 2, 64, 1)])
@pytest.mark.parametrize("interleaved", [False, True])
def test_fp16_experts(width, ff, experts, tokens, top, interleaved):
    """Blocks of 32 and 64 slots in pieces of 32 and 64 rows, experts of one piece and of two."""
    from lite_llama_amd.kernels.fused_moe import fused_moe

    g = torch.Generator(device=DEV).manual_seed(width + ff)
    w1, w2 = ((torch.randn(experts, *s, generator=g, device=DEV) * s[1] ** -0.5).half() for s in ((2 * ff, width), (width, ff)))
    x = torch.randn(tokens, width, generator=g, device=DEV).half()
    ids, weights = _ids(tokens, experts, top, g, False), torch.rand(tokens, top, generator=g, device=DEV).half()
    got = fused_moe(x, w1, w2, weights, ids, w1_interleaved=interleaved)
    y = torch.einsum("enk,tk->ten", w1.double().cpu(), x.double().cpu()).to(DEV)   # (every expert of every token)
    gate, u = (y[..., 0::2], y[..., 1::2]) if interleaved else (y[..., :ff], y[..., ff:])
    act = torch.nn.functional.silu(gate) * u
    out = torch.einsum("enk,tek->ten", w2.double().cpu(), act.cpu()).to(DEV)
    spread = torch.einsum("enk,tek->ten", w2.double().cpu() ** 2, act.cpu().abs().clamp(min=0.05) ** 2).to(DEV).sqrt()
    slot = torch.zeros(tokens, experts, dtype=F64, device=DEV).scatter_(1, ids.long(), weights.to(F64)).unsqueeze(-1)
    want = (out * slot).sum(1)
    # gate, up and their product are each rounded to fp16 (three half units, |silu'| <= 1.1), and so are a slot's result and the sum
    bound = 2.0 ** -11 * ((out.abs() + 6 * 3.3 * spread) * slot).sum(1)
    assert ((got.to(F64) - want).abs() <= bound + 2.0 ** -11 * want.abs() + 1e-6).all()


@pytest.mark.parametrize("experts", [16, 17])          # runs within one expert / across them
@pytest.mark.parametrize("groups", [3, 4, 5, 8, 9, 16, 17, 25])
def test_runs_of_row_groups(experts, groups):
    """A row per expert; a workgroup's run is ``groups`` row groups long: one more than the small units hold, than a tile, than two."""
    from lite_llama_amd.kernels.fused_moe import sparse_square_experts

    cus = torch.cuda.get_device_properties(0).multi_processor_count
    width, ff = 136, 16 * (cus * groups // experts)
    g = torch.Generator(device=DEV).manual_seed(groups)
    up, down = ((torch.randn(experts, *s, generator=g, device=DEV) * s[1] ** -0.5).bfloat16() for s in ((ff, width), (width, ff)))
    h, ids = torch.randn(experts, width, generator=g, device=DEV).bfloat16(), torch.randperm(experts, generator=g, device=DEV).to(torch.int32)[:, None]
    weights = torch.rand(experts, 1, generator=g, device=DEV) + 0.1
    got = sparse_square_experts(h, up, down, ids, weights)[:, 0].double()
    act = torch.stack([torch.relu(up[e].double() @ h[t].double() * weights[t].double()) ** 2 for t, e in enumerate(ids[:, 0].tolist())])
    want = torch.stack([down[e].double() @ act[t] for t, e in enumerate(ids[:, 0].tolist())])
    # the activations' rounding, met by weights of deviation ff^-1/2 (6 deviations), and the result's own
    assert ((got - want).abs() <= 2.0 ** -8 * (want.abs() + 6 * act.norm(dim=1, keepdim=True) * ff ** -0.5)).all()


@pytest.mark.parametrize("units", [1, 2, 4, 5, 6, 7, 24])
@pytest.mark.parametrize("groups", [1, 2])
@pytest.mark.parametrize("tokens", [1, 3])
def test_narrow_runs_of_any_length(units, groups, tokens):
    """Runs of one and two row groups, whose units stand in a ring of six: contractions shorter than it, as long, longer; rows in one piece and in two."""
    from lite_llama_amd.kernels.fused_moe import sparse_square_experts

    cus, experts = torch.cuda.get_device_properties(0).multi_processor_count, 16
    width, ff = 128 * units - 8, 16 * (cus * groups // experts)
    g = torch.Generator(device=DEV).manual_seed(units + groups)
    up, down = ((torch.randn(experts, *s, generator=g, device=DEV) * s[1] ** -0.5).bfloat16() for s in ((ff, width), (width, ff)))
    h = torch.randn(tokens, width, generator=g, device=DEV).bfloat16()
    ids = torch.stack([torch.randperm(experts, generator=g, device=DEV) for _ in range(tokens)]).to(torch.int32)
    weights = torch.rand(tokens, experts, generator=g, device=DEV) + 0.1
    got = sparse_square_experts(h, up, down, ids, weights).double()
    for t in range(tokens):
        for k, e in enumerate(ids[t].tolist()):
            act = torch.relu(up[e].double() @ h[t].double() * weights[t, k].double()) ** 2
            want = down[e].double() @ act
            # the activations' rounding, met by weights of deviation ff^-1/2 (6 deviations), and the result's own
            assert ((got[t, k] - want).abs() <= 2.0 ** -8 * (want.abs() + 6 * act.norm() * ff ** -0.5)).all()


@pytest.mark.parametrize("fmt", ["fp8", "int8"])
@pytest.mark.parametrize("width", [256, 768, 1280, 1536, 3072])
@pytest.mark.parametrize("tokens,group", [(1, 128), (2, 4096), (24, 128)])
@pytest.mark.parametrize("interleaved", [False, True])
def test_narrow_runs_of_8_bit_experts(fmt, width, tokens, group, interleaved):
    """The same in 8 bits, scales per row and alike in 16 rows, rows in pieces of 16 and of 32."""
    test_8_bit_experts(fmt, width, 256, 4 if tokens > 2 else 8, tokens, 2, group, interleaved)
