"""Grouped expert products over sorted blocks of 128 rows (csrc/moe_sparse.hip) against 64-bit products of the same operands: experts
whose last block holds one row, a row tile, a row more; contractions and widths off every tile; the plain form over the same order."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, F64 = "cuda", torch.float64


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("width,ff", [(8, 8), (72, 200), (136, 64), (192, 132), (100, 72), (256, 24), (3000, 1504)])
@pytest.mark.parametrize("form", ["silu", "clamped", "square"])
def test_experts_of_every_load(dtype, width, ff, form):
    from lite_llama_amd.kernels.fused_moe import sparse_glu_experts, sparse_square_experts

    loads = [1, 0, 31, 32, 33, 64, 65, 96, 127, 128, 129, 300]
    experts, top = len(loads), 2
    g = torch.Generator(device=DEV).manual_seed(width + ff)

    def r(*s, std=1.0):
        return (torch.randn(*s, generator=g, device=DEV) * std).to(dtype)

    ids = torch.cat([torch.full((c,), e) for e, c in enumerate(loads)] + [torch.full((sum(loads) % 2,), 11)])
    ids = ids[torch.randperm(ids.numel(), generator=torch.Generator().manual_seed(1))].view(-1, top).to(torch.int32).to(DEV)
    if form != "square":
        ids[5, 1] = experts + 3          # a slot that no expert serves
    n = ids.shape[0]
    h, weights = r(n, width), torch.rand(n, top, generator=g, device=DEV) + 0.1
    up = r(experts, ff if form == "square" else 2 * ff, width, std=width ** -0.5)
    down = r(experts, width, ff, std=ff ** -0.5)
    if form == "square":
        got = sparse_square_experts(h, up, down, ids, weights)
    else:
        got = sparse_glu_experts(h, up, down, ids, weights, limit=1.5 if form == "clamped" else None, skipped_ids=True)
    want, mid = torch.zeros(n, top, width, dtype=F64, device=DEV), torch.zeros(n, top, 1, dtype=F64, device=DEV)
    for e in range(experts):
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


def test_rows_beyond_32_bit_offsets():
    from lite_llama_amd import _lib as L

    tokens, experts, width, ff, ld = 300, 2, 200, 136, (1 << 23) + 8      # (rows 16 MB apart: the last ones lie 5 GB in)
    g = torch.Generator(device=DEV).manual_seed(3)
    rows = torch.empty((tokens - 1) * ld + width, dtype=torch.bfloat16, device=DEV).as_strided((tokens, width), (ld, 1))
    rows.copy_(torch.randn(tokens, width, generator=g, device=DEV))
    w = (torch.randn(experts, ff, width, generator=g, device=DEV) * width ** -0.5).to(torch.bfloat16)
    ids = torch.randint(0, experts, (tokens, 1), generator=g, device=DEV, dtype=torch.int32)
    block = 128
    padded = tokens + experts * (block - 1)
    meta = torch.empty(experts + padded + -(-padded // block) + 1, dtype=torch.int32, device=DEV)
    srt, owner, post = meta[experts:experts + padded], meta[experts + padded:-1], meta[-1:]
    L.check(L.lib().ll_moe_sort(ids.data_ptr(), tokens, experts, block, meta[:experts].data_ptr(), srt.data_ptr(), owner.data_ptr(),
                                post.data_ptr(), L.stream_ptr()), "moe_sort")
    out = {}
    for name, a in (("far", rows), ("near", rows.contiguous())):
        out[name] = torch.empty(tokens, ff, dtype=torch.bfloat16, device=DEV)
        L.check(L.lib().ll_moe_rows_gemm(a.data_ptr(), a.stride(0), 1, w.data_ptr(), w.stride(0), width, ff, 0, 0, out[name].data_ptr(), ff,
                                         srt.data_ptr(), owner.data_ptr(), post.data_ptr(), tokens, experts, block, 0.0,
                                         L.dtype_code(torch.bfloat16), L.stream_ptr()), "moe_rows_gemm")
    assert torch.equal(out["far"], out["near"])
    want = (rows.to(F64)[:, None] @ w[ids[:, 0].long()].to(F64).transpose(1, 2).contiguous())[:, 0]
    assert ((out["near"].to(F64) - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -18).all()


@pytest.mark.parametrize("slots,experts,block", [(1, 1, 32), (7, 5, 32), (256, 34, 128), (257, 300, 32), (5000, 64, 128), (13057, 3, 128), (900, 9000, 32)])
@pytest.mark.parametrize("skipped", [False, True])
def test_slots_sorted_by_expert(slots, experts, block, skipped):
    """Every expert's slots in their order, padded to blocks; with a run of their own, the slots that no expert serves behind them."""
    from lite_llama_amd import _lib as L

    if skipped and experts > 8192:
        pytest.skip("a run of skipped slots stands beside 8192 experts at most")
    g = torch.Generator().manual_seed(slots)
    ids = torch.randint(-1, experts + 2, (slots,), generator=g, dtype=torch.int32)
    runs = [(e, (ids == e).nonzero()[:, 0].tolist()) for e in range(experts)]
    if skipped:
        runs.append((-1, ((ids < 0) | (ids >= experts)).nonzero()[:, 0].tolist()))
    want, want_expert = [], []
    for e, run in runs:
        blocks = -(-len(run) // block)
        want += run + [slots] * (blocks * block - len(run))
        want_expert += [e] * blocks
    room = slots + (experts + 1) * (block - 1)
    dev = ids.to(DEV)
    counts, out = (torch.empty(k, dtype=torch.int32, device=DEV) for k in (experts, room))
    expert, post = torch.empty(-(-room // block), dtype=torch.int32, device=DEV), torch.empty(1, dtype=torch.int32, device=DEV)
    sort = L.lib().ll_moe_sort_skipped if skipped else L.lib().ll_moe_sort
    L.check(sort(dev.data_ptr(), slots, experts, block, counts.data_ptr(), out.data_ptr(), expert.data_ptr(), post.data_ptr(),
                 L.stream_ptr()), "moe_sort")
    assert post.item() == len(want) and out[:len(want)].tolist() == want and expert[:len(want_expert)].tolist() == want_expert
