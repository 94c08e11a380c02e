"""A layered step's ends of a sublayer: the norm that adds a projection's split-K planes up itself, and embedding rows as residual and as they
are."""

import pytest
import torch

from lite_llama_amd.kernels.norm_act import GatedUpdate, PartialSums, embed_rows, gated_group_norm

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n,width,groups,planes", [(1, 4, 1, 1), (3, 1024, 1, 4), (7, 1028, 1, 5), (2, 2048, 4, 12), (32, 2048, 1, 4), (5, 4096, 1, 7)])
def test_norm_over_planes(dtype, n, width, groups, planes):
    g = torch.Generator().manual_seed(width + planes)
    y = torch.randn(planes, n, width, generator=g)
    pw, nw = ((1 + 0.1 * torch.randn(width, generator=g)).to(dtype) for _ in range(2))
    bias, own, gate = (torch.randn(*s, generator=g).to(dtype) for s in ((width,), (n, width), (n, width)))
    scale, x = torch.rand(n, generator=g), torch.randn(n, width, generator=g)
    for full in (False, True):
        s = y.double().sum(0)
        if full:
            s = (s + bias.double() + scale.double()[:, None] * own.double()) * torch.sigmoid(gate.double())
        parts = s.view(n, groups, -1)
        s = (parts / torch.sqrt((parts ** 2).mean(-1, keepdim=True) + 1e-6)).view(n, width)
        want_x = x.double() + s * pw.double()
        parts = want_x.view(n, groups, -1)
        want_h = (parts / torch.sqrt((parts ** 2).mean(-1, keepdim=True) + 1e-6)).view(n, width) * nw.double()
        got_x = x.to(DEV)
        sums = PartialSums(y.to(DEV), (n, width), dtype)
        kw = dict(bias=bias.to(DEV), shared=own.to(DEV), shared_scale=scale.to(DEV), gate=gate.to(DEV)) if full else {}
        update = GatedUpdate(sums, pw.to(DEV), **kw)
        pick = update.rows(torch.tensor([n - 1], device=DEV))
        one = x[n - 1:].to(DEV)
        gated_group_norm(one, pick, None, 1e-6, groups)
        h = gated_group_norm(got_x, update, nw.to(DEV), 1e-6, groups)
        # fp32 sums of at most 4096 squares and a hardware sigmoid: 1e-5; then one rounding to the storage type
        assert (got_x.double().cpu() - want_x).abs().max() <= 2e-5 * want_x.abs().max()
        assert torch.equal(one[0], got_x[n - 1])
        assert (h.double().cpu() - want_h).abs().max() <= (6e-4 if dtype == torch.float16 else 5e-3) * want_h.abs().max()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("index", [torch.int32, torch.int64])
@pytest.mark.parametrize("n,width", [(1, 8), (5, 2048), (3, 2056), (2, 4104), (4, 12)])
def test_embedding_rows(dtype, index, n, width):
    table = torch.randn(9, width, device=DEV).to(dtype)
    ids = torch.arange(n, device=DEV, dtype=index)
    x, first = embed_rows(ids, table)
    assert torch.equal(first.rows, table[:n]) and torch.equal(x, table[:n].float())
    ids[n - 1] = 9
    x, first = embed_rows(ids, table)
    assert x[n - 1].isnan().all() and first.rows[n - 1].isnan().all()
    assert embed_rows(ids, table.t().contiguous().t()) is None and embed_rows(ids.cpu(), table) is None
