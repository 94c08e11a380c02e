"""Embedding rows that open a layered step, as the residual and as they are."""

import pytest
import torch

from lite_llama_amd.kernels.norm_act import embed_rows

pytestmark = pytest.mark.gpu
DEV = "cuda"


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
