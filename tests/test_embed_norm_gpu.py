"""The first norm of a step reading its rows from the embedding table, and the copy of a captured step's inputs in one launch."""

import pytest
import torch
import torch.nn.functional as F

from lite_llama_amd.executor.slots import copy_words
from lite_llama_amd.kernels import skip_rmsnorm
from lite_llama_amd.kernels.norm_act import EmbeddedRows, embed_rmsnorm, skip_rmsnorm_q8

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,n", [(1, 8), (3, 128), (17, 256), (5, 512), (64, 2048), (2, 2056), (7, 4096), (1, 8192)])
def test_first_norm_reads_the_table(dtype, rows, n):
    g = torch.Generator().manual_seed(rows + n)
    table = torch.randn(50, n, generator=g).to(dtype).to(DEV)
    weight = (1 + 0.1 * torch.randn(n, generator=g)).to(dtype).to(DEV)
    ids = torch.randint(0, 50, (rows, 1), generator=g).to(DEV)
    ids[0, 0], ids[-1, 0] = 49, 0
    assert EmbeddedRows.served(ids, table)
    y, r = embed_rmsnorm(EmbeddedRows(ids, table), weight, 1e-6)
    x = F.embedding(ids, table)
    want, _ = skip_rmsnorm(x, None, weight, 1e-6)
    assert y.shape == want.shape and torch.equal(r, x) and torch.equal(y, want)
    if dtype == torch.float16:
        got, r = skip_rmsnorm_q8(EmbeddedRows(ids, table), None, weight, 1e-6)
        want, _ = skip_rmsnorm_q8(x, None, weight, 1e-6)
        assert torch.equal(r, x) and torch.equal(got.q, want.q) and torch.equal(got.scale, want.scale)
    for odd in (50, -1, 1 << 40):   # no such row: nothing outside the table is read
        ids[0, 0] = odd
        y, r = embed_rmsnorm(EmbeddedRows(ids, table), weight, 1e-6)
        assert r[0].isnan().all() and y[0].isnan().all() and (rows == 1 or torch.equal(r[1:], x[1:]))
    assert not EmbeddedRows.served(ids.int(), table) and not EmbeddedRows.served(ids, table[:, 1:]) and not EmbeddedRows.served(ids, table.t())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n", [896, 1536, 2048, 2056, 3584, 4096, 4104, 5120, 8192])
def test_a_wide_first_norm_rounds_as_the_norm_of_rows_does(dtype, n):
    """Rows in one, two and four pieces of 2048 columns, values enough that a product rounded once instead of twice shows (about one in 2^13 does)."""
    g = torch.Generator(device=DEV).manual_seed(n)
    table = torch.randn(500, n, generator=g, device=DEV).to(dtype)
    weight = (1 + 0.1 * torch.randn(n, generator=g, device=DEV)).to(dtype)
    ids = torch.randperm(500, generator=g, device=DEV)[:200].view(200, 1)
    y, r = embed_rmsnorm(EmbeddedRows(ids, table), weight, 1e-6)
    x = F.embedding(ids, table)
    want, _ = skip_rmsnorm(x, None, weight, 1e-6)
    assert torch.equal(r, x) and torch.equal(y, want)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_a_step_without_rows(dtype):
    table, weight = torch.randn(50, 128, device=DEV).to(dtype), torch.ones(128, dtype=dtype, device=DEV)
    for shape in ((0, 1), (3, 0)):
        rows = EmbeddedRows(torch.zeros(shape, dtype=torch.int64, device=DEV), table)
        y, r = embed_rmsnorm(rows, weight, 1e-6)
        assert y.shape == r.shape == (*shape, 128)
        if dtype == torch.float16:
            got, r = skip_rmsnorm_q8(rows, None, weight, 1e-6)
            assert got.q.shape == (0, 128) and got.scale.shape == (0,) and r.shape == (*shape, 128)


@pytest.mark.parametrize("n", [128, 3584])
def test_a_norms_weight_inside_a_flat_tensor(n):
    """Weights that begin where no 16-byte piece does."""
    table, flat = torch.randn(50, n, device=DEV).half(), 1 + 0.1 * torch.randn(n + 8, device=DEV).half()
    ids = torch.arange(20, device=DEV).view(20, 1)
    for at in (1, 2, 4):
        weight = flat[at:at + n]
        y, r = embed_rmsnorm(EmbeddedRows(ids, table), weight, 1e-6)
        want, _ = skip_rmsnorm(F.embedding(ids, table), None, weight.clone(), 1e-6)
        assert torch.equal(y, want)


def test_copies_of_a_steps_inputs():
    src = [torch.randint(0, 1 << 20, (n,), device=DEV, dtype=dt) for n, dt in ((1, torch.int64), (64, torch.int64), (300, torch.int32), (7, torch.int32))]
    dst = [torch.full((s.numel() + 1,), -5, device=DEV, dtype=s.dtype) for s in src]
    copy_words([(d.data_ptr(), s.data_ptr(), s.numel() * s.element_size() // 4) for d, s in zip(dst, src)])
    for d, s in zip(dst, src):
        assert torch.equal(d[:-1], s) and d[-1] == -5


def test_a_hook_on_the_embedding_still_sees_it():
    from lite_llama_amd.model import CausalLM, tiny_geometry
    with torch.device(DEV):
        model = CausalLM(tiny_geometry(hidden_size=64, intermediate_size=128, num_layers=1, num_heads=4, num_kv_heads=2, head_dim=16, vocab_size=32))
    ids = torch.zeros(2, 1, dtype=torch.int64, device=DEV)
    assert isinstance(model._embed(ids), EmbeddedRows)
    assert torch.is_tensor(model._embed(ids.expand(2, 3)))   # a short prefill's own launches
    seen = []
    handle = model.embed_tokens.register_forward_hook(lambda *_: seen.append(1))
    assert torch.is_tensor(model._embed(ids)) and seen
    handle.remove()
    handle = model.layers[0].register_forward_pre_hook(lambda *_: None)
    assert torch.is_tensor(model._embed(ids))
    handle.remove()
