"""Embedding rows that open a layered step, as the residual and as they are."""

import pytest
import torch
import torch.nn.functional as F

from lite_llama_amd.kernels.norm_act import EmbeddedRows, embed_rows, embedding

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


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("index", [torch.int32, torch.int64])
@pytest.mark.parametrize("width", [8, 12, 2056])
def test_rows_without_the_residual(dtype, index, width):
    table = torch.randn(9, width, device=DEV).to(dtype)
    for ids in (torch.randint(0, 9, (2, 5), device=DEV, dtype=index), torch.arange(8, device=DEV, dtype=index).view(2, 4).t(),
                torch.tensor(3, device=DEV, dtype=index), torch.zeros(0, 3, device=DEV, dtype=index)):
        assert torch.equal(embedding(ids, table), F.embedding(ids, table))
    assert embedding(ids.cpu(), table) is None and embedding(ids, table.float()) is None and embedding(ids, table[:, 1:]) is None


@pytest.mark.parametrize("index", [torch.int32, torch.int64])
@pytest.mark.parametrize("shape", [(2, 1), (2, 3), (1, 200), (7,)])
def test_an_id_outside_the_table_is_nan_on_every_route(index, shape):
    """Decoded tokens, short prefills, long ones: no route reads past the table."""
    from lite_llama_amd.model import CausalLM, tiny_geometry

    with torch.device(DEV):
        model = CausalLM(tiny_geometry(hidden_size=64, intermediate_size=128, num_layers=1, num_heads=4, num_kv_heads=2, head_dim=16, vocab_size=32))
    ids = torch.randint(0, 32, shape, device=DEV, dtype=index)
    for odd in (32, -1, 1 << 30):
        ids.view(-1)[0] = odd
        rows = model._embed(ids)
        if isinstance(rows, EmbeddedRows):
            assert index == torch.int64 and len(shape) == 2 and (shape[1] == 1 or shape[1] > 192)   # (left to the first norm: tests/test_embed_norm_gpu.py)
            continue
        assert rows.shape == (*shape, 64)
        assert rows.view(-1, 64)[0].isnan().all() and torch.equal(rows.view(-1, 64)[1:], model.embed_tokens.weight[ids.view(-1)[1:].long()])


class Halved(torch.Tensor):
    """A table that means half of what it holds."""

    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        out = super().__torch_function__(func, types, args, kwargs or {})
        return out.as_subclass(torch.Tensor) * 0.5 if func is F.embedding else out


def test_a_table_of_another_class_answers_for_itself():
    from lite_llama_amd.model import CausalLM, tiny_geometry

    with torch.device(DEV):
        model = CausalLM(tiny_geometry(hidden_size=64, intermediate_size=128, num_layers=1, num_heads=4, num_kv_heads=2, head_dim=16, vocab_size=32))
    plain = model.embed_tokens.weight.detach().clone().normal_()
    table = plain.as_subclass(Halved)
    model.embed_tokens._parameters["weight"] = table
    for shape in ((3, 1), (2, 5), (1, 200)):
        ids = torch.randint(0, 32, shape, device=DEV)
        assert embedding(ids, table) is None and embed_rows(ids.view(-1), table) is None and not EmbeddedRows.served(ids, table)
        assert torch.equal(model._embed(ids), plain[ids] * 0.5)
