"""cos / sin rows of a prefill in one launch, against the tensor operations they replace; the last norm on the rows that are asked for."""

import types

import pytest
import torch

from lite_llama_amd.kernels.norm_act import rotary_rows
from lite_llama_amd.model import CausalLM, RotaryEmbedding, tiny_geometry

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("index", [torch.int32, torch.int64])
@pytest.mark.parametrize("batch,seq,half", [(1, 1, 1), (1, 37, 32), (3, 129, 64), (2, 5, 48), (1, 4096, 64)])
def test_rows_are_those_of_the_tensor_operations(dtype, index, batch, seq, half):
    rope = RotaryEmbedding(tiny_geometry(hidden_size=64, intermediate_size=64, num_layers=1, num_heads=1, num_kv_heads=1, head_dim=2 * half,
                                         vocab_size=8)).to(DEV)
    for pos in (torch.arange(seq, device=DEV, dtype=index).unsqueeze(0).expand(batch, seq),
                torch.randint(0, 1 << 20, (seq, batch), device=DEV, dtype=index).t()):
        cos, sin = rotary_rows(pos, rope.inv_freq, dtype)
        want = rope._tables(pos, dtype)
        assert cos.shape == want[0].shape and cos.is_contiguous() and torch.equal(cos, want[0]) and torch.equal(sin, want[1])
    assert rotary_rows(pos, rope.inv_freq.double(), dtype) is None and rotary_rows(pos.cpu(), rope.inv_freq, dtype) is None


def test_tables_of_another_kind_are_asked():
    class Scaled(RotaryEmbedding):
        def _tables(self, pos, dtype):
            cos, sin = super()._tables(pos, torch.float32)
            return (1.5 * cos).to(dtype), (1.5 * sin).to(dtype)

    geo = tiny_geometry(head_dim=64)
    plain, scaled, patched = RotaryEmbedding(geo).to(DEV), Scaled(geo).to(DEV), RotaryEmbedding(geo).to(DEV)
    patched._tables = scaled._tables
    x, pos = torch.zeros(1, device=DEV, dtype=torch.float16), torch.arange(37, device=DEV)[None]
    for rope in (scaled, patched):
        for got, want in zip(rope(x, pos), scaled._tables(pos, torch.float16)):
            assert torch.equal(got, want)
    assert torch.equal(plain(x, pos)[0], plain._tables(pos, torch.float16)[0]) and not torch.equal(plain(x, pos)[0], scaled(x, pos)[0])


def _prompt(seq, **kw):
    """A model and a prompt of ``seq`` tokens: what its ``forward`` takes."""
    geo = tiny_geometry(hidden_size=128, intermediate_size=256, num_layers=2, num_heads=4, num_kv_heads=2, head_dim=32, vocab_size=64, **kw)
    with torch.device(DEV):
        model = CausalLM(geo)
    g = torch.Generator().manual_seed(1)
    with torch.no_grad():
        for p in model.parameters():
            p.copy_((torch.randn(p.shape, generator=g) * 0.1 + (1.0 if p.dim() == 1 else 0.0)).to(p.dtype))
    ids = torch.randint(0, 64, (1, seq), generator=g).to(DEV)
    info = types.SimpleNamespace(kv_buffer=[torch.zeros(seq, 4, 32, dtype=torch.float16, device=DEV) for _ in range(2)],
                                 cur_select_index=torch.arange(seq, dtype=torch.int32, device=DEV),
                                 b_req_tokens_table=torch.arange(seq, dtype=torch.int32, device=DEV)[None],
                                 b_start_loc=torch.zeros(1, dtype=torch.int32, device=DEV), b_req_idx=torch.zeros(1, dtype=torch.int32, device=DEV),
                                 b_seq_len=torch.tensor([seq], dtype=torch.int32, device=DEV), max_actual_seq_len=seq)
    return model, ids, torch.arange(seq, device=DEV)[None], info


@pytest.mark.parametrize("experts", [0, 4])
@pytest.mark.parametrize("form", ["indices", "table", "mask", "list", "slice", "one", "none"])
def test_every_form_of_asking_for_rows(experts, form):
    """More than 192 tokens, the last layer's update a tensor or the rows of its experts: whatever indexes the rows of the logits does."""
    from lite_llama_amd.model import _rows_of
    from lite_llama_amd.kernels.norm_act import SlotSums

    seq = 260
    model, ids, pos, info = _prompt(seq, num_experts=experts, num_experts_per_tok=2 if experts else 0, moe_intermediate_size=128 if experts else 0)
    rows = {"indices": torch.tensor([seq - 1, 0, 17, 17], device=DEV), "table": torch.tensor([[3, 259], [0, 3]], device=DEV),
            "mask": torch.arange(seq, device=DEV) % 50 == 7, "list": [5, 200], "slice": slice(3, 100, 9), "one": torch.tensor(259, device=DEV),
            "none": torch.zeros(0, dtype=torch.int64, device=DEV)}[form]
    every = model(ids, pos, info).view(seq, -1)
    some = model(ids, pos, info, logits_rows=rows)
    want = every[rows]
    assert some.shape == want.shape
    # (the head's product over few rows and over 260 rounds its sums in another order: one unit of fp16)
    assert torch.allclose(some.float(), want.float(), rtol=2e-3, atol=2e-3 * every.abs().max().item())
    if form != "none":   # (the rows of the experts' sums themselves)
        parts = torch.randn(seq, 2, 128, device=DEV).half()
        done, picked, residual = _rows_of(SlotSums(parts, (1, seq, 128)), torch.randn(1, seq, 128, device=DEV).half(), rows)
        assert done and residual.shape == (*want.shape[:-1], 128) and torch.equal(picked.materialise(), SlotSums(parts, (seq, 128)).materialise()[rows])


def test_logits_of_few_rows_are_those_of_all():
    geo = tiny_geometry(hidden_size=128, intermediate_size=256, num_layers=2, num_heads=4, num_kv_heads=2, head_dim=32, vocab_size=64)
    with torch.device(DEV):
        model = CausalLM(geo)
    g = torch.Generator().manual_seed(1)
    with torch.no_grad():
        for p in model.parameters():
            p.copy_((torch.randn(p.shape, generator=g) * 0.1 + (1.0 if p.dim() == 1 else 0.0)).to(p.dtype))
    seq = 260
    ids = torch.randint(0, 64, (1, seq), generator=g).to(DEV)
    info = types.SimpleNamespace(kv_buffer=[torch.zeros(seq, 4, 32, dtype=torch.float16, device=DEV) for _ in range(2)],
                                 cur_select_index=torch.arange(seq, dtype=torch.int32, device=DEV),
                                 b_req_tokens_table=torch.arange(seq, dtype=torch.int32, device=DEV)[None],
                                 b_start_loc=torch.zeros(1, dtype=torch.int32, device=DEV), b_req_idx=torch.zeros(1, dtype=torch.int32, device=DEV),
                                 b_seq_len=torch.tensor([seq], dtype=torch.int32, device=DEV), max_actual_seq_len=seq)
    pos = torch.arange(seq, device=DEV)[None]
    rows = torch.tensor([seq - 1, 0, 17, 17], device=DEV)
    every = model(ids, pos, info).view(seq, -1)
    some = model(ids, pos, info, logits_rows=rows)
    # (the head's product over 4 rows and over 260 rounds its sums in another order: one unit of fp16)
    assert torch.allclose(some.float(), every[rows].float(), rtol=2e-3, atol=2e-3 * every.abs().max().item())
