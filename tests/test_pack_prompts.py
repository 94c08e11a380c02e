"""Prefill on the prompts' tokens alone: the packing launch against plain torch, and whole prefills packed against the padded grid."""

import types

import pytest
import torch

from lite_llama_amd.executor.slots import PromptGrid


def _info(lens, longest):
    n = len(lens)
    return types.SimpleNamespace(b_seq_len=torch.tensor(lens), b_start_loc=torch.arange(n, dtype=torch.int32) * longest,
                                 cur_select_index=torch.arange(n * longest, dtype=torch.int32), max_actual_seq_len=longest)


def test_grid_describes_only_the_vectors_it_was_made_with():
    info = _info([3, 5], 5)
    grid = PromptGrid(info, [3, 5])
    assert (grid.batch, grid.longest, grid.total) == (2, 5, 8) and grid.describes(info)
    info.b_seq_len[0] = 4                      # written in place
    assert not grid.describes(info)
    info = _info([3, 5], 5)
    grid = PromptGrid(info, [3, 5])
    info.cur_select_index = info.cur_select_index.clone()
    assert not grid.describes(info)
    info = _info([3, 5], 5)
    grid = PromptGrid(info, [3, 5])
    info.max_actual_seq_len = 6
    assert not grid.describes(info)


@pytest.mark.gpu
@pytest.mark.parametrize("lens", [[1, 2], [255, 256, 257], [1, 600, 1], [37] * 5 + [1], [5] + [3] * 300])
@pytest.mark.parametrize("sel_dtype,len_dtype,expanded", [(torch.int32, torch.int64, True), (torch.int64, torch.int32, False)])
def test_pack_prompts(lens, sel_dtype, len_dtype, expanded):
    from lite_llama_amd.kernels.kv_cache import pack_prompts

    dev, n, longest = "cuda", len(lens), max(lens)
    g = torch.Generator(device=dev).manual_seed(sum(lens))
    ids = torch.randint(0, 1 << 40, (n, 2 * longest), generator=g, device=dev)[:, ::2]     # (strided rows)
    pos = torch.arange(longest, device=dev).unsqueeze(0).expand(n, longest) if expanded else torch.randint(0, 99, (n, longest), generator=g, device=dev)
    sel = torch.randperm(n * longest, generator=g, device=dev).to(sel_dtype)
    keep = torch.tensor([i * longest + j for i, c in enumerate(lens) for j in range(c)], device=dev)
    starts = [sum(lens[:i]) for i in range(n)]
    asked = [i * longest + c - 1 for i, c in enumerate(lens)] + [-1, 0, n * longest, -n * longest - 1]
    want_rows = [s + c - 1 for s, c in zip(starts, lens)] + [sum(lens) - 1, 0, sum(lens), sum(lens)]
    out = pack_prompts(ids, pos, sel, torch.tensor(lens, device=dev, dtype=len_dtype), sum(lens), torch.tensor(asked, device=dev))
    assert torch.equal(out[0][0], ids.reshape(-1)[keep]) and torch.equal(out[1][0], pos.reshape(-1)[keep])
    assert torch.equal(out[2], sel[keep]) and out[2].dtype == sel_dtype
    assert out[3].tolist() == starts and out[4].tolist() == list(lens) and out[5].tolist() == want_rows


@pytest.mark.gpu
@pytest.mark.parametrize("lens", [[9, 2, 5], [70, 33, 64, 1]])
@pytest.mark.parametrize("quant", ["none", "int4", "smoothquant"])
def test_packed_prefill_is_the_padded_one(lens, quant):
    """Rows do not depend on which other rows a projection runs on, up to the engine its row count selects (fp16 sums in another
    order: 2^-10 of a value, carried through two layers)."""
    from lite_llama_amd.executor import SlotRunner
    from lite_llama_amd.model import CausalLM, tiny_geometry
    from lite_llama_amd.quantization import QuantConfig

    cfg = {"none": None, "int4": QuantConfig.int4_groupwise(128), "smoothquant": QuantConfig.smoothquant_per_channel()}[quant]
    model = CausalLM(tiny_geometry()).init_synthetic(3, cfg)
    n, longest = len(lens), max(lens)
    ids = torch.randint(0, 1024, (n, longest), device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    pos = torch.arange(longest, device="cuda").unsqueeze(0).expand(n, longest)
    last = torch.tensor([i * longest + c - 1 for i, c in enumerate(lens)], device="cuda")
    got = []
    for packed in (True, False):
        runner = SlotRunner(model, n + 1, longest)
        runner.enable_slot_kv_cache().begin_prefill(list(range(n)), lens)
        info = runner.atten_info
        assert model._packs(ids, pos, info, last)
        if not packed:
            info.prompt_grid = None
        logits = model(ids, pos, info, logits_rows=last)
        assert info.b_seq_len.tolist() == list(lens)   # (the caller's struct is as it was)
        kv = [p.view(n + 1, longest, *p.shape[1:])[i, :c] for p in info.kv_buffer for i, c in enumerate(lens)]
        got.append([logits] + kv)
    for a, b in zip(*got):
        assert (a.float() - b.float()).norm() <= 4e-3 * b.float().norm()
    with torch.inference_mode():
        runner.enable_slot_kv_cache().begin_prefill(list(range(n)), lens)
        assert runner.atten_info.prompt_grid is None
        model(ids, pos, runner.atten_info, logits_rows=last)
