"""Which layers of a short prefill go out in one host call (prefill_layers.py) and which prefills run on the prompts' tokens alone
(model.py::CausalLM._packs), without a GPU: tensors that call themselves GPU tensors, and a library that notes what it is asked for."""

import types

import pytest
import torch
from torch import nn

import lite_llama_amd.prefill_layers as P
from lite_llama_amd.model import CausalLM, RotaryEmbedding, tiny_geometry


@pytest.fixture
def plain(monkeypatch):
    """A two-layer model with merged projections, a pass over 5 tokens of it, and the layer calls that reached the library."""
    monkeypatch.setattr(torch.Tensor, "is_cuda", True)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    calls = []
    monkeypatch.setattr(P.L, "lib", lambda: types.SimpleNamespace(ll_prefill_layer16=lambda *a: (calls.append(a), 0)[1]))
    monkeypatch.setattr(P.L, "has", lambda name: True)
    monkeypatch.setattr(P.L, "stream_ptr", lambda: 0)
    model = CausalLM(tiny_geometry())
    info = types.SimpleNamespace(cur_select_index=torch.arange(5), b_start_loc=torch.zeros(1, dtype=torch.int32), b_seq_len=torch.tensor([5]),
                                 max_actual_seq_len=5, kv_buffer=[torch.zeros(8, 4, 64, dtype=torch.float16)] * 2)
    hidden = torch.zeros(1, 5, 256, dtype=torch.float16)
    position = RotaryEmbedding(model.geo)(hidden, torch.arange(5)[None])

    def issued():
        """Whether layer 0 goes out in one call."""
        del calls[:]
        short = P.ShortPrefill.of(model, hidden, position, info)
        if short is not None:
            assert short.layer(model.layers[0], 0, hidden.clone(), None) is None   # (the library declines)
        return len(calls) == 1

    assert issued()
    return types.SimpleNamespace(model=model, info=info, issued=issued)


def _meta(t):
    return torch.empty_like(t, device="meta")


@pytest.mark.parametrize("what", ["input_layernorm_weight", "post_attention_layernorm_weight", "o_proj", "down_proj", "bias", "pool", "lens", "starts",
                                  "select"])
def test_tensors_on_another_device_keep_the_layers_own_forward(plain, what):
    layer, info = plain.model.layers[0], plain.info
    if "layernorm" in what:
        setattr(layer, what, nn.Parameter(_meta(getattr(layer, what)), requires_grad=False))
    elif what in ("o_proj", "down_proj"):
        module = layer.self_attn.o_proj if what == "o_proj" else layer.mlp.down_proj
        module.weight = nn.Parameter(_meta(module.weight), requires_grad=False)
    elif what == "bias":
        layer.self_attn._qkv._holder.bias = _meta(layer.self_attn._qkv._holder.bias)
    elif what == "pool":
        info.kv_buffer = [_meta(t) for t in info.kv_buffer]
    else:
        name = {"lens": "b_seq_len", "starts": "b_start_loc", "select": "cur_select_index"}[what]
        setattr(info, name, _meta(getattr(info, name)))
    assert not plain.issued()


@pytest.mark.parametrize("what", ["o_proj", "down_proj"])
def test_a_bias_behind_a_row_parallel_projection_is_added_by_the_layer(plain, what):
    layer = plain.model.layers[0]
    module = layer.self_attn.o_proj if what == "o_proj" else layer.mlp.down_proj
    module.bias = nn.Parameter(torch.ones(256, dtype=torch.float16), requires_grad=False)
    assert not plain.issued()


@pytest.mark.parametrize("switch", ["LL_DENSE16_ROWS_OFF", "LL_DENSE_NO_PARTIALS", "LL_DENSE16_OFF", "LL_DENSE16_NARROW_OFF", "LL_NO_LAYER_CALLS"])
def test_switches_of_the_routes_that_a_call_contains(plain, monkeypatch, switch):
    monkeypatch.setenv(switch, "1")
    assert not plain.issued()


@pytest.fixture
def grid(plain):
    """Whether two prompts of 2 and 5 tokens on a grid of 10 run packed through the model."""
    from lite_llama_amd.executor.slots import PromptGrid

    info = types.SimpleNamespace(b_seq_len=torch.tensor([2, 5]), b_start_loc=torch.arange(2, dtype=torch.int32) * 5,
                                 cur_select_index=torch.arange(10, dtype=torch.int32), max_actual_seq_len=5)
    info.prompt_grid = PromptGrid(info, [2, 5])
    ids, positions, last = torch.zeros(2, 5, dtype=torch.int64), torch.arange(5).expand(2, 5), torch.tensor([1, 9])
    assert plain.model._packs(ids, positions, info, last)
    experts = CausalLM(tiny_geometry(num_experts=8, num_experts_per_tok=2, moe_intermediate_size=64, use_qk_norm=True))
    assert experts._packs(ids, positions, info, last)
    return types.SimpleNamespace(model=plain.model, packs=lambda: plain.model._packs(ids, positions, info, last))


@pytest.mark.parametrize("at", ["embed_tokens", "layers.1", "layers.0.self_attn.attn", "layers.1.mlp.down_proj"])
@pytest.mark.parametrize("hook", ["register_forward_hook", "register_forward_pre_hook", "register_full_backward_hook"])
def test_hooks_see_the_grid(grid, at, hook):
    handle = getattr(grid.model.get_submodule(at), hook)(lambda *a: None)
    assert not grid.packs()
    handle.remove()
    assert grid.packs()


def test_modules_of_other_origin_see_the_grid(grid):
    model, attention = grid.model, grid.model.layers[0].self_attn

    class Other(type(attention)):
        pass

    handle = torch.nn.modules.module.register_module_forward_hook(lambda *a: None)
    assert not grid.packs()
    handle.remove()
    model.layers[0].self_attn = nn.Identity()
    assert not grid.packs()
    model.layers[0].self_attn = attention
    attention.__class__ = Other
    assert not grid.packs()
    attention.__class__ = Other.__bases__[0]
    model.layers[1].forward = types.MethodType(type(model.layers[1]).forward, model.layers[1])
    assert not grid.packs()
    del model.layers[1].forward
    model.register_forward_hook(lambda *a: None)   # (the model's own inputs and logits are the same either way)
    assert grid.packs()


def test_more_prompts_than_the_packing_launch_takes_run_on_the_grid(grid):
    from lite_llama_amd.executor.slots import PromptGrid

    for n in (65534, 65535):
        info = types.SimpleNamespace(b_seq_len=torch.ones(n), b_start_loc=torch.zeros(n), cur_select_index=torch.zeros(2 * n), max_actual_seq_len=2)
        info.prompt_grid = PromptGrid(info, [1] * (n - 1) + [2])
        ids = torch.zeros(n, 2, dtype=torch.int64)
        assert grid.model._packs(ids, ids, info, torch.tensor([0])) == (n == 65534)
