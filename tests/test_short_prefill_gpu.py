"""The prefill of few tokens through an unquantised model, a host call per layer (csrc/prefill_layer.hip), against the layers' own forward: logits and
cache rows, at the edges of the parts that the tokens go through in; and what has to keep the layers' own forward."""

import types

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _model(dtype, layers=3, **kw):
    from lite_llama_amd.model import CausalLM, RotaryEmbedding, tiny_geometry

    torch.manual_seed(3)
    with torch.device(DEV):
        model = CausalLM(tiny_geometry(num_layers=layers, **kw)).to(dtype)
        model.rotary_emb = RotaryEmbedding(model.geo)
    g = torch.Generator(device=DEV).manual_seed(5)
    for name, p in model.named_parameters():
        std = 0.1 if p.dim() == 1 else 1.0 if "embed" in name else p.shape[-1] ** -0.5
        p.data.copy_(torch.randn(p.shape, generator=g, device=DEV) * std + (1.0 if "norm" in name else 0.0))
    return model


def _prefill(model, dtype, lens, by_call, monkeypatch):
    """(logits, cache rows of every layer, layers that were issued by one call)"""
    import lite_llama_amd.prefill_layers as P
    from lite_llama_amd.executor import SlotRunner

    longest, batch = max(lens), len(lens)
    runner = SlotRunner(model, batch + 1, longest, device=DEV, kv_dtype=dtype)
    slots = runner.enable_slot_kv_cache()
    slots.begin_prefill(list(range(batch)), lens)
    g = torch.Generator(device=DEV).manual_seed(sum(lens))
    grid = torch.randint(0, model.geo.vocab_size, (batch, longest), generator=g, device=DEV)
    positions = torch.arange(longest, device=DEV).unsqueeze(0).expand(batch, longest)
    last = torch.tensor([i * longest + n - 1 for i, n in enumerate(lens)], device=DEV)
    calls, one = [0], P.ShortPrefill.layer

    def layer(self, *a):
        out = one(self, *a)
        calls[0] += out is not None
        return out

    with monkeypatch.context() as m:
        m.setattr(P.ShortPrefill, "layer", layer)
        if not by_call:
            m.setenv("LL_NO_LAYER_CALLS", "1")
        logits = model(grid, positions, runner.atten_info, logits_rows=last).float()
    rows = [torch.cat([pool.view(batch + 1, longest, *pool.shape[1:])[i, :n] for i, n in enumerate(lens)]).float()
            for pool in runner.atten_info.kv_buffer]
    return logits, rows, calls[0]


def _near(a, b, dtype, layers=3):
    # eight roundings to the storage type on a layer's way, every one passed on: their sum as a bound of the 2-norm
    bar = 8 * layers * 2.0 ** (-11 if dtype == torch.float16 else -8)
    assert (a - b).norm() <= bar * b.norm()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("lens", [[2], [64], [65], [128], [129], [192], [31, 17, 40], [3, 3], [100, 60]])
def test_like_the_layers(dtype, lens, monkeypatch):
    model = _model(dtype)
    want, rows, none = _prefill(model, dtype, lens, False, monkeypatch)
    got, mine, calls = _prefill(model, dtype, lens, True, monkeypatch)
    assert none == 0 and calls == 3
    _near(got, want, dtype)
    for a, b in zip(mine, rows):
        _near(a, b, dtype)


def test_what_keeps_the_layers_own_forward(monkeypatch):
    dtype = torch.float16
    model = _model(dtype)
    assert _prefill(model, dtype, [193], True, monkeypatch)[2] == 0
    want, _, calls = _prefill(model, dtype, [70], True, monkeypatch)
    assert calls == 3
    seen = []
    hook = model.layers[1].mlp.register_forward_hook(lambda *a: seen.append(1))   # (this layer and those behind it run themselves)
    got, _, calls = _prefill(model, dtype, [70], True, monkeypatch)
    hook.remove()
    assert calls == 1 and seen == [1]
    _near(got, want, dtype)
    model.layers[0].forward = types.MethodType(type(model.layers[0]).forward, model.layers[0])
    assert _prefill(model, dtype, [70], True, monkeypatch)[2] < 3
    del model.layers[0].forward
    odd = _model(dtype, intermediate_size=480)   # a contraction that the split-K engine declines
    assert _prefill(odd, dtype, [20], True, monkeypatch)[2] == 0
    normed = _model(dtype, use_qk_norm=True)
    assert _prefill(normed, dtype, [20], True, monkeypatch)[2] == 0


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("lens", [[1, 2], [37], [65], [31, 17, 40], [70, 90], [192]])
@pytest.mark.parametrize("heads,kv_heads,dim", [(4, 2, 64), (2, 1, 128), (6, 2, 64), (8, 4, 32)])
def test_rotation_and_attention_in_one_launch(dtype, lens, heads, kv_heads, dim, monkeypatch):
    """Heads of 64 and 128 (heads of 32 keep two launches): a tile of queries and more, prompts of one length and of several, whose places
    behind a prompt's end are written to the cache as well."""
    model = _model(dtype, layers=2, hidden_size=256, num_heads=heads, num_kv_heads=kv_heads, head_dim=dim)
    want, rows, none = _prefill(model, dtype, lens, False, monkeypatch)
    got, mine, calls = _prefill(model, dtype, lens, True, monkeypatch)
    assert none == 0 and calls == 2
    _near(got, want, dtype, 2)
    for a, b in zip(mine, rows):
        _near(a, b, dtype, 2)
