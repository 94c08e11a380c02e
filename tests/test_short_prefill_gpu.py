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
    """Heads of 64 and 128 (heads of 32 keep two launches): a tile of queries and more, one prompt and several of different lengths, which run packed
    into one row (grids: the test below)."""
    model = _model(dtype, layers=2, hidden_size=256, num_heads=heads, num_kv_heads=kv_heads, head_dim=dim)
    want, rows, none = _prefill(model, dtype, lens, False, monkeypatch)
    got, mine, calls = _prefill(model, dtype, lens, True, monkeypatch)
    assert none == 0 and calls == 2
    _near(got, want, dtype, 2)
    for a, b in zip(mine, rows):
        _near(a, b, dtype, 2)


def _grid(model, dtype, lens, by_call, odd, monkeypatch):
    """(logits of the last tokens, the pools' rows) of a prefill that runs the padded grid; ``odd``: pools that begin off the 16-byte pieces."""
    from lite_llama_amd.executor import SlotRunner

    longest, batch = max(lens), len(lens)
    runner = SlotRunner(model, batch + 1, longest, device=DEV, kv_dtype=dtype)
    slots = runner.enable_slot_kv_cache()
    slots.begin_prefill(list(range(batch)), lens)
    info = runner.atten_info
    info.prompt_grid = None
    if odd:
        info.kv_buffer = [torch.zeros(pool.numel() + 8, dtype=dtype, device=DEV)[4:4 + pool.numel()].view(pool.shape) for pool in info.kv_buffer]
        assert all(pool.data_ptr() % 16 for pool in info.kv_buffer)
    for pool in info.kv_buffer:
        pool.fill_(7.0)
    g = torch.Generator(device=DEV).manual_seed(sum(lens))
    grid = torch.randint(0, model.geo.vocab_size, (batch, longest), generator=g, device=DEV)
    positions = torch.arange(longest, device=DEV).unsqueeze(0).expand(batch, longest)
    positions = positions + 5 * torch.arange(batch, device=DEV)[:, None]   # (every sequence at positions of its own)
    last = torch.tensor([i * longest + n - 1 for i, n in enumerate(lens)], device=DEV)
    with monkeypatch.context() as m:
        if not by_call:
            m.setenv("LL_NO_LAYER_CALLS", "1")
        logits = model(grid, positions, info, logits_rows=last)
    return logits, [pool.view(batch + 1, longest, *pool.shape[1:]) for pool in info.kv_buffer]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("lens", [[70, 70], [40, 40, 40], [31, 17, 40], [100, 60], [5, 3, 6, 2], [192], [64, 64, 64]])
@pytest.mark.parametrize("heads,kv_heads,dim", [(4, 2, 64), (2, 1, 128), (6, 2, 64)])
def test_the_grid_in_one_launch_and_in_two(dtype, lens, heads, kv_heads, dim, monkeypatch):
    """Sequences of a grid, each with its own rows of the rotary tables.  Pools off the 16-byte pieces keep the rotation in a launch of its own: both forms leave
    the same bits, cache rows behind a prompt's end among them.  Against the layers' own forward every head of every token by itself."""
    model = _model(dtype, layers=2, hidden_size=256, num_heads=heads, num_kv_heads=kv_heads, head_dim=dim)
    one, rows = _grid(model, dtype, lens, True, False, monkeypatch)
    two, apart = _grid(model, dtype, lens, True, True, monkeypatch)
    own, want = _grid(model, dtype, lens, False, False, monkeypatch)
    assert torch.equal(one, two)
    # (the first layer's rows hang on nothing but the tokens; what attention leaves behind a prompt's end is undefined)
    assert torch.equal(rows[0], apart[0]) and (rows[0][len(lens)] == 7).all() and not (rows[0][:len(lens)] == 7).all(-1).any()
    for i, n in enumerate(lens):
        assert torch.equal(rows[1][i, :n], apart[1][i, :n])
    a, b = rows[0][:len(lens)].double(), want[0][:len(lens)].double()
    # norm, product and rotation are each rounded once on either side, the norm's rounding passed through the product: their sum
    bar = 6 * 2.0 ** (-11 if dtype == torch.float16 else -8)
    assert ((a - b).norm(dim=-1) <= bar * b.norm(dim=-1)).all()
    _near(one.double(), own.double(), dtype, 2)
