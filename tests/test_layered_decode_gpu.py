"""Steps of decoded tokens through layers called as one native call (csrc/layered_decode.hip) against the modules' single launches: the same bits in the
logits and in everything the cache keeps, over every mixer and feed-forward, each route of a projection, one token and the most of a step; what is not
plain goes through the modules."""

import copy
import ctypes

import pytest
import torch

from tests import _nivotar as T

pytestmark = pytest.mark.gpu
DEV = "cuda"
DECAYS = [1.0 - 2.0 ** -(5 + 3 * i / 15) for i in range(16)]
LARGE = T.config([T.parallel(16, 4, 128, 128, 512, 64, 32, 64, 128, 4, 4, 4, mlp=T.dense(5632)), T.gla(8, 128, 256, 8.0, 16, mlp=T.moe(8, 2, 4, 704)),
                  T.lightning(16, 128, 128, DECAYS)], width=2048, vocab=64)


def _model(cfg, dtype):
    from lite_llama_amd.model_layers import LayeredGeometry, LayeredLM

    cfg = copy.deepcopy(cfg)
    for entry in cfg["layers"]:
        if "_rank" in entry:
            entry["mixer"]["rank"] = entry.pop("_rank")
    return LayeredLM(LayeredGeometry.from_config(cfg, name="nivotar"), dtype=dtype).init_synthetic(3, DEV)


def _run(model, batch, steps=3):
    from lite_llama_amd.executor.ragged import RaggedRunner

    g = torch.Generator().manual_seed(batch)
    runner = RaggedRunner(model, 64 * batch, batch, block_size=16, device=DEV)
    slots = [runner.admit() for _ in range(batch)]
    draw = lambda count: torch.randint(0, model.geo.vocab_size, (count,), generator=g).tolist()  # noqa: E731
    runner.step([(s, draw(3 + i % 5)) for i, s in enumerate(slots)])
    logits = [runner.step([(s, draw(1)) for s in slots]) for _ in range(steps)]
    kept = [t for group in (runner.cache.recurrent, runner.cache.conv) for t in group if t is not None]
    kept += [t for pair in runner.cache.kv_buffer if pair is not None for t in (pair if isinstance(pair, (tuple, list)) else [pair])]
    runner.check_errors()
    return logits, kept


def _count(monkeypatch):
    from lite_llama_amd import model_layers

    served, real = [], model_layers.decode_layer

    def counted(*args):
        out = real(*args)
        served.append(out is not None)
        return out

    monkeypatch.setattr(model_layers, "decode_layer", counted)
    return served


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("name,batch", [("mix", 1), ("mix", 12), ("mix", 33), ("mix", 64), ("large", 1), ("large", 16), ("large", 17), ("large", 32), ("large", 50)])
def test_the_same_bits_as_single_launches(monkeypatch, name, batch, dtype):
    from lite_llama_amd import model_layers

    model = _model(LARGE if name == "large" else T.CONFIGS[name], dtype)
    served = _count(monkeypatch)
    got, kept = _run(model, batch)
    layers = len(model.run_order)
    assert len(served) == 4 * layers and not any(served[:layers])
    if not (name == "large" and batch > 32):      # (a projection of more rows than its own kernels take: the library's)
        assert all(served[layers:])
    monkeypatch.setattr(model_layers, "decode_layer", lambda *a: None)
    want, old = _run(model, batch)
    assert all(torch.equal(a, b) for a, b in zip(got, want)) and all(torch.isfinite(a.float()).all() for a in got)
    assert len(kept) == len(old) and all(torch.equal(a, b) for a, b in zip(kept, old))


@pytest.mark.parametrize("what", ["odd", "one", "fp32", "hook", "grad", "env", "switch", "replaced", "eps", "off"])
def test_what_goes_through_the_modules(monkeypatch, what):
    from lite_llama_amd import model_layers

    model = _model(T.CONFIGS[what if what in ("odd", "one") else "mix"], torch.float32 if what == "fp32" else torch.bfloat16)
    first = model.layers[0]
    seen = []
    if what == "hook":
        for layer in model.layers:
            layer.mixer.in_proj.register_forward_hook(lambda *a: seen.append(1))
    if what == "env":
        monkeypatch.setenv("LL_DENSE16_NARROW_OFF", "1")
    if what == "switch":
        monkeypatch.setenv("LL_NO_LAYER_CALLS", "1")
    if what == "eps":
        for layer in model.layers:
            layer.mixer.eps = 0.5          # (its own norms', not the layer's)
    if what == "replaced":
        first.mixer.in_proj.weight = torch.nn.Parameter(first.mixer.in_proj.weight.detach().t().contiguous().t(), requires_grad=False)
    if what == "off":                      # (the rows that open the stack, off a 16-byte border)
        rows_of = model_layers.embed_rows

        def moved(*args):
            x, opening = rows_of(*args)
            room = torch.empty(opening.rows.numel() + 1, dtype=opening.rows.dtype, device=DEV)[1:].view(opening.rows.shape)
            return x, model_layers.FirstRows(room.copy_(opening.rows))

        monkeypatch.setattr(model_layers, "embed_rows", moved)
    if what == "grad":
        inner = model_layers.decode_layer

        def with_grad(*args):
            with torch.enable_grad():
                return inner(*args)

        monkeypatch.setattr(model_layers, "decode_layer", with_grad)
    served = _count(monkeypatch)
    got, _ = _run(model, 2)
    assert not any(served[0::len(model.run_order)]) if what in ("replaced", "off") else not any(served)
    assert not seen or len(seen) == len(served)
    monkeypatch.setattr(model_layers, "decode_layer", lambda *a: None)
    want, _ = _run(model, 2)
    assert all(torch.equal(a, b) for a, b in zip(got, want))


class _Recorded:
    """The library, with a native layer call that is counted and not served: nothing is launched."""

    def __init__(self, lib):
        self._lib, self.asked = lib, 0

    def __getattr__(self, name):
        return getattr(self._lib, name)

    def ll_layered_decode_bytes(self, args, count, *floats):
        self.asked += 1
        self.args = list((ctypes.c_int64 * count).from_address(args))
        return 0


def _places(layer, x, pending, cache, run):
    """Every tensor that the layer's call hands on: (name, its container, its key)."""
    out = [(f"{name}.{key}", module._parameters, key) for name, module in layer.named_modules() for key, p in module._parameters.items()
           if p is not None and (name, key) not in (("", "norm2_weight"), ("mlp", "down_bias"))]      # (these ride on with the result)
    for kind, group in (("recurrent", cache.recurrent), ("conv", cache.conv)):
        if group[run] is not None:
            out.append((kind, group, run))
    for i in range(2 if cache.kv_buffer[run] is not None else 0):
        out.append((f"kv {i}", cache.kv_buffer[run], i))
    keys = ("y", "post_weight", "shared", "shared_scale", "bias") if hasattr(pending, "y") else ("rows",)
    return out + [(key, pending, key) for key in keys if getattr(pending, key) is not None]


@pytest.mark.parametrize("at", [0, 1, 2, 3])
def test_an_operand_elsewhere_is_refused(monkeypatch, at):
    """Every operand of a layer on the host in its turn: the call is refused before it is made, as the modules' wrappers refuse it."""
    from lite_llama_amd import layered_decode, model_layers
    from lite_llama_amd.executor.ragged import RaggedRunner

    model = _model(T.CONFIGS["mix"], torch.bfloat16)
    lib, real, checked = _Recorded(layered_decode.L.lib()), model_layers.decode_layer, []

    def look(layer, x, pending, step, cache, run, table, *kinds):
        if layer is not model.layers[at] or step.longest_run != 1:
            return real(layer, x, pending, step, cache, run, table, *kinds)
        cache.kv_buffer[run] = list(cache.kv_buffer[run]) if cache.kv_buffer[run] is not None else None
        with monkeypatch.context() as m:
            m.setattr(layered_decode.L, "lib", lambda: lib)
            m.setattr(layered_decode.L, "has", lambda name: True)

            def asked(x=x, table=table):
                lib.asked = 0
                assert real(layer, x, pending, step, cache, run, table, *kinds) is None
                return lib.asked

            assert asked() == 1
            assert asked(x=x.cpu()) == 0 and asked(table=table.cpu()) == 0
            for name, held, key in _places(layer, x, pending, cache, run):
                own = held[key] if isinstance(held, (dict, list)) else getattr(held, key)
                away = torch.nn.Parameter(own.detach().cpu(), requires_grad=False) if isinstance(own, torch.nn.Parameter) else own.cpu()
                put = held.__setitem__ if isinstance(held, (dict, list)) else lambda k, v: setattr(held, k, v)
                put(key, away)
                assert asked() == 0, name
                put(key, own)
                checked.append(name)
            assert asked() == 1
        return real(layer, x, pending, step, cache, run, table, *kinds)

    monkeypatch.setattr(model_layers, "decode_layer", look)
    runner = RaggedRunner(model, 64, 1, block_size=16, device=DEV)
    slot = runner.admit()
    runner.step([(slot, [1, 2, 3])])
    assert torch.isfinite(runner.step([(slot, [4])]).float()).all()
    assert len(checked) >= 8


def test_a_layer_reads_the_step_as_it_is(monkeypatch):
    """A step's vector that is replaced between two layers: the next layer is handed the new one."""
    from lite_llama_amd import layered_decode, model_layers
    from lite_llama_amd.executor.ragged import RaggedRunner

    model = _model(T.CONFIGS["mix"], torch.bfloat16)
    lib, real, seen = _Recorded(layered_decode.L.lib()), model_layers.decode_layer, []

    def look(layer, x, pending, step, *rest):
        if step.longest_run == 1:
            step.tok_pos = step.tok_pos.clone()
            seen.append(step.tok_pos)
            with monkeypatch.context() as m:
                m.setattr(layered_decode.L, "lib", lambda: lib)
                assert real(layer, x, pending, step, *rest) is None
            assert step.tok_pos.data_ptr() in lib.args
        return None

    monkeypatch.setattr(model_layers, "decode_layer", look)
    runner = RaggedRunner(model, 64, 1, block_size=16, device=DEV)
    slot = runner.admit()
    runner.step([(slot, [1, 2, 3])])
    runner.step([(slot, [4])])
    assert len(seen) == len(model.run_order) > 1
