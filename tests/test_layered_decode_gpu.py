"""Steps of decoded tokens through layers called as one native call (csrc/layered_decode.hip) against the modules' single launches: the same bits in the
logits and in everything the cache keeps, over every mixer and feed-forward, each route of a projection, one token and the most of a step; what is not
plain goes through the modules."""

import copy

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
@pytest.mark.parametrize("name,batch", [("mix", 1), ("mix", 33), ("mix", 64), ("large", 1), ("large", 17), ("large", 32), ("large", 50)])
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


@pytest.mark.parametrize("what", ["odd", "one", "fp32", "hook", "grad", "env", "replaced"])
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
    if what == "replaced":
        first.mixer.in_proj.weight = torch.nn.Parameter(first.mixer.in_proj.weight.detach().t().contiguous().t(), requires_grad=False)
    if what == "grad":
        inner = model_layers.decode_layer

        def with_grad(*args):
            with torch.enable_grad():
                return inner(*args)

        monkeypatch.setattr(model_layers, "decode_layer", with_grad)
    served = _count(monkeypatch)
    got, _ = _run(model, 2)
    assert not any(served[0::len(model.run_order)]) if what == "replaced" else not any(served)
    assert not seen or len(seen) == len(served)
    monkeypatch.setattr(model_layers, "decode_layer", lambda *a: None)
    want, _ = _run(model, 2)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
