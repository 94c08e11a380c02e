"""The work that this framework is used for, as cases that can be timed and checked one by one.

Two families of models are served, and both are represented at the widths of the configurations that the framework names:

* llama-shaped models (``CausalLM``) in every weight format that is served -- 4-bit groups, per-channel int8 with dynamic int8
  activations, 8-bit floats in blocks with routed experts, plain 16-bit -- through ``SlotRunner`` / ``SlotBatch``: a captured
  decode step over a ragged running set, and the prefill of newly admitted prompts;
* layered models (``LayeredLM``) through ``RaggedRunner``: whole prompts, generation, and prompt portions next to decoded tokens.

A case runs a stack of a few layers of the model's true widths, heads, experts and vocabulary (a model is the same layers more
often), so that weights are quickly made and a check in 64 bits is affordable.  Weights, cached keys and values and tokens are
random, of the magnitudes that trained models show: unit activations, projections that keep them so, scores of a few units.
"""

from __future__ import annotations

import math
import types

import torch

DEVICE = "cuda"

# ---------------------------------------------------------------------------------------------------------------------- #
# the cases
# ---------------------------------------------------------------------------------------------------------------------- #
# (model, weight format, layers of a decode case, layers of a prefill case)
LLAMA = {
    "qwen2.5-7b": ("int4", 8, 2),
    "llama-3-8b": ("smoothquant", 4, 2),
    "qwen3-30b-a3b": ("fp8", 4, 2),
    "qwen2.5-1.5b": ("bf16", 8, 4),
    "qwen2.5-0.5b": ("f16", 12, 12),
}


def _llama(kind: str, model: str, batch: int, longest: int) -> dict:
    fmt, decode_layers, prefill_layers = LLAMA[model]
    return {"kind": kind, "model": model, "format": fmt, "layers": decode_layers if kind == "decode" else prefill_layers,
            "batch": batch, "longest": longest}


def listed() -> list[dict]:
    return [
        # one user of a chat server at night: a step is nothing but weights and launches
        dict(_llama("decode", "qwen2.5-7b", 1, 300), name="decode_w4a16_1"),
        # the framework's headline: a full running set on 4-bit weights at ordinary contexts
        dict(_llama("decode", "qwen2.5-7b", 64, 700), name="decode_w4a16_64"),
        # a small 16-bit model over long documents: the cache is read more than the weights
        dict(_llama("decode", "qwen2.5-1.5b", 27, 3000), name="decode_bf16_long"),
        # int8 weights and activations, a running set that does not fill the captured batch size
        dict(_llama("decode", "llama-3-8b", 30, 1000), name="decode_w8a8_30"),
        # routed experts in 8-bit floats: nearly every expert is read, few rows each
        dict(_llama("decode", "qwen3-30b-a3b", 64, 600), name="decode_moe_64"),
        # the first answer to one short question: launches and host work
        dict(_llama("prefill", "qwen2.5-0.5b", 1, 37), name="prefill_f16_short"),
        # newly admitted prompts of ordinary lengths, one batch per weight format
        dict(_llama("prefill", "qwen2.5-7b", 16, 509), name="prefill_w4a16"),
        dict(_llama("prefill", "llama-3-8b", 5, 1000), name="prefill_w8a8"),
        dict(_llama("prefill", "qwen3-30b-a3b", 16, 512), name="prefill_moe"),
        # the layered family: whole prompts and the first decoded token after them
        {"kind": "prompts", "size": "compact", "batch": 8, "longest": 512, "steps": 1, "portion": 0, "name": "layered_prompts"},
        # short questions, answers of some length: captured decode steps
        {"kind": "generate", "size": "compact", "batch": 32, "longest": 120, "steps": 24, "portion": 0, "name": "layered_generate"},
        # continuous batching: requests join one after the other and feed portions of their prompts next to decoded tokens
        {"kind": "portions", "size": "wide", "batch": 6, "longest": 700, "steps": 10, "portion": 256, "name": "layered_portions"},
    ]


def _log_int(rng, low: int, high: int) -> int:
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng) -> dict:
    """Decode batches of 1 .. 64 over contexts of 32 .. 4096, prefills of 1 .. 16 prompts of 16 .. 4096 tokens (at most 8192 in
    all), layered steps of 1 .. 32 requests with prompts of 16 .. 1024 (at most 4096 in all)."""
    kind = rng.choice(["decode"] * 4 + ["prefill"] * 3 + ["prompts", "generate", "portions"])
    if kind == "decode":
        batch = _log_int(rng, 1, 64)
        return _llama(kind, rng.choice(sorted(LLAMA)), batch, _log_int(rng, 32, min(4096, 65536 // batch)))
    if kind == "prefill":
        batch = _log_int(rng, 1, 16)
        return _llama(kind, rng.choice(sorted(LLAMA)), batch, _log_int(rng, 16, min(4096, 8192 // batch)))
    batch = _log_int(rng, 1, 8 if kind == "portions" else 32)
    return {"kind": kind, "size": rng.choice(["compact", "wide"]), "batch": batch, "longest": _log_int(rng, 16, min(1024, 4096 // batch)),
            "steps": {"prompts": 1, "generate": rng.randint(4, 24), "portions": rng.randint(4, 10)}[kind],
            "portion": rng.choice([64, 128, 256]) if kind == "portions" else 0}


def _gen(seed: int, salt: int) -> torch.Generator:
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed * 64 + salt)
    return g


def _lengths(case: dict) -> list[int]:
    """Ragged: one sequence is as long as the case says, the others down to half of it."""
    longest, batch = case["longest"], case["batch"]
    r = torch.Generator().manual_seed(64 * longest + batch)
    out = [longest] + torch.randint((longest + 1) // 2, longest + 1, (batch - 1,), generator=r).tolist()
    return [out[i] for i in torch.randperm(batch, generator=r).tolist()]


def _mean_length(case: dict) -> float:
    return (case["longest"] + (case["batch"] - 1) * 0.75 * case["longest"]) / case["batch"]


# ---------------------------------------------------------------------------------------------------------------------- #
# llama-shaped models: weights in the checkpoint's own layouts
# ---------------------------------------------------------------------------------------------------------------------- #
# (hidden, heads, key/value heads, head size, intermediate, vocabulary, epsilon, rotary base, q|k|v bias, experts, top, expert width)
_SHAPES = {
    "qwen2.5-0.5b": (896, 14, 2, 64, 4864, 151936, 1e-6, 1e6, True, 0, 0, 0),
    "qwen2.5-1.5b": (1536, 12, 2, 128, 8960, 151936, 1e-6, 1e6, True, 0, 0, 0),
    "qwen2.5-7b": (3584, 28, 4, 128, 18944, 152064, 1e-6, 1e6, True, 0, 0, 0),
    "llama-3-8b": (4096, 32, 8, 128, 14336, 128256, 1e-5, 5e5, False, 0, 0, 0),
    "qwen3-30b-a3b": (2048, 32, 4, 128, 6144, 151936, 1e-6, 1e6, False, 128, 8, 768),
}
_TIED = ("qwen2.5-0.5b", "qwen2.5-1.5b")
_GROUP = 128


def _dims(case: dict):
    names = "hidden heads kv_heads dim inter vocab eps base bias experts top expert_inter".split()
    return types.SimpleNamespace(**dict(zip(names, _SHAPES[case["model"]])))


def _plain_dtype(case: dict):
    return torch.bfloat16 if case["format"] == "bf16" else torch.float16


def _linear(case: dict, g, prefix: str, out: int, inp: int) -> dict:
    """One projection of standard deviation about 1 / sqrt(inp) under the checkpoint's names."""
    std, fmt = inp ** -0.5, case["format"]
    x = torch.randn(out, inp, generator=g, device=DEVICE)
    if fmt == "int4":
        q = (x * 2.5 + 7.5).round_().clamp_(0, 15).to(torch.int32).view(out, inp // 8, 8)
        words = q[..., 0].clone()
        for j in range(1, 8):
            words |= q[..., j] << (4 * j)
        wiggle = torch.rand(out, inp // _GROUP, generator=g, device=DEVICE)
        zeros = torch.randint(7, 9, (out, inp // _GROUP), generator=g, device=DEVICE).float()
        return {prefix + "weight": words, prefix + "weight_scale": (0.8 + 0.4 * wiggle) * (std / 2.5), prefix + "weight_zeros": zeros}
    if fmt == "smoothquant":
        wiggle = torch.rand(out, 1, generator=g, device=DEVICE)
        return {prefix + "weight": (x * 32).round_().clamp_(-127, 127).to(torch.int8),
                prefix + "weight_scale_inv": (0.8 + 0.4 * wiggle) * (std / 32)}
    if fmt == "fp8":
        wiggle = torch.rand(-(-out // 128), -(-inp // 128), generator=g, device=DEVICE)
        return {prefix + "weight": (x * 100).clamp_(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8),
                prefix + "weight_scale_inv": (0.8 + 0.4 * wiggle) * (std / 100)}
    return {prefix + "weight": (x * std).to(_plain_dtype(case))}


def _layer(case: dict, seed: int, index: int) -> dict:
    """The tensors of decoder layer ``index``, without the ``layers.<index>.`` in front."""
    d, g = _dims(case), _gen(seed, 16 + index)
    plain = _plain_dtype(case)

    def vec(n, mean=0.0, std=0.1):
        return (mean + std * torch.randn(n, generator=g, device=DEVICE)).to(plain)

    t = {"input_layernorm_weight": vec(d.hidden, 1.0), "post_attention_layernorm_weight": vec(d.hidden, 1.0)}
    q, kv = d.heads * d.dim, d.kv_heads * d.dim
    t.update(_linear(case, g, "self_attn.q_proj.", q, d.hidden))
    t.update(_linear(case, g, "self_attn.kv_proj.", 2 * kv, d.hidden))
    t.update(_linear(case, g, "self_attn.o_proj.", d.hidden, q))
    if d.bias:
        t["self_attn.q_proj.bias"], t["self_attn.kv_proj.bias"] = vec(q), vec(2 * kv)
    if not d.experts:
        for name, out, inp in (("gate_proj", d.inter, d.hidden), ("up_proj", d.inter, d.hidden), ("down_proj", d.hidden, d.inter)):
            t.update(_linear(case, g, f"mlp.{name}.", out, inp))
        return t
    t["self_attn.q_norm_weight"], t["self_attn.k_norm_weight"] = vec(d.dim, 1.0), vec(d.dim, 1.0)
    t["mlp.gate_weight"] = (torch.randn(d.experts, d.hidden, generator=g, device=DEVICE) * (2.0 * d.hidden ** -0.5)).to(plain)
    for name, out, inp in (("gate_up_proj", 2 * d.expert_inter, d.hidden), ("down_proj", d.hidden, d.expert_inter)):
        one = _linear(case, g, "", d.experts * out, inp)
        t[f"mlp.experts.{name}"] = one["weight"].view(d.experts, out, inp)
        t[f"mlp.experts.{name}_scale_inv"] = one["weight_scale_inv"].view(d.experts, out // 128, inp // 128)
    return t


def _ends(case: dict, seed: int) -> dict:
    d, g, plain = _dims(case), _gen(seed, 1), _plain_dtype(case)
    t = {"embed_tokens.weight": torch.randn(d.vocab, d.hidden, generator=g, device=DEVICE).to(plain),
         "norm_weight": (1.0 + 0.1 * torch.randn(d.hidden, generator=g, device=DEVICE)).to(plain)}
    if case["model"] in _TIED:
        t["embed_tokens.weight"] *= 0.05
        t["lm_head_weight"] = t["embed_tokens.weight"]
    else:
        t["lm_head_weight"] = (torch.randn(d.vocab, d.hidden, generator=g, device=DEVICE) * d.hidden ** -0.5).to(plain)
    return t


def _model(case: dict, seed: int):
    from dataclasses import replace

    from lite_llama_amd.model import GEOMETRY, CausalLM, RotaryEmbedding
    from lite_llama_amd.quantization import QuantConfig

    quant = {"int4": QuantConfig.int4_groupwise(_GROUP), "smoothquant": QuantConfig.smoothquant_per_channel(),
             "fp8": QuantConfig.fp8_block(), "bf16": None, "f16": None}[case["format"]]
    with torch.device(DEVICE):
        model = CausalLM(replace(GEOMETRY[case["model"]], num_layers=case["layers"]), quant)
    if case["format"] == "bf16":
        model = model.to(torch.bfloat16)
        with torch.device(DEVICE):
            model.rotary_emb = RotaryEmbedding(model.geo)   # (angles stay in 32 bits)
    tensors = _ends(case, seed)
    for i in range(case["layers"]):
        tensors.update({f"layers.{i}.{name}": v for name, v in _layer(case, seed, i).items()})
    model.load_state_dict(tensors, strict=True)
    del tensors
    model.compact_weights()   # as the checkpoint loader leaves a model
    return model


def _context(case: dict, seed: int, layer: int, slots: int, rows: int) -> torch.Tensor:
    """What earlier steps left in the cache of one layer: ``[slots * rows, 2 * kv_heads, dim]``."""
    d = _dims(case)
    return torch.randn(slots * rows, 2 * d.kv_heads, d.dim, generator=_gen(seed, 40 + layer), device=DEVICE).to(_plain_dtype(case))


def _tokens(case: dict, seed: int, count: int) -> torch.Tensor:
    return torch.randint(0, _dims(case).vocab, (count,), generator=_gen(seed, 2), device=DEVICE)


def _bucket(case: dict) -> int:
    """The smallest captured context length that holds the longest sequence."""
    return next(b for b in (256, 512, 1024, 2048, 4096) if b >= case["longest"])


def _prepare_llama(case: dict, seed: int):
    from lite_llama_amd.executor import SlotRunner

    lens, batch = _lengths(case), case["batch"]
    decode = case["kind"] == "decode"
    model = _model(case, seed)
    row = _bucket(case) if decode else case["longest"]
    size = next(b for b in (1, 2, 4, 8, 16, 32, 64) if b >= batch) if decode else batch
    runner = SlotRunner(model, size + 1, row, device=DEVICE, kv_dtype=_plain_dtype(case))   # (the last slot backs filler rows)
    if decode:
        runner.enable_graphs(batch_sizes=(size,), seq_len_buckets=(row,))
    slots = runner.enable_slot_kv_cache()
    pools = runner.atten_info.kv_buffer
    if decode:
        for i, pool in enumerate(pools):
            pool[:batch * row] = _context(case, seed, i, batch, row)
        padded = slots.begin_decode(list(range(batch)), lens)
        ids = torch.zeros(padded, 1, dtype=torch.long, device=DEVICE)
        ids[:batch, 0] = _tokens(case, seed, batch)
        positions = (slots.seq_lens.long() - 1).view(-1, 1).clone()
        runner.forward(ids, positions)   # the first step of a running set captures it
        return types.SimpleNamespace(runner=runner, ids=ids, positions=positions, batch=batch)
    slots.begin_prefill(list(range(batch)), lens)
    grid = torch.zeros(batch, row, dtype=torch.long, device=DEVICE)
    flat = _tokens(case, seed, sum(lens)).split(lens)
    for i, n in enumerate(lens):
        grid[i, :n] = flat[i]
    last = torch.tensor([i * row + n - 1 for i, n in enumerate(lens)], device=DEVICE)
    positions = torch.arange(row, device=DEVICE).unsqueeze(0).expand(batch, row)
    written = [[pool.view(batch + 1, row, *pool.shape[1:])[i, :n] for i, n in enumerate(lens)] for pool in pools]
    return types.SimpleNamespace(model=model, info=runner.atten_info, grid=grid, positions=positions, last=last, written=written)


def _run_llama(case_state):
    s = case_state
    if hasattr(s, "runner"):
        logits = s.runner.forward(s.ids, s.positions)[:s.batch, 0]
        return {"logits": logits, "cache": s.runner.atten_info.kv_buffer}
    return {"logits": s.model(s.grid, s.positions, s.info, logits_rows=s.last), "cache": s.written}


# ---------------------------------------------------------------------------------------------------------------------- #
# layered models: sliding-window attention beside a state-space mixer, linear attention with a fixed decay and with a decay per
# key entry, experts behind a corrected softmax, the norm on every sublayer's result
# ---------------------------------------------------------------------------------------------------------------------- #
SIZES = {
    "compact": dict(width=2048, heads=16, kv_heads=4, dim=128, vdim=128, rot=64, window=512, ssd_heads=32, ssd_vdim=64, state=128, groups=4,
                    taps=4, parts=4, lin_heads=16, lin_dim=128, lin_vdim=128, gla_heads=8, gla_dim=128, gla_vdim=256, rank=16, ff=5632,
                    experts=32, identity=2, top=4, expert_ff=704, vocab=32768),
    "wide": dict(width=3072, heads=24, kv_heads=8, dim=128, vdim=96, rot=128, window=1024, ssd_heads=48, ssd_vdim=64, state=64, groups=8,
                 taps=4, parts=8, lin_heads=24, lin_dim=64, lin_vdim=128, gla_heads=12, gla_dim=128, gla_vdim=256, rank=32, ff=8192,
                 experts=64, identity=4, top=8, expert_ff=512, vocab=32768),
}
_EPS, _TAU, _LIMIT, _LEFT, _RIGHT, _BASE = 1e-6, 8.0, 7.0, 0.5, 1.5, 10000.0


def _decays(z) -> list[float]:
    return [1.0 - 2.0 ** -(5 + 3 * i / (z.lin_heads - 1)) for i in range(z.lin_heads)]


def _layered_config(z) -> dict:
    moe = {"kind": "moe", "expert": {"ff": z.expert_ff, "limit": _LIMIT},
           "router": {"experts": z.experts, "identity": z.identity, "top": z.top}}
    parallel = {"left": {"heads": z.heads, "kv_heads": z.kv_heads, "dim": z.dim, "vdim": z.vdim, "mask": {"size": z.window},
                         "rot": {"base": _BASE, "dims": z.rot}, "scale": z.dim ** -0.5},
                "right": {"heads": z.ssd_heads, "vdim": z.ssd_vdim, "state": z.state, "groups": z.groups, "conv": z.taps,
                          "norm_groups": z.parts},
                "left_scale": _LEFT, "right_scale": _RIGHT}
    gla = {"heads": z.gla_heads, "dim": z.gla_dim, "vdim": z.gla_vdim, "tau": _TAU, "rank": z.rank}
    lightning = {"heads": z.lin_heads, "dim": z.lin_dim, "vdim": z.lin_vdim, "decay": _decays(z)}
    layers = [{"type": "parallel", "mixer": parallel, "mlp": {"kind": "dense", "ff": z.ff}},
              {"type": "lightning", "mixer": lightning, "mlp": moe},
              {"type": "gla", "mixer": gla, "mlp": moe}, {"type": "gla", "mixer": gla, "mlp": moe}]
    return {"architecture": "Nivotar", "layers": layers, "norm": {"eps": _EPS}, "vocab": z.vocab, "width": z.width}


def _layered_tensors(z, seed: int) -> dict:
    g = _gen(seed, 3)
    t = {}

    def put(name, *shape, std=None, mean=0.0, low=None, high=None):
        if low is not None:
            v = torch.rand(*shape, generator=g, device=DEVICE) * (high - low) + low
        else:
            v = torch.randn(*shape, generator=g, device=DEVICE) * (shape[-1] ** -0.5 if std is None else std) + mean
        t[name] = v.to(torch.bfloat16)

    def norm(name, n):
        put(name, n, std=0.1, mean=1.0)

    put("embed_tokens.weight", z.vocab, z.width, std=1.0)
    norm("norm_weight", z.width)
    inner, gn = z.ssd_heads * z.ssd_vdim, z.groups * z.state
    for i in range(4):
        p, m = f"layers.{i}.", f"layers.{i}.mixer."
        norm(p + "norm1_weight", z.width)
        norm(p + "norm2_weight", z.width)
        if i == 0:
            norm(m + "q_norm_weight", z.heads * z.dim)
            norm(m + "k_norm_weight", z.kv_heads * z.dim)
            put(m + "conv_weight", inner + 2 * gn, z.taps)
            put(m + "conv_bias", inner + 2 * gn, std=0.3)
            put(m + "dt_bias", z.ssd_heads, std=0.5)
            put(m + "a_log", z.ssd_heads, low=-1.0, high=1.0)
            put(m + "skip", z.ssd_heads, low=-1.0, high=1.0)
            norm(m + "ssd_norm_weight", inner)
            put(m + "in_proj.weight", (z.heads + z.kv_heads) * z.dim + z.kv_heads * z.vdim + 2 * inner + 2 * gn + z.ssd_heads, z.width)
            put(m + "out_proj.weight", z.width, z.heads * z.vdim + inner)
            put(p + "mlp.down_bias", z.width, std=0.1)
            put(p + "mlp.in_proj.weight", 2 * z.ff, z.width)
            put(p + "mlp.in_proj.bias", 2 * z.ff, std=0.1)
            put(p + "mlp.down_proj.weight", z.width, z.ff)
            continue
        h, dk, dv = (z.lin_heads, z.lin_dim, z.lin_vdim) if i == 1 else (z.gla_heads, z.gla_dim, z.gla_vdim)
        norm(m + "out_norm_weight", h * dv if i == 1 else dv)
        put(m + "in_proj.weight", 2 * h * dk + 2 * h * dv + (0 if i == 1 else z.rank), z.width)
        put(m + "o_proj.weight", z.width, h * dv)
        if i > 1:
            put(m + "decay_proj.weight", h * dk, z.rank)
            put(m + "decay_bias", h * dk, std=1.0, mean=2.0)
        put(p + "mlp.router_weight", z.experts + z.identity, z.width, std=4.0 * z.width ** -0.5)
        put(p + "mlp.correction", z.experts + z.identity, std=0.02)
        put(p + "mlp.gate_up_weight", z.experts, 2 * z.expert_ff, z.width)
        put(p + "mlp.down_weight", z.experts, z.width, z.expert_ff)
    t["lm_head.weight"] = t["embed_tokens.weight"]
    return t


def _layered_tokens(case: dict, seed: int) -> list[list[int]]:
    """Per request the prompt and the tokens that are fed after it."""
    r = torch.Generator().manual_seed(seed * 64 + 9)
    vocab = SIZES[case["size"]]["vocab"]
    return [torch.randint(0, vocab, (n + case["steps"],), generator=r).tolist() for n in _lengths(case)]


def _schedule(case: dict, lens: list[int]) -> list[list[tuple[int, int, int]]]:
    """The steps of a pass: per step the entries ``(request, first token, token after the last)``."""
    steps, batch = case["steps"], case["batch"]
    if case["kind"] != "portions":
        return [[(i, 0, n) for i, n in enumerate(lens)]] + [[(i, n + k, n + k + 1) for i, n in enumerate(lens)] for k in range(steps)]
    out, at, k = [], [0] * batch, 0
    while any(a < n + steps for a, n in zip(at, lens)):
        entries = []
        for i in range(min(batch, k + 1)):   # request i joins in step i
            if at[i] < lens[i]:
                entries.append((i, at[i], min(at[i] + case["portion"], lens[i])))
            elif at[i] < lens[i] + steps:
                entries.append((i, at[i], at[i] + 1))
        for i, _, stop in entries:
            at[i] = stop
        if entries:
            out.append(entries)
        k += 1
    return out


def _prepare_layered(case: dict, seed: int):
    from lite_llama_amd.executor.ragged import RaggedRunner
    from lite_llama_amd.model_layers import LayeredGeometry, LayeredLM

    z = types.SimpleNamespace(**SIZES[case["size"]])
    with torch.device(DEVICE):
        model = LayeredLM(LayeredGeometry.from_config(_layered_config(z), name="nivotar"), dtype=torch.bfloat16)
    model.load_state_dict(_layered_tensors(z, seed), strict=True)
    lens, tokens = _lengths(case), _layered_tokens(case, seed)
    pages = sum(-(-len(t) // 64) for t in tokens)
    runner = RaggedRunner(model, pages * 64, case["batch"], 64, DEVICE, capture_decode=case["kind"] == "generate")
    steps = [[(i, tokens[i][a:b]) for i, a, b in entries] for entries in _schedule(case, lens)]
    return types.SimpleNamespace(ragged=runner, steps=steps, batch=case["batch"], vocab=z.vocab)


def _run_layered(s):
    slots = [s.ragged.admit() for _ in range(s.batch)]
    out = torch.empty(sum(len(entries) for entries in s.steps), s.vocab, dtype=torch.bfloat16, device=DEVICE)
    at = 0
    for entries in s.steps:   # (a captured step's logits live until the next one: a program that keeps them copies them)
        out[at:at + len(entries)] = s.ragged.step([(slots[i], toks) for i, toks in entries])
        at += len(entries)
    s.ragged.release(slots)
    return out


# ---------------------------------------------------------------------------------------------------------------------- #
# what a measurement calls
# ---------------------------------------------------------------------------------------------------------------------- #
def prepare(case: dict, seed: int):
    return _prepare_llama(case, seed) if "model" in case else _prepare_layered(case, seed)


def run(state):
    with torch.no_grad():
        return _run_layered(state) if hasattr(state, "ragged") else _run_llama(state)


def tolerance(case: dict) -> dict:
    # 16-bit activations between the kernels; a routed token whose last expert is a near tie may take the other one
    return {"rel": 0.03, "max": 0.9}


def _touched(experts: int, top: float, tokens: float) -> float:
    return experts * (1.0 - (1.0 - 1.0 / experts) ** (top * tokens))


def _work_llama(case: dict) -> dict:
    d, batch = _dims(case), case["batch"]
    per = {"int4": 0.5 + 8.0 / _GROUP, "smoothquant": 1.0, "fp8": 1.0, "bf16": 2.0, "f16": 2.0}[case["format"]]
    mean = _mean_length(case)
    tokens = batch * (1 if case["kind"] == "decode" else mean)
    attn = d.hidden * (d.heads + 2 * d.kv_heads) * d.dim + d.heads * d.dim * d.hidden
    if d.experts:
        expert = 3 * d.hidden * d.expert_inter
        weights = (attn + _touched(d.experts, d.top, tokens) * expert) * per + d.experts * d.hidden * 2
        active = attn + d.top * expert + d.experts * d.hidden
    else:
        weights, active = (attn + 3 * d.hidden * d.inter) * per, attn + 3 * d.hidden * d.inter
    row = 2 * d.kv_heads * d.dim * 2
    pairs = batch * (mean if case["kind"] == "decode" else mean * (mean + 1) / 2)
    cached = batch * mean * row if case["kind"] == "decode" else tokens * row
    flops = case["layers"] * (2.0 * tokens * active + 4.0 * pairs * d.heads * d.dim) + 2.0 * batch * d.hidden * d.vocab
    return {"bytes": case["layers"] * (weights + cached) + d.hidden * d.vocab * 2 + batch * d.vocab * 2 + tokens * d.hidden * 2, "flops": flops}


def _work_layered(case: dict) -> dict:
    z = types.SimpleNamespace(**SIZES[case["size"]])
    inner, gn = z.ssd_heads * z.ssd_vdim, z.groups * z.state
    first = z.width * ((z.heads + z.kv_heads) * z.dim + z.kv_heads * z.vdim + 2 * inner + 2 * gn + z.ssd_heads + z.heads * z.vdim + inner + 3 * z.ff)
    lin = z.width * (2 * z.lin_heads * z.lin_dim + 3 * z.lin_heads * z.lin_vdim)
    gla = z.width * (2 * z.gla_heads * z.gla_dim + 3 * z.gla_heads * z.gla_vdim + z.rank) + z.rank * z.gla_heads * z.gla_dim
    dense = first + lin + 2 * gla + 3 * (z.experts + z.identity) * z.width
    expert = 3 * z.width * z.expert_ff
    routed = z.top * z.experts / (z.experts + z.identity)
    states = z.ssd_heads * z.state * z.ssd_vdim + z.lin_heads * z.lin_dim * z.lin_vdim + 2 * z.gla_heads * z.gla_dim * z.gla_vdim
    per_token = 2.0 * (dense + 3 * routed * expert) + 4.0 * states
    mean = _mean_length(case)
    lens = [mean] * case["batch"] if case["kind"] != "portions" else [int(mean)] * case["batch"]
    total_bytes = flops = 0.0
    for entries in _schedule(case, lens):
        tokens = sum(b - a for _, a, b in entries)
        total_bytes += 2.0 * (dense + 3 * _touched(z.experts, routed, tokens) * expert + z.vocab * z.width)
        flops += tokens * per_token + 2.0 * len(entries) * z.vocab * z.width
        for _, a, b in entries:
            seen = (b - a) * min(z.window, (a + b) / 2)
            flops += 2.0 * seen * z.heads * (z.dim + z.vdim)
            total_bytes += min(z.window, b) * z.kv_heads * (z.dim + z.vdim) * 2 + (4.0 if a == 0 else 8.0) * states
    return {"bytes": total_bytes, "flops": flops}


def work(case: dict) -> dict:
    return _work_llama(case) if "model" in case else _work_layered(case)


# ---------------------------------------------------------------------------------------------------------------------- #
# the same results in 64 bits
# ---------------------------------------------------------------------------------------------------------------------- #
def _wide_weight(case: dict, t: dict, prefix: str) -> torch.Tensor:
    """A projection's dequantised weight."""
    fmt, w = case["format"], t[prefix + "weight"]
    if fmt == "int4":
        q = torch.stack([(w >> (4 * j)) & 15 for j in range(8)], dim=-1).view(w.shape[0], -1, _GROUP).double()
        q = (q - t[prefix + "weight_zeros"].double()[..., None]) * t[prefix + "weight_scale"].double()[..., None]
        return q.view(w.shape[0], -1)
    if fmt == "smoothquant":
        return w.double() * t[prefix + "weight_scale_inv"].double()
    if fmt == "fp8":
        return _wide_blocks(w, t[prefix + "weight_scale_inv"])
    return w.double()


def _wide_blocks(w, scale):
    n, k = w.shape
    s = scale.double().repeat_interleave(128, 0)[:n].repeat_interleave(128, 1)[:, :k]
    return w.view(torch.float8_e4m3fn).double() * s


def _rms(x, weight, eps):
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)
    return y if weight is None else y * weight.double()


def _project(case, t, prefix, x):
    if case["format"] == "smoothquant":   # activations become int8 codes per row, truncated towards zero
        scale = x.abs().amax(-1, keepdim=True) / 127.0
        x = torch.trunc(x / torch.where(scale > 0, scale, torch.ones_like(scale))) * scale
    y = x @ _wide_weight(case, t, prefix).T
    bias = t.get(prefix + "bias")
    return y if bias is None else y + bias.double()


def _rotate(x, positions, base):
    """``x [n, heads, dim]``: entry i paired with entry i + dim / 2."""
    half = x.shape[-1] // 2
    freq = base ** (-2.0 * torch.arange(half, device=x.device, dtype=torch.float64) / x.shape[-1])
    ang = positions.double()[:, None] * freq
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1)


def _attend(q, k, v, scale, first):
    """Queries ``[n, heads, d]`` at positions ``first ..`` over ``[m, kv_heads, d]`` keys and values."""
    n, heads, _ = q.shape
    kvh = k.shape[1]
    out = []
    for h in range(kvh):   # a group of query heads at a time: full score matrices of long prompts are large
        qs = q[:, h * (heads // kvh):(h + 1) * (heads // kvh)].transpose(0, 1)
        s = (qs @ k[:, h].T) * scale
        t = torch.arange(first, first + n, device=q.device)
        s = s.masked_fill(torch.arange(k.shape[0], device=q.device)[None, :] > t[:, None], -math.inf)
        out.append(torch.softmax(s, -1) @ v[:, h])
    return torch.cat(out, 0).transpose(0, 1)


def _experts(case, d, t, x):
    probs = torch.softmax(x @ t["mlp.gate_weight"].double().T, -1)
    w, ids = torch.topk(probs, d.top, -1)
    w = w / w.sum(-1, keepdim=True)
    y = torch.zeros_like(x)
    for e in range(d.experts):
        rows, slot = (ids == e).nonzero(as_tuple=True)
        if rows.numel() == 0:
            continue
        gate_up = x[rows] @ _wide_blocks(t["mlp.experts.gate_up_proj"][e], t["mlp.experts.gate_up_proj_scale_inv"][e]).T
        g, u = gate_up.chunk(2, -1)
        down = _wide_blocks(t["mlp.experts.down_proj"][e], t["mlp.experts.down_proj_scale_inv"][e])
        y.index_add_(0, rows, ((torch.nn.functional.silu(g) * u) @ down.T) * w[rows, slot, None])
    return y


def _exact_llama(case: dict, seed: int):
    d, batch, decode = _dims(case), case["batch"], case["kind"] == "decode"
    lens = _lengths(case)
    ends = _ends(case, seed)
    dev = ends["norm_weight"].device
    tokens = _tokens(case, seed, batch if decode else sum(lens))
    starts = [0]
    for n in lens:
        starts.append(starts[-1] + (1 if decode else n))
    pos = torch.tensor([n - 1 for n in lens], device=dev) if decode else torch.cat([torch.arange(n, device=dev) for n in lens])
    row = _bucket(case)
    x = ends["embed_tokens.weight"][tokens].double()
    caches = []
    q_size, kv = d.heads * d.dim, d.kv_heads * d.dim
    for i in range(case["layers"]):
        t = _layer(case, seed, i)
        h = _rms(x, t["input_layernorm_weight"], d.eps)
        q = _project(case, t, "self_attn.q_proj.", h).view(-1, d.heads, d.dim)
        k, v = _project(case, t, "self_attn.kv_proj.", h).view(-1, 2, d.kv_heads, d.dim).unbind(1)
        if d.experts:
            q, k = _rms(q, t["self_attn.q_norm_weight"], d.eps), _rms(k, t["self_attn.k_norm_weight"], d.eps)
        q, k = _rotate(q, pos, d.base), _rotate(k, pos, d.base)
        fresh = torch.cat([k, v], 1)
        heads = []
        if decode:
            pool = _context(case, seed, i, batch, row).double().view(batch, row, 2 * d.kv_heads, d.dim)
            for b, n in enumerate(lens):
                pool[b, n - 1] = fresh[b]
                heads.append(_attend(q[b:b + 1], pool[b, :n, :d.kv_heads], pool[b, :n, d.kv_heads:], d.dim ** -0.5, n - 1))
        else:
            for b in range(batch):
                at = slice(starts[b], starts[b + 1])
                heads.append(_attend(q[at], k[at], v[at], d.dim ** -0.5, 0))
            caches.append(list(fresh.split(lens)))
        x = x + _project(case, t, "self_attn.o_proj.", torch.cat(heads, 0).reshape(-1, q_size))
        h = _rms(x, t["post_attention_layernorm_weight"], d.eps)
        if d.experts:
            x = x + _experts(case, d, t, h)
        else:
            act = torch.nn.functional.silu(_project(case, t, "mlp.gate_proj.", h)) * _project(case, t, "mlp.up_proj.", h)
            x = x + _project(case, t, "mlp.down_proj.", act)
        del t
    if not decode:
        x = x[torch.tensor(starts[1:], device=dev) - 1]
    logits = _rms(x, ends["norm_weight"], d.eps) @ ends["lm_head_weight"].double().T
    # (a decode step's pools hold slots that no request owns: their content is no result)
    return {"logits": logits, "cache": None if decode else caches}


def _scan(q, k, v, decay):
    """``q, k [B, T, H, dk]``, ``v [B, T, H, dv]``, ``decay [B, T, H, dk or 1]``: S <- decay S + k v^T, o = S^T q, per token."""
    state = torch.zeros(*q.shape[:1], q.shape[2], q.shape[3], v.shape[3], dtype=q.dtype, device=q.device)
    out = torch.empty_like(v)
    for i in range(q.shape[1]):
        state = decay[:, i, :, :, None] * state + k[:, i, :, :, None] * v[:, i, :, None, :]
        out[:, i] = (q[:, i, :, None, :] @ state)[:, :, 0]
    return out


def _exact_layered(case: dict, seed: int):
    z = types.SimpleNamespace(**SIZES[case["size"]])
    lens, tokens = _lengths(case), _layered_tokens(case, seed)
    b, longest = case["batch"], max(len(t) for t in tokens)
    if b * longest * (z.ssd_heads * z.state * z.ssd_vdim) > 2e11:
        return None
    t = _layered_tensors(z, seed)
    dev = t["norm_weight"].device
    grid = torch.zeros(b, longest, dtype=torch.long)
    for i, row in enumerate(tokens):
        grid[i, :len(row)] = torch.tensor(row)
    x = t["embed_tokens.weight"][grid.to(dev)].double()
    T, silu = longest, torch.nn.functional.silu
    inner, gn = z.ssd_heads * z.ssd_vdim, z.groups * z.state
    for i in range(4):
        p, m = f"layers.{i}.", f"layers.{i}.mixer."
        w = lambda name: t[name].double()  # noqa: E731
        rows = x @ w(m + "in_proj.weight").T
        if i == 0:
            qn, kn, vn = z.heads * z.dim, z.kv_heads * z.dim, z.kv_heads * z.vdim
            q, k, v, gate, ubc, dt = rows.split([qn, kn, vn, inner, inner + 2 * gn, z.ssd_heads], -1)
            q = _rms(q, t[m + "q_norm_weight"], _EPS).view(b, T, z.heads, z.dim)
            k = _rms(k, t[m + "k_norm_weight"], _EPS).view(b, T, z.kv_heads, z.dim)
            v = v.reshape(b, T, z.kv_heads, z.vdim)
            pos, half = torch.arange(T, device=dev, dtype=torch.float64), z.rot // 2
            ang = pos[:, None] * _BASE ** (-2.0 * torch.arange(half, device=dev, dtype=torch.float64) / z.rot)
            cos, sin = ang.cos()[None, :, None], ang.sin()[None, :, None]

            def turn(y):
                a, c = y[..., :half], y[..., half:z.rot]
                return torch.cat([a * cos - c * sin, c * cos + a * sin, y[..., z.rot:]], -1)

            q, k = turn(q), turn(k)
            far = pos[:, None] - pos[None, :]
            hidden = (far < 0) | (far >= z.window)
            heads = []
            for h in range(z.heads):
                g = h // (z.heads // z.kv_heads)
                s = (q[:, :, h] @ k[:, :, g].transpose(1, 2)) * z.dim ** -0.5
                heads.append(torch.softmax(s.masked_fill(hidden, -math.inf), -1) @ v[:, :, g])
            left = torch.cat(heads, -1) * _LEFT
            taps = w(m + "conv_weight")
            conv = torch.nn.functional.pad(ubc, (0, 0, z.taps - 1, 0))
            ubc = silu(sum(conv[:, j:j + T] * taps[:, j] for j in range(z.taps)) + w(m + "conv_bias"))
            u = ubc[..., :inner].reshape(b, T, z.ssd_heads, z.ssd_vdim)
            share = z.ssd_heads // z.groups
            bm = ubc[..., inner:inner + gn].reshape(b, T, z.groups, z.state).repeat_interleave(share, 2)
            cm = ubc[..., inner + gn:].reshape(b, T, z.groups, z.state).repeat_interleave(share, 2)
            dt = torch.nn.functional.softplus(dt + w(m + "dt_bias"))
            keep = torch.exp(-w(m + "a_log").exp() * dt)
            y = _scan(cm, bm, dt[..., None] * u, keep[..., None]) + w(m + "skip")[:, None] * u
            y = (y.reshape(b, T, inner) * silu(gate)).view(b, T, z.parts, inner // z.parts)
            right = _rms(y, None, _EPS).reshape(b, T, inner) * w(m + "ssd_norm_weight") * _RIGHT
            y = torch.cat([left, right], -1) @ w(m + "out_proj.weight").T
        else:
            h, dk, dv = (z.lin_heads, z.lin_dim, z.lin_vdim) if i == 1 else (z.gla_heads, z.gla_dim, z.gla_vdim)
            q, k, v, gate = rows[..., :2 * h * (dk + dv)].split([h * dk, h * dk, h * dv, h * dv], -1)
            shape = lambda y, n: y.reshape(b, T, h, n)  # noqa: E731
            if i == 1:
                decay = torch.tensor(_decays(z), device=dev, dtype=torch.float64).view(1, 1, h, 1).expand(b, T, h, 1)
                o = _scan(shape(silu(q), dk), shape(silu(k), dk), shape(silu(v), dv), decay)
                o = _rms(o.reshape(b, T, h * dv), t[m + "out_norm_weight"], _EPS) * torch.sigmoid(gate)
            else:
                logits = rows[..., 2 * h * (dk + dv):] @ w(m + "decay_proj.weight").T + w(m + "decay_bias")
                decay = torch.exp(torch.nn.functional.logsigmoid(logits) / _TAU)
                o = _scan(shape(q, dk) * dk ** -0.5, shape(k, dk), shape(v, dv), shape(decay, dk))
                o = _rms(o, t[m + "out_norm_weight"], _EPS).reshape(b, T, h * dv) * silu(gate)
            y = o @ w(m + "o_proj.weight").T
        x = x + _rms(y, t[p + "norm1_weight"], _EPS)
        if i == 0:
            g, u = (x @ w(p + "mlp.in_proj.weight").T + w(p + "mlp.in_proj.bias")).chunk(2, -1)
            y = (silu(g) * u) @ w(p + "mlp.down_proj.weight").T + w(p + "mlp.down_bias")
        else:
            flat = x.reshape(b * T, z.width)
            score = torch.softmax(flat @ w(p + "mlp.router_weight").T, -1)
            ids = torch.topk(score + w(p + "mlp.correction"), z.top, -1).indices
            y = torch.zeros_like(flat)
            for e in range(z.experts + z.identity):
                r = (ids == e).any(-1).nonzero(as_tuple=True)[0]
                if e >= z.experts:
                    y[r] += flat[r] * score[r, e, None]
                    continue
                g, u = (flat[r] @ w(p + "mlp.gate_up_weight")[e].T).chunk(2, -1)
                g, u = g.clamp(max=_LIMIT), u.clamp(-_LIMIT, _LIMIT)
                y[r] += ((g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ w(p + "mlp.down_weight")[e].T) * score[r, e, None]
            y = y.view(b, T, z.width)
        x = x + _rms(y, t[p + "norm2_weight"], _EPS)
    head = t["embed_tokens.weight"].double()
    final = _rms(x, t["norm_weight"], _EPS)
    return torch.stack([final[i, stop - 1] for entries in _schedule(case, lens) for i, _, stop in entries]) @ head.T


def exact(case: dict, seed: int):
    with torch.no_grad():
        return _exact_llama(case, seed) if "model" in case else _exact_layered(case, seed)
