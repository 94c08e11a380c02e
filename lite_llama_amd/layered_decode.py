"""A step of decoded tokens through a layer whose norms sit on its sublayers' results, as one native call (csrc/layered_decode.hip): the same launches
in the same order as the modules make one by one, without the interpreter between them.  What is not exactly that -- another mixer, a quantised or
replaced projection, a hook, a tensor that something follows, an operand of another shape -- is refused before anything is launched, and the
modules run: their checks and their errors are theirs."""

from __future__ import annotations

from array import array

import torch
import torch.nn.modules.module as _nn
from torch.autograd import forward_ad

from . import _lib as L
from .kernels.norm_act import FirstRows, GatedUpdate
from .kernels.quantization import _dispatch_modes, _tracing_state, _transform_level
from .linear import ReplicatedLinear
from .prefill_layers import _plain
from .quantization.methods import UnquantizedLinearMethod

_SCORINGS = {"sigmoid": 0, "softmax_chosen": 1, "softmax_all": 2, "sigmoid_plain": 3, "softmax_groups": 4}
_CODES = {torch.float16: L.LL_F16, torch.bfloat16: L.LL_BF16}


class _NotServed(Exception):
    pass


def _need(holds) -> None:
    if not holds:
        raise _NotServed


# (here: the index of the step's device.  The kernels are handed addresses, whatever these point at, so every operand is asked where it is.)
def _vector(module, name: str, here: int, dt, *shape: int) -> int:
    """The address of a parameter that is stored plainly and has this shape."""
    p = module._parameters.get(name)
    _need(type(p) is torch.nn.Parameter and p.dtype == dt and tuple(p.shape) == shape and p.is_contiguous() and p.get_device() == here)
    return p.data_ptr()


def _projection(lin, here: int, dt, out: int, inp: int, biased: bool = False) -> tuple:
    _need(_plain(lin, ReplicatedLinear) and type(lin.quant_method) is UnquantizedLinearMethod and (lin._parameters.get("bias") is not None) == biased)
    return _vector(lin, "weight", here, dt, out, inp), (_vector(lin, "bias", here, dt, out) if biased else 0), out, inp


def _rows(t, here: int, dt, *shape: int) -> int:
    _need(type(t) is torch.Tensor and t.dtype == dt and tuple(t.shape) == shape and t.is_contiguous() and t.get_device() == here)
    return t.data_ptr()


_NONE = (0, 0, 0, 0)


def _pending(pending, here, dt, n: int, width: int) -> list:
    if type(pending) is FirstRows:
        return [_rows(pending.rows, here, dt, n, width), 0, 0, 0, 0, 0, 0]
    _need(type(pending) is GatedUpdate and pending.gate is None and pending.y.dim() == 3)
    u, parts = pending, pending.y.shape[1]
    w = u.post_weight
    _need(w.dtype == dt and w.numel() == width and w.is_contiguous() and w.get_device() == here)
    shared = scale = bias = 0
    if u.shared is not None:
        shared = _rows(u.shared, here, dt, n, width)
        _need(u.shared_scale.dtype == torch.float32 and u.shared_scale.numel() == n and u.shared_scale.is_contiguous()
              and u.shared_scale.get_device() == here)
        scale = u.shared_scale.data_ptr()
    if u.bias is not None:
        _need(u.bias.dtype == dt and u.bias.numel() == width and u.bias.is_contiguous() and u.bias.get_device() == here)
        bias = u.bias.data_ptr()
    return [0, _rows(u.y, here, dt, n, parts, width), parts, shared, scale, bias, w.data_ptr()]


def _state(cache, run: int, here: int, heads: int, dk: int, dv: int) -> int:
    t = cache.recurrent[run]
    _need(t is not None and t.dtype == torch.float32 and t.is_contiguous() and tuple(t.shape[1:]) == (heads, dk, dv)
          and t.get_device() == here)
    return t.data_ptr()


_NO_ATTENTION = [0] * 19


def _attention_ssd(m, here, dt, width, step, cache, run, device):
    s, r = m.spec, m.spec.ssd
    gn, channels = r.groups * r.state, r.conv_channels
    _need(channels == r.inner + 2 * gn and r.inner == r.heads * r.vdim and r.conv_taps > 1)
    k_cache, v_cache = cache.kv_buffer[run]
    conv = cache.conv[run]
    for t, shape in ((k_cache, (s.kv_heads, s.dim)), (v_cache, (s.kv_heads, s.vdim)), (conv, (conv.shape[1], r.conv_taps - 1, channels))):
        _need(t.dtype == dt and tuple(t.shape[1:]) == shape and t.is_contiguous() and t.get_device() == here)
    _need(conv.shape[0] == 2)
    freq = m.frequencies(device) if m.pairs else None
    mixer = [0, *_projection(m.in_proj, here, dt, m.dt_off + r.heads, width), *_NONE,
             *_projection(m.out_proj, here, dt, width, m.heads_width + r.inner),
             r.heads, r.groups, r.state, r.vdim, _state(cache, run, here, r.heads, r.state, r.vdim), 0, 0,
             _vector(m, "ssd_norm_weight", here, dt, r.inner), r.inner, r.norm_groups,
             s.heads, s.kv_heads, s.dim, s.vdim, s.window, m.pairs, _vector(m, "q_norm_weight", here, dt, s.heads * s.dim),
             _vector(m, "k_norm_weight", here, dt, s.kv_heads * s.dim), L.ptr(freq), k_cache.data_ptr(), v_cache.data_ptr(),
             _vector(m, "conv_weight", here, dt, channels, r.conv_taps), _vector(m, "conv_bias", here, dt, channels), channels, r.conv_taps,
             conv.data_ptr(), conv[0].numel(), _vector(m, "dt_bias", here, dt, r.heads), _vector(m, "a_log", here, dt, r.heads),
             _vector(m, "skip", here, dt, r.heads)]
    return mixer, (s.branch_scales[0], s.branch_scales[1], s.scale, 1.0, 1.0)


def _fixed_decay(m, here, dt, width, step, cache, run, device):
    s, qk, v = m.spec, m.qk, m.v
    mixer = [1, *_projection(m.in_proj, here, dt, 2 * qk + 2 * v, width), *_NONE, *_projection(m.o_proj, here, dt, width, v),
             s.heads, s.heads, s.dim, s.vdim, _state(cache, run, here, s.heads, s.dim, s.vdim), _rows(m.decays(device), here, torch.float32, s.heads), 0,
             _vector(m, "out_norm_weight", here, dt, v), v, 1, *_NO_ATTENTION, 0]
    return mixer, (1.0, 1.0, 1.0, 1.0, 1.0)


def _entry_decay(m, here, dt, width, step, cache, run, device):
    s, qk, v, rank = m.spec, m.qk, m.v, m.spec.decay_rank
    mixer = [2, *_projection(m.in_proj, here, dt, 2 * qk + 2 * v + rank, width), *_projection(m.decay_proj, here, dt, qk, rank),
             *_projection(m.o_proj, here, dt, width, v), s.heads, s.heads, s.dim, s.vdim, _state(cache, run, here, s.heads, s.dim, s.vdim), 0,
             _vector(m, "decay_bias", here, dt, qk), _vector(m, "out_norm_weight", here, dt, s.vdim), s.vdim, s.heads, *_NO_ATTENTION, 0]
    return mixer, (1.0, 1.0, 1.0, s.dim ** -0.5, 1.0 / float(s.tau))


def _dense(m, here, dt, width):
    ff = m.ff
    return [1, *_projection(m.in_proj, here, dt, 2 * ff, width, biased=True), *_projection(m.down_proj, here, dt, width, ff), ff, *[0] * 10], 0.0


def _routed(m, here, dt, width):
    s = m.spec
    outputs = s.experts + s.identity
    _need(s.scoring == "softmax_all")
    return [2, *_NONE, *_NONE, s.ff, _vector(m, "router_weight", here, dt, outputs, width), _vector(m, "correction", here, dt, outputs),
            outputs, s.identity, s.top, _SCORINGS[s.scoring], s.experts, _vector(m, "gate_up_weight", here, dt, s.experts, 2 * s.ff, width),
            _vector(m, "down_weight", here, dt, s.experts, width, s.ff), int(s.limit is not None)], 0.0 if s.limit is None else float(s.limit)


def _decode(layer, x, pending, step, cache, run, token_table, mixers, feed_forwards):
    n, width = x.shape
    mixer, mlp = layer.mixer, layer.mlp
    take, give = mixers.get(type(mixer)), feed_forwards.get(type(mlp)) if mlp is not None else None
    _need(take is not None and (mlp is None or give is not None) and n == step.num_tokens == step.num_seqs and 1 <= n <= 64)
    norm = layer._parameters.get("norm1_weight")
    _need(norm is not None and norm.dtype in _CODES and not torch.is_grad_enabled() and L.has("ll_layered_decode"))
    _need(not (_nn._global_forward_hooks or _nn._global_forward_pre_hooks) and _plain(mixer, type(mixer)) and (mlp is None or _plain(mlp, type(mlp))))
    _need(forward_ad._current_level < 0 and _transform_level() is None and _dispatch_modes() == 0 and not torch.is_autocast_enabled()
          and _tracing_state() is None)
    _need(mixer.eps == layer.eps)   # (one number for all norms of the layer)
    dt, device, here = norm.dtype, x.device, x.get_device()
    _need(here >= 0 and token_table.dtype == torch.int32 and token_table.stride(1) == 1 and token_table.get_device() == here)
    at = [t.data_ptr() for t in (step.tok_seq, step.tok_pos, step.select, step.seq_start, step.seq_first_pos, step.seq_slot, step.seq_parity)]
    norm1 = _vector(layer, "norm1_weight", here, dt, width)
    middle, scales = take(mixer, here, dt, width, step, cache, run, device)
    if mlp is None:
        tail, limit = [0, norm1, *_NONE, *_NONE, *[0] * 11], 0.0
    else:
        tail, limit = give(mlp, here, dt, width)
        tail.insert(1, norm1)
    args = array("q", [_CODES[dt], n, step.num_seqs, width, step.longest_context, *at, token_table.data_ptr(), token_table.stride(0),
                       _rows(x, here, torch.float32, n, width), *_pending(pending, here, dt, n, width), *middle, *tail, 0, 0, 0])
    floats = array("d", [layer.eps, *scales, limit])
    lib, a, f = L.lib(), args.buffer_info(), floats.buffer_info()
    size = lib.ll_layered_decode_bytes(a[0], a[1], f[0], f[1])
    _need(size > 0)
    scratch = torch.empty(size, dtype=torch.uint8, device=device)
    rows = own = None
    parts = 1
    if mlp is not None:
        rows = torch.empty(n, width, dtype=dt, device=device)
        args[-3] = rows.data_ptr()
        if tail[0] == 2:
            parts = mlp.spec.top
            if mlp.spec.identity:
                own = torch.empty(n, dtype=torch.float32, device=device)
                args[-1] = own.data_ptr()
    result = torch.empty(n, parts, width, dtype=dt, device=device)
    args[-2] = result.data_ptr()
    L.check(lib.ll_layered_decode(a[0], a[1], f[0], f[1], scratch.data_ptr(), size, L.stream_ptr()), "layered_decode")
    if mlp is None:
        return x, GatedUpdate(result, norm)
    if tail[0] == 1:
        return x, GatedUpdate(result, layer.norm2_weight, bias=mlp.down_bias)
    return x, GatedUpdate(result, layer.norm2_weight, shared=rows if own is not None else None, shared_scale=own)


def decode_layer(layer, x, pending, step, cache, run: int, token_table, mixers: dict, feed_forwards: dict):
    """``layer.forward(...)`` as one call, or ``None`` where it is not served.  ``mixers`` / ``feed_forwards``: what reads the operands of which class."""
    if step.longest_run != 1:
        return None
    try:
        return _decode(layer, x, pending, step, cache, run, token_table, mixers, feed_forwards)
    except _NotServed:
        return None
