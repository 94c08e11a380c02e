"""The eager prefill of few tokens through an unquantised model, a host call per layer (csrc/prefill_layer.hip).

Such a prefill is bound by the host: eight launches per layer, each behind about 20 us of interpreter.  ``ShortPrefill`` reads a layer's
tensors afresh on every forward pass and issues the layer in one call; whatever differs from the plain case -- quantised or sharded projections,
head norms, an fp8 pool, replaced modules, forward hooks, a shape that one of the launches declines -- makes it hand the layer back, and the
layer's own ``forward`` runs."""

from __future__ import annotations

import os

import torch
from torch.nn.modules import module as _nn

from . import _lib as L
from .distributed.parallel_state import collective_forced, get_tp_world_size, shard_simulated
from .kernels.norm_act import PartialSums

_LOG2E = 1.4426950408889634
_MAX_PLANES = 12
_KNOBS = ("LL_DENSE16_ROWS_OFF", "LL_DENSE_NO_PARTIALS", "LL_DENSE16_OFF", "LL_DENSE16_NARROW_OFF", "LL_NO_LAYER_CALLS")


def _plain(module, kind) -> bool:
    """``module`` is of exactly this class, and calling it runs nothing but its ``forward``."""
    return (type(module) is kind and "forward" not in module.__dict__ and not module._forward_hooks and not module._forward_pre_hooks
            and not module._backward_hooks and not module._backward_pre_hooks)


class RowParts:
    """A projection's output left as :class:`PartialSums` of consecutive parts of its rows."""

    __slots__ = ("parts", "shape", "dtype")

    def __init__(self, parts, shape, dtype):
        self.parts, self.shape, self.dtype = parts, tuple(shape), dtype

    def materialise(self) -> torch.Tensor:
        return torch.cat([p.sum(0) for p in self.parts]).to(self.dtype).view(self.shape)


class ShortPrefill:
    """One forward pass over ``hidden [batch, seq, width]`` (at most 192 tokens, more than one per sequence)."""

    MAX_TOKENS = 192   # in parts of up to 64 rows: what the row-group loop and the split-K engine serve

    @staticmethod
    def of(model, hidden, position_embeddings, info):
        """The pass, or ``None`` where none of its layers would be served."""
        if not hidden.is_cuda or hidden.dim() != 3 or hidden.dtype not in (torch.float16, torch.bfloat16) or not hidden.is_contiguous():
            return None
        batch, seq, width = hidden.shape
        if seq < 2 or batch * seq > ShortPrefill.MAX_TOKENS or model.quant is not None or get_tp_world_size() != 1:
            return None
        if collective_forced() or shard_simulated() or any(os.environ.get(k) for k in _KNOBS) or not L.has("ll_prefill_layer16"):
            return None
        if type(position_embeddings) is not tuple or len(position_embeddings) != 2:
            return None
        cos, sin = position_embeddings
        select, starts, lens = info.cur_select_index, info.b_start_loc, info.b_seq_len
        if not all(torch.is_tensor(t) and t.device == hidden.device for t in (cos, sin, select, starts, lens)):
            return None
        if (cos.dim() != 3 or cos.shape != sin.shape or cos.dtype != sin.dtype or not cos.is_contiguous() or not sin.is_contiguous()
                or cos.dtype not in (torch.float16, torch.bfloat16, torch.float32)
                or any(t.dtype not in (torch.int32, torch.int64) or t.dim() != 1 or not t.is_contiguous() for t in (select, starts, lens))):
            return None
        if _nn._global_forward_hooks or _nn._global_forward_pre_hooks or _nn._global_backward_hooks or _nn._global_backward_pre_hooks:
            return None
        return ShortPrefill(hidden, cos, sin, info)

    def __init__(self, hidden, cos, sin, info):
        self.batch, self.seq, self.width = hidden.shape
        self.tokens, self.dtype, self.device = self.batch * self.seq, hidden.dtype, hidden.device
        self.cos, self.sin, self.info = cos, sin, info
        self.parts = -(-self.tokens // 64)
        self.part = -(-self.tokens // self.parts)
        self._space = None

    def _scratch(self, row, q_size, inter):
        """Rows of 16 bits and the planes behind them, in one allocation for the pass."""
        key = (row, q_size, inter)
        if self._space is None or self._space[0] != key:
            t, sizes, at = self.tokens, [], 0
            for n in (self.width, row, q_size, inter):
                sizes.append(at)
                at += -(-t * n * 2 // 256) * 256
            buf = torch.empty(at + 4 * _MAX_PLANES * self.parts * self.part * self.width, dtype=torch.uint8, device=self.device)
            base = buf.data_ptr()
            self._space = key, buf, [base + o for o in sizes], base + at, buf[at:].view(torch.float32)
        return self._space

    def layer(self, layer, index: int, hidden, residual):
        """``(hidden, residual)`` as ``DecoderLayer.forward`` returns them, or ``None``: not served, nothing has run."""
        from .linear import ColumnParallelLinear, RowParallelLinear
        from .model import Attention, DecoderLayer, FusedMLP, PagedAttention
        from .quantization.methods import UnquantizedLinearMethod

        if not _plain(layer, DecoderLayer):
            return None
        attn, mlp = layer.self_attn, layer.mlp
        if not _plain(attn, Attention) or not _plain(mlp, FusedMLP) or attn.use_qk_norm:
            return None
        o, down, paged = attn.o_proj, mlp.down_proj, attn.attn
        if not _plain(o, RowParallelLinear) or not _plain(down, RowParallelLinear) or not _plain(paged, PagedAttention):
            return None
        if (type(o.quant_method) is not UnquantizedLinearMethod or type(down.quant_method) is not UnquantizedLinearMethod
                or o.bias is not None or down.bias is not None):
            return None
        qkv, gate_up = attn._qkv, mlp._gate_up
        if not qkv.refresh() or not gate_up.refresh():
            return None
        qkv, gate_up = qkv._holder, gate_up._holder
        if (qkv.interleaved or not gate_up.interleaved or type(qkv.quant_method) is not UnquantizedLinearMethod
                or type(gate_up.quant_method) is not UnquantizedLinearMethod or gate_up.bias is not None):
            return None
        heads, kv_heads, dim, width, dt = attn.num_heads, attn.num_kv_heads, attn.head_dim, self.width, self.dtype
        q_size, inter = heads * dim, down.input_size
        row = q_size + 2 * kv_heads * dim
        pool, info = self.info.kv_buffer[index], self.info
        norm1, norm2 = layer.input_layernorm_weight, layer.post_attention_layernorm_weight
        weights = ((qkv.weight, row, width), (o.weight, width, q_size), (gate_up.weight, 2 * inter, width), (down.weight, width, inter))
        for w, n, k in weights:
            if w.dtype != dt or w.device != self.device or tuple(w.shape) != (n, k) or not w.is_contiguous():
                return None
        bias = qkv.bias
        if bias is not None and (bias.dtype != dt or bias.device != self.device or bias.numel() != row or not bias.is_contiguous()):
            return None
        for w in (norm1, norm2):
            if w.dtype != dt or w.device != self.device or w.numel() != width or not w.is_contiguous():
                return None
        if (pool.dtype != dt or pool.device != self.device or pool.dim() != 3 or pool.shape[1] != 2 * kv_heads or pool.shape[2] != dim or pool.stride(2) != 1
                or self.cos.shape[2] < dim // 2 or info.cur_select_index.numel() < self.tokens):
            return None
        _, buf, (x, qkv_rows, attn_rows, act_rows), planes, plane_view = self._scratch(row, q_size, inter)
        if residual is None:
            if not torch.is_tensor(hidden):
                return None
            residual, planes_in = hidden, 0
        elif type(hidden) is RowParts and hidden.parts[0].data_ptr() == planes:
            planes_in = hidden.parts[0].shape[0]
        else:
            return None
        cos, sin = self.cos, self.sin
        left = L.lib().ll_prefill_layer16(
            residual.data_ptr(), x, planes_in, planes, qkv_rows, attn_rows, act_rows, norm1.data_ptr(), norm2.data_ptr(), float(layer.eps),
            qkv.weight.data_ptr(), L.ptr(bias), o.weight.data_ptr(), gate_up.weight.data_ptr(), down.weight.data_ptr(), cos.data_ptr(),
            sin.data_ptr(), cos.stride(0), cos.stride(1), sin.stride(0), sin.stride(1), pool.data_ptr(), pool.stride(0), pool.stride(1),
            info.cur_select_index.data_ptr(), L.index_width(info.cur_select_index), info.b_start_loc.data_ptr(),
            L.index_width(info.b_start_loc), info.b_seq_len.data_ptr(), L.index_width(info.b_seq_len), info.b_seq_len.shape[0],
            int(info.max_actual_seq_len), self.tokens, self.seq, width, heads, kv_heads, dim, inter, float(paged.scale * _LOG2E),
            L.dtype_code(dt), L.dtype_code(cos.dtype), _MAX_PLANES, L.stream_ptr())
        if left == 0:
            return None
        if left < 0:
            L.check(left, "prefill_layer16")
        sums, each = [], _MAX_PLANES * self.part * width
        for i in range(self.parts):
            rows = min(self.part, self.tokens - i * self.part)
            sums.append(plane_view[i * each:i * each + left * rows * width].view(left, rows, width))
        return RowParts(sums, (self.batch, self.seq, width), dt), residual

    def done(self, hidden):
        """What the layers left, as the model's other code takes it."""
        if type(hidden) is not RowParts:
            return hidden
        return PartialSums(hidden.parts[0], hidden.shape, hidden.dtype) if len(hidden.parts) == 1 else hidden.materialise()
