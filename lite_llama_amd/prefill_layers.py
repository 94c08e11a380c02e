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
    """A projection's output left as the split-K planes of consecutive parts of its rows, in ``view`` (fp32)."""

    __slots__ = ("view", "planes", "rows", "part", "shape", "dtype")

    def __init__(self, view, planes, rows, part, shape, dtype):
        self.view, self.planes, self.rows, self.part, self.shape, self.dtype = view, planes, rows, part, tuple(shape), dtype

    @property
    def parts(self):
        """``[planes, rows, width]`` of every part."""
        out, width = [], self.shape[-1]
        for i in range(-(-self.rows // self.part)):
            rows, at = min(self.part, self.rows - i * self.part), i * _MAX_PLANES * self.part * width
            out.append(self.view[at:at + self.planes * rows * width].view(self.planes, rows, width))
        return out

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
        # what every layer of the pass is handed alike (the pass holds the tensors)
        from .linear import ColumnParallelLinear, RowParallelLinear
        from .model import Attention, DecoderLayer, FusedMLP, PagedAttention
        from .quantization.methods import UnquantizedLinearMethod

        self.kinds = (ColumnParallelLinear, RowParallelLinear, Attention, DecoderLayer, FusedMLP, PagedAttention, UnquantizedLinearMethod)
        select, starts, lens = info.cur_select_index, info.b_start_loc, info.b_seq_len
        self._held, self._longest = (select, starts, lens), info.max_actual_seq_len
        self.tables = (cos.data_ptr(), sin.data_ptr(), cos.stride(0), cos.stride(1), sin.stride(0), sin.stride(1))
        self.metadata = (select.data_ptr(), L.index_width(select), starts.data_ptr(), L.index_width(starts), lens.data_ptr(), L.index_width(lens),
                         lens.shape[0], int(info.max_actual_seq_len))
        self.codes = (L.dtype_code(self.dtype), L.dtype_code(cos.dtype))
        self.run, self.stream = L.lib().ll_prefill_layer16, L.stream_ptr()

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
        # (the tables of modules and parameters straight: a module's attribute lookup costs 0.3 us, and the pass looks at sixteen a layer)
        ColumnParallelLinear, RowParallelLinear, Attention, DecoderLayer, FusedMLP, PagedAttention, Plain = self.kinds
        if not _plain(layer, DecoderLayer):
            return None
        mods, params = layer._modules, layer._parameters
        attn, mlp = mods.get("self_attn"), mods.get("mlp")
        if not _plain(attn, Attention) or not _plain(mlp, FusedMLP) or attn.use_qk_norm:
            return None
        mods = attn._modules
        o, down, paged = mods.get("o_proj"), mlp._modules.get("down_proj"), mods.get("attn")
        if not _plain(o, RowParallelLinear) or not _plain(down, RowParallelLinear) or not _plain(paged, PagedAttention):
            return None
        # (``bias=None`` is an ordinary attribute, a bias set later is not)
        if type(o.quant_method) is not Plain or type(down.quant_method) is not Plain or o.bias is not None or down.bias is not None:
            return None
        qkv, gate_up = attn._qkv, mlp._gate_up
        if not qkv.refresh() or not gate_up.refresh():
            return None
        qkv, gate_up = qkv._holder, gate_up._holder
        if (qkv.interleaved or not gate_up.interleaved or type(qkv.quant_method) is not Plain or type(gate_up.quant_method) is not Plain
                or gate_up.bias is not None):
            return None
        heads, kv_heads, dim, width, dt, device = attn.num_heads, attn.num_kv_heads, attn.head_dim, self.width, self.dtype, self.device
        q_size, inter = heads * dim, down.input_size
        row = q_size + 2 * kv_heads * dim
        pool, info = self.info.kv_buffer[index], self.info
        if (info.cur_select_index is not self._held[0] or info.b_start_loc is not self._held[1] or info.b_seq_len is not self._held[2]
                or info.max_actual_seq_len != self._longest):   # (something between the layers gave the pass other metadata)
            return None
        norm1, norm2 = params.get("input_layernorm_weight"), params.get("post_attention_layernorm_weight")
        w_qkv, w_o, w_gate_up, w_down, bias = qkv.weight, o._parameters.get("weight"), gate_up.weight, down._parameters.get("weight"), qkv.bias
        if norm1 is None or norm2 is None or w_o is None or w_down is None:
            return None
        for w, shape in ((w_qkv, (row, width)), (w_o, (width, q_size)), (w_gate_up, (2 * inter, width)), (w_down, (width, inter))):
            if w.dtype != dt or w.device != device or w.shape != shape or not w.is_contiguous():
                return None
        if bias is not None and (bias.dtype != dt or bias.device != device or bias.numel() != row or not bias.is_contiguous()):
            return None
        for w in (norm1, norm2):
            if w.dtype != dt or w.device != device or w.numel() != width or not w.is_contiguous():
                return None
        if (pool.dtype != dt or pool.device != device or pool.dim() != 3 or pool.shape[1] != 2 * kv_heads or pool.shape[2] != dim or pool.stride(2) != 1
                or self.cos.shape[2] < dim // 2 or info.cur_select_index.numel() < self.tokens):
            return None
        _, buf, (x, qkv_rows, attn_rows, act_rows), planes, plane_view = self._scratch(row, q_size, inter)
        if residual is None:
            if not torch.is_tensor(hidden):
                return None
            residual, planes_in = hidden, 0
        elif type(hidden) is RowParts and hidden.view is plane_view:
            planes_in = hidden.planes
        else:
            return None
        left = self.run(
            residual.data_ptr(), x, planes_in, planes, qkv_rows, attn_rows, act_rows, norm1.data_ptr(), norm2.data_ptr(), float(layer.eps),
            w_qkv.data_ptr(), 0 if bias is None else bias.data_ptr(), w_o.data_ptr(), w_gate_up.data_ptr(), w_down.data_ptr(), *self.tables,
            pool.data_ptr(), pool.stride(0), pool.stride(1), *self.metadata, self.tokens, self.seq, width, heads, kv_heads, dim, inter,
            float(paged.scale * _LOG2E), *self.codes, _MAX_PLANES, self.stream)
        if left == 0:
            return None
        if left < 0:
            L.check(left, "prefill_layer16")
        return RowParts(plane_view, left, self.tokens, self.part, (self.batch, self.seq, width), dt), residual

    def done(self, hidden):
        """What the layers left, as the model's other code takes it."""
        if type(hidden) is not RowParts:
            return hidden
        return PartialSums(hidden.parts[0], hidden.shape, hidden.dtype) if hidden.rows <= hidden.part else hidden.materialise()
