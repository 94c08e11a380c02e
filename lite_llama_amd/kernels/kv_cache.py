"""update_kv_buffer / update_kv_index -- mirror of lite_llama/kernels/update_kv_buffer.py:54-89
and update_kv_index.py:50-88 over the HIP C-ABI (bit-exact integer / byte moves)."""

from __future__ import annotations

import torch

from .. import _lib as L


@L.without_grad
def update_kv_buffer(KV_Values, Select_Index, KV_Buffer):
    """``KV_Buffer[Select_Index[i], :, :] = KV_Values[i, :, :]``; other rows untouched."""
    L.require_cuda(KV_Values, Select_Index, KV_Buffer)
    assert KV_Values.shape[1] == KV_Buffer.shape[1] and KV_Values.shape[2] == KV_Buffer.shape[2]
    assert KV_Values.dtype == KV_Buffer.dtype and KV_Values.element_size() == 2
    if KV_Values.stride(2) != 1:
        KV_Values = KV_Values.contiguous()
    assert KV_Buffer.stride(2) == 1
    L.check(
        L.lib().ll_update_kv_buffer(
            KV_Values.data_ptr(), Select_Index.data_ptr(), KV_Buffer.data_ptr(),
            Select_Index.shape[0], KV_Values.shape[1], KV_Values.shape[2], KV_Values.stride(0),
            KV_Values.stride(1), KV_Buffer.stride(0), KV_Buffer.stride(1),
            L.index_width(Select_Index), L.stream_ptr(),
        ),
        "update_kv_buffer",
    )
    return


FP8_KV_DTYPES = (torch.uint8, torch.float8_e4m3fn)


@L.without_grad
def update_kv_buffer_fp8(KV_Values, Select_Index, KV_Buffer, num_k_heads: int, k_scale: float = 1.0, v_scale: float = 1.0):
    """``update_kv_buffer`` into an fp8 (OCP e4m3) pool (extension): ``KV_Buffer[Select_Index[i]] = e4m3(KV_Values[i] /
    scale)`` with ``k_scale`` for the first ``num_k_heads`` heads of a row and ``v_scale`` for the rest; values are
    clamped to +-448 and rounded to nearest even.  ``KV_Buffer``: uint8 or float8_e4m3fn ``[rows, heads, hd]``."""
    L.require_cuda(KV_Values, Select_Index, KV_Buffer)
    assert KV_Values.shape[1] == KV_Buffer.shape[1] and KV_Values.shape[2] == KV_Buffer.shape[2]
    assert KV_Buffer.dtype in FP8_KV_DTYPES and KV_Values.dtype in (torch.float16, torch.bfloat16)
    if KV_Values.stride(2) != 1:
        KV_Values = KV_Values.contiguous()
    assert KV_Buffer.stride(2) == 1
    L.check(
        L.lib().ll_update_kv_buffer_fp8(
            KV_Values.data_ptr(), Select_Index.data_ptr(), KV_Buffer.data_ptr(), Select_Index.shape[0], KV_Values.shape[1],
            num_k_heads, KV_Values.shape[2], KV_Values.stride(0), KV_Values.stride(1), KV_Buffer.stride(0),
            KV_Buffer.stride(1), float(k_scale), float(v_scale), L.dtype_code(KV_Values.dtype),
            L.index_width(Select_Index), L.stream_ptr(),
        ),
        "update_kv_buffer_fp8",
    )


@L.without_grad
def update_kv_index(req_to_token_indexs, b_req_idx, b_seq_len, select_index):
    """``table[b_req_idx[i], b_seq_len[i] - 1] = select_index[i]``."""
    L.require_cuda(req_to_token_indexs, b_req_idx, b_seq_len, select_index)
    assert (
        b_seq_len.shape[0] == select_index.shape[0] and b_req_idx.shape[0] == b_seq_len.shape[0]
    ), "b_req_idx, b_seq_len and select_index must have the same length"
    assert req_to_token_indexs.dtype == torch.int32
    L.check(
        L.lib().ll_update_kv_index(
            req_to_token_indexs.data_ptr(), b_req_idx.data_ptr(), b_seq_len.data_ptr(),
            select_index.data_ptr(), b_seq_len.shape[0], req_to_token_indexs.stride(0),
            req_to_token_indexs.stride(1), L.index_width(b_req_idx), L.index_width(b_seq_len),
            L.index_width(select_index), L.stream_ptr(),
        ),
        "update_kv_index",
    )
    return


@L.without_grad
def pack_prompts(input_ids, position_ids, select_index, b_seq_len, total: int, rows):
    """Prompts on a padded grid ``[batch, longest]`` -> the tokens of all prompts one after the other (``total`` = the sum of their
    lengths): ``(ids [1, total], positions [1, total], select_index [total], starts int32 [batch], lengths int64 [batch], rows)``, with
    ``rows`` the packed places of the asked grid rows."""
    L.require_cuda(input_ids, position_ids, select_index, b_seq_len, rows)
    batch, longest = input_ids.shape
    if input_ids.dtype != torch.int64 or position_ids.dtype != torch.int64 or rows.dtype != torch.int64 or rows.dim() != 1 \
            or position_ids.shape != input_ids.shape or select_index.numel() != batch * longest or not select_index.is_contiguous() \
            or b_seq_len.numel() != batch or not b_seq_len.is_contiguous() or not rows.is_contiguous():
        raise ValueError("pack_prompts: int64 ids and positions [batch, longest], one scatter target per grid row, one length per prompt")
    dev = input_ids.device
    out = torch.empty(2 * total + batch + rows.numel(), dtype=torch.int64, device=dev)
    ids, positions, lens, packed_rows = out.split([total, total, batch, rows.numel()])
    select = torch.empty(total, dtype=select_index.dtype, device=dev)
    starts = torch.empty(batch, dtype=torch.int32, device=dev)
    L.check(
        L.lib().ll_pack_prompts(
            input_ids.data_ptr(), input_ids.stride(0), input_ids.stride(1), position_ids.data_ptr(), position_ids.stride(0),
            position_ids.stride(1), select_index.data_ptr(), L.index_width(select_index), b_seq_len.data_ptr(), L.index_width(b_seq_len),
            batch, longest, total, rows.data_ptr(), rows.numel(), ids.data_ptr(), positions.data_ptr(), select.data_ptr(),
            starts.data_ptr(), lens.data_ptr(), packed_rows.data_ptr(), L.stream_ptr(),
        ),
        "pack_prompts",
    )
    return ids.view(1, total), positions.view(1, total), select, starts, lens, packed_rows
