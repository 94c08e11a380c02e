"""Ragged attention, 16-bit forms (ragged_attn_mfma.hip), against softmax attention in 64 bits: contexts, windows and kept first keys at the edges of
tiles (32 keys), of partitions (256) and of a workgroup's queries (64), heads per group on either side of 4, 8 and 16, widths that are no multiple
of 32 (the cache around a head holds infinities, which must not be met), a latent cache."""

import types

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def reference(q, k, v, scale, firsts, runs, table, window, keep, sink):
    out, at, rep = [], 0, q.shape[1] // k.shape[1]
    for i, (first, run) in enumerate(zip(firsts, runs)):
        rows = table[i, :first + run].long()
        kk, vv = (x[rows].double().repeat_interleave(rep, 1) for x in (k, v))
        s = torch.matmul(q[at:at + run].double().transpose(0, 1), kk.permute(1, 2, 0).contiguous()) * scale
        pos, key = first + torch.arange(run, device=DEV)[:, None], torch.arange(first + run, device=DEV)[None]
        seen = (key <= pos) & ((key > pos - window) | (key < keep) if window else key >= 0)
        s = s.masked_fill(~seen, float("-inf"))
        if sink is not None:
            s = torch.cat([s, sink.double()[:, None, None].expand(-1, run, 1)], -1)
        p = torch.softmax(s, -1)[..., :first + run]
        out.append(torch.matmul(p, vv.transpose(0, 1).contiguous()).transpose(0, 1).reshape(run, -1))
        at += run
    return torch.cat(out)


DECODED = [(n, 1) for n in (0, 30, 31, 32, 63, 254, 255, 256, 257, 287, 511, 512, 700)]
PORTIONS = [(0, 1), (0, 65), (31, 64), (32, 33), (255, 16), (300, 130), (513, 1)]


@pytest.mark.parametrize("heads,kv_heads,dk,dv,dtype,window,keep,sink", [
    (16, 4, 128, 128, torch.bfloat16, 0, 0, False),
    (5, 1, 128, 96, torch.float16, 256, 0, True),
    (18, 2, 64, 64, torch.bfloat16, 100, 33, True),      # nine heads a group, kept keys and window in one partition
    (20, 1, 40, 24, torch.float16, 33, 70, False),       # two column tiles
    (8, 8, 72, 256, torch.bfloat16, 300, 260, True),     # kept keys over a partition's end
    (6, 2, 256, 200, torch.float16, 0, 0, False),
    (12, 1, 120, 0, torch.bfloat16, 64, 8, False),       # dv 0: a latent cache, values are the first 96 columns of the keys
])
@pytest.mark.parametrize("runs", [DECODED, PORTIONS], ids=["decoded", "portions"])
def test_tiles_and_widths(heads, kv_heads, dk, dv, dtype, window, keep, sink, runs):
    from lite_llama_amd.kernels.attention import ragged_attention

    g = torch.Generator(device=DEV).manual_seed(heads + dk)
    firsts, counts = [f for f, _ in runs], [c for _, c in runs]
    ctx = [f + c for f, c in runs]
    total = sum(ctx)
    pad = 8
    if dv:
        rows = torch.full((total, kv_heads * (dk + dv) + pad), float("inf"), device=DEV, dtype=dtype)   # (pad: what a read past a row would meet)
        rows[:, :-pad] = torch.randn(total, kv_heads * (dk + dv), generator=g, device=DEV).to(dtype)
        k = rows[:, :kv_heads * dk].unflatten(1, (kv_heads, dk))
        v = rows[:, kv_heads * dk:-pad].unflatten(1, (kv_heads, dv))
    else:
        rows = torch.randn(total, dk, generator=g, device=DEV).to(dtype)
        k, v = rows.unflatten(1, (1, dk)), rows[:, :96].unflatten(1, (1, 96))
    table = torch.full((len(runs), max(ctx) + 3), total - 1, dtype=torch.int32, device=DEV)
    for i, r in enumerate(torch.randperm(total, generator=g, device=DEV).to(torch.int32).split(ctx)):
        table[i, :ctx[i]] = r
    n = sum(counts)
    q = torch.randn(n, heads, dk, generator=g, device=DEV).to(dtype)
    sk = torch.randn(heads, generator=g, device=DEV).to(dtype) if sink else None
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)  # noqa: E731
    starts = [0]
    for c in counts:
        starts.append(starts[-1] + c)
    step = types.SimpleNamespace(num_tokens=n, num_seqs=len(runs), longest_run=max(counts), longest_context=max(ctx), seq_req=i32(list(range(len(runs)))),
                                 seq_start=i32(starts), seq_first_pos=i32(firsts))
    scale = 2.0 * dk ** -0.5
    got = ragged_attention(q, k, v, scale, step, table, sk, window, keep)
    want = reference(q, k, v, scale, firsts, counts, table, window, keep, sk)
    # the result is rounded to the storage type: half a unit on values up to about 4; the weights carry 16 bits and more
    assert (got.double() - want).abs().max().item() < 2.0 ** (-9 if dtype == torch.float16 else -6)
    assert torch.equal(ragged_attention(q, k, v, scale, step, table, sk, window, keep), got)
