"""Decode attention over contexts of more than eight 128-token partitions at few (row, KV head) pairs: several workgroups share a
row (flash_decoding.hip::fd_plan), each merges its waves' partials, the last to arrive merges the workgroups'."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def reference(q, kc, vc, scale, table, seq):
    """One query per row against its cached rows, in 64 bits."""
    out = []
    rep = q.shape[1] // kc.shape[1]
    for i, n in enumerate(seq.tolist()):
        rows = table[i, :n].long()
        k = kc[rows].double().repeat_interleave(rep, 1)
        v = vc[rows].double().repeat_interleave(rep, 1)
        p = torch.softmax(torch.einsum("hd,nhd->hn", q[i].double(), k) * scale, -1)
        out.append(torch.einsum("hn,nhd->hd", p, v))
    return torch.stack(out)


# lengths at the edges of a tile (32), a partition (128), a workgroup (1024) and of the even shares of 2 .. 32 workgroups' waves; rows
# that need one workgroup beside rows that need all, and a pair count that is no power of two
CASES = [(1, 1, 1, 128, torch.float16, [1025]),
         (1, 4, 7, 128, torch.float16, [4096]),
         (3, 2, 20, 64, torch.bfloat16, [1, 1024, 3001]),
         (9, 7, 1, 128, torch.float16, [1025, 1024, 1, 33, 129, 2048, 2047, 1500, 700]),
         (21, 3, 6, 128, torch.bfloat16, [1100 + 53 * i for i in range(20)] + [32])]


@pytest.mark.parametrize("b,hkv,rep,d,dtype,lens", CASES)
def test_rows_shared_by_several_workgroups(b, hkv, rep, d, dtype, lens):
    from lite_llama_amd.kernels import flash_decoding
    from lite_llama_amd.kernels.attention import _fd_counters

    g = torch.Generator(device=DEV).manual_seed(b)
    longest = max(lens)
    pool = torch.randn(sum(lens), 2 * hkv, d, generator=g, device=DEV).to(dtype)
    table = torch.zeros(b, longest, dtype=torch.int32, device=DEV)
    perm = torch.randperm(sum(lens), generator=g, device=DEV).to(torch.int32)
    for i, rows in enumerate(perm.split(lens)):
        table[i, :lens[i]] = rows
    q = torch.randn(b, hkv * rep, d, generator=g, device=DEV).to(dtype)
    seq = torch.tensor(lens, dtype=torch.int32, device=DEV)
    req = torch.arange(b, dtype=torch.int32, device=DEV)
    scale = 2.0 / math.sqrt(d)
    args = (q, pool[:, :hkv], pool[:, hkv:], scale, table, req, seq)
    want = reference(q, pool[:, :hkv], pool[:, hkv:], scale, table, seq)
    got = flash_decoding(*args, longest)
    # probabilities and the result are rounded to the storage type: half a unit each, on values of up to about 4
    bar = 4 * 2.0 ** (-10 if dtype == torch.float16 else -7)
    assert (got.double() - want).abs().max().item() < bar
    for _ in range(3):
        assert torch.equal(flash_decoding(*args, longest), got)      # the order of arrival is no part of the result
    # a longer bound, as a captured step's bucket gives it: other shares, the same value
    assert (flash_decoding(*args, 8192).double() - want).abs().max().item() < bar
    assert all(int(c.abs().sum()) == 0 for c in _fd_counters.values())


def test_projection_planes_are_taken_from_64_pairs_on():
    """q | k | v as split-K planes == the finished projection, bit for bit, output and written cache rows; fewer pairs decline."""
    from lite_llama_amd.kernels.attention import decode_attention, decode_attention_partials, decode_attention_partials_supported
    from lite_llama_amd.kernels.norm_act import PartialSums

    hq, hkv, d, b, longest = 12, 2, 128, 32, 2300
    g = torch.Generator(device=DEV).manual_seed(3)
    lens = [longest - 37 * i for i in range(b)]
    lens[5], lens[6] = 1, 1025
    total = sum(lens)
    pool = torch.randn(total, 2 * hkv, d, generator=g, device=DEV).to(torch.bfloat16)
    table = torch.zeros(b, longest, dtype=torch.int32, device=DEV)
    perm = torch.randperm(total, generator=g, device=DEV).to(torch.int32)
    for i, rows in enumerate(perm.split(lens)):
        table[i, :lens[i]] = rows
    seq = torch.tensor(lens, dtype=torch.int64, device=DEV)
    req = torch.arange(b, dtype=torch.int64, device=DEV)
    sel, pos = table[req, seq - 1].contiguous(), seq - 1
    ang = torch.arange(longest, device=DEV)[:, None] * torch.rand(d // 2, generator=g, device=DEV)[None]
    cos, sin = (torch.cat([f(ang)] * 2, -1).to(torch.bfloat16) for f in (torch.cos, torch.sin))
    row = (hq + 2 * hkv) * d
    planes = torch.randn(5, b, row, generator=g, device=DEV)
    bias = torch.randn(row, generator=g, device=DEV).to(torch.bfloat16)
    total_ = planes[0]
    for p in planes[1:]:
        total_ = total_ + p
    x = (total_ + bias.float()).to(torch.bfloat16)
    pool_a, pool_b = pool.clone(), pool.clone()
    want = decode_attention(x[:, :hq * d].view(b, hq, d), x[:, hq * d:].view(b, 2 * hkv, d), cos, sin, pos, sel, pool_a, 0.1, table, req, seq,
                            longest)
    parts = PartialSums(planes, (b, row), torch.bfloat16)
    got = decode_attention_partials(parts, bias, hq, hkv, d, cos, sin, pos, sel, pool_b, 0.1, table, req, seq, longest)
    assert torch.equal(pool_a, pool_b) and torch.equal(got, want)
    assert decode_attention_partials_supported(longest, hq, hkv, d, batch=32)
    assert not decode_attention_partials_supported(longest, hq, hkv, d, batch=31)
