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


# a case on either side of every line of fd_plan: pairs of 32 / 64 / 127, 16 and 127 partitions, eight heads, heads of 256; short rows and a
# long one, and rows of no tokens beside them
@pytest.mark.parametrize("b,hkv,rep,d,longest", [(32, 1, 4, 128, 1100), (33, 1, 4, 128, 2049), (16, 4, 1, 64, 2048), (13, 5, 8, 128, 2200),
                                                 (13, 5, 9, 128, 2200), (127, 1, 4, 128, 5000), (2, 1, 16, 128, 16257), (65, 1, 2, 64, 16384),
                                                 (3, 2, 4, 256, 3000)])
def test_short_rows_beside_a_long_one(b, hkv, rep, d, longest):
    from lite_llama_amd.kernels import flash_decoding

    g = torch.Generator(device=DEV).manual_seed(b + d)
    lens = [longest if i == b // 2 else (37 * i) % 700 + 1 for i in range(b)]
    pool = torch.randn(sum(lens), 2 * hkv, d, generator=g, device=DEV).half()
    table = torch.zeros(b, longest, dtype=torch.int32, device=DEV)
    for i, rows in enumerate(torch.randperm(sum(lens), generator=g, device=DEV).to(torch.int32).split(lens)):
        table[i, :lens[i]] = rows
    q = torch.randn(b, hkv * rep, d, generator=g, device=DEV).half()
    seq, req = torch.tensor(lens, dtype=torch.int32, device=DEV), torch.arange(b, dtype=torch.int32, device=DEV)
    args = (q, pool[:, :hkv], pool[:, hkv:], 2.0 / math.sqrt(d), table, req)
    got = flash_decoding(*args, seq, longest)
    # probabilities and the result are rounded to the storage type: half a unit each, on values of up to about 4
    assert (got.double() - reference(q, pool[:, :hkv], pool[:, hkv:], 2.0 / math.sqrt(d), table, seq)).abs().max().item() < 4 * 2.0 ** -10
    assert torch.equal(flash_decoding(*args, seq, longest), got)
    empty = seq.clone()
    empty[0] = 0                                                      # 0 / 0, and nothing else changes
    again = flash_decoding(*args, empty, longest)
    assert again[0].isnan().all() and torch.equal(again[1:], got[1:])


def _planes(b, longest, seed):
    """A decode step of ``b`` rows over contexts up to ``longest`` as split-K planes: arguments behind ``parts`` and ``bias``."""
    from lite_llama_amd.kernels.norm_act import PartialSums

    hq, hkv, d = 12, 2, 128
    g = torch.Generator(device=DEV).manual_seed(seed)
    lens = [longest - 37 * i for i in range(b)]
    pool = torch.randn(sum(lens), 2 * hkv, d, generator=g, device=DEV).to(torch.bfloat16)
    table = torch.zeros(b, longest, dtype=torch.int32, device=DEV)
    for i, rows in enumerate(torch.randperm(sum(lens), generator=g, device=DEV).to(torch.int32).split(lens)):
        table[i, :lens[i]] = rows
    seq = torch.tensor(lens, dtype=torch.int64, device=DEV)
    req = torch.arange(b, dtype=torch.int64, device=DEV)
    ang = torch.arange(longest, device=DEV)[:, None] * torch.rand(d // 2, generator=g, device=DEV)[None]
    cos, sin = (torch.cat([f(ang)] * 2, -1).to(torch.bfloat16) for f in (torch.cos, torch.sin))
    row = (hq + 2 * hkv) * d
    planes = torch.randn(5, b, row, generator=g, device=DEV)
    return PartialSums(planes, (b, row), torch.bfloat16), hq, hkv, d, cos, sin, seq - 1, table[req, seq - 1].contiguous(), pool, table, req, seq


@pytest.mark.parametrize("b,longest,served", [(32, 2300, True), (63, 3000, True), (31, 2300, False), (2, 1024, True)])
def test_planes_without_scratch(b, longest, served):
    """The entry point without the merge's scratch serves what ll_flash_decoding_group_waves says, one workgroup per pair, and refuses the rest."""
    from lite_llama_amd import _lib as L
    from lite_llama_amd.kernels.attention import decode_attention_partials

    parts, hq, hkv, d, cos, sin, pos, sel, pool, table, req, seq = _planes(b, longest, b)
    pool_a, pool_b = pool.clone(), pool.clone()
    out = torch.zeros(b, hq, d, dtype=pool.dtype, device=DEV)
    rc = L.lib().ll_decode_attention_partials(
        out.data_ptr(), parts.parts.data_ptr(), 5, 0, cos.data_ptr(), sin.data_ptr(), cos.stride(0), pos.data_ptr(), sel.data_ptr(),
        L.index_width(sel), pool_a.data_ptr(), pool_a[:, hkv:].data_ptr(), table.data_ptr(), req.data_ptr(), seq.data_ptr(), b, hq, hkv, d,
        longest, 0.1, *pool_a.stride()[:2], *pool_a.stride()[:2], out.stride(0), out.stride(1), table.stride(0), L.dtype_code(pool.dtype),
        L.index_width(req), L.index_width(seq), 0, 0, 0.0, 0, 0, L.stream_ptr())
    assert (rc == 0) == served == (L.lib().ll_flash_decoding_group_waves(longest, b * hkv) > 0)
    got = decode_attention_partials(parts, None, hq, hkv, d, cos, sin, pos, sel, pool_b, 0.1, table, req, seq, longest)
    if not served:
        assert got is None and torch.equal(pool_a, pool)
        return
    assert torch.equal(pool_a, pool_b)
    # the same context in other shares: probabilities and the result rounded to the storage type
    assert (out.double() - got.double()).abs().max().item() < 4 * 2.0 ** -7


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


# five to eight partitions: several workgroups of two partitions per pair where all of them find a CU (heads of 128), one workgroup beside that line
@pytest.mark.parametrize("b,hkv,rep,d,longest,bound", [(1, 1, 1, 128, 513, 640), (1, 4, 7, 128, 1000, 1024), (3, 2, 16, 128, 1024, 1024), (16, 4, 8, 128, 700, 768),
                                                       (13, 5, 3, 128, 900, 1024), (2, 2, 15, 128, 640, 640), (9, 2, 7, 64, 1000, 1024)])
def test_middle_contexts(b, hkv, rep, d, longest, bound):
    from lite_llama_amd.kernels import flash_decoding
    from lite_llama_amd.kernels.attention import _fd_counters

    g = torch.Generator(device=DEV).manual_seed(longest)
    lens = [longest if i == b // 2 else (131 * i) % longest + 1 for i in range(b)]
    pool = torch.randn(sum(lens), 2 * hkv, d, generator=g, device=DEV).half()
    table = torch.zeros(b, bound, dtype=torch.int32, device=DEV)
    for i, rows in enumerate(torch.randperm(sum(lens), generator=g, device=DEV).to(torch.int32).split(lens)):
        table[i, :lens[i]] = rows
    q = torch.randn(b, hkv * rep, d, generator=g, device=DEV).half()
    seq, req = torch.tensor(lens, dtype=torch.int32, device=DEV), torch.arange(b, dtype=torch.int32, device=DEV)
    args = (q, pool[:, :hkv], pool[:, hkv:], 2.0 / math.sqrt(d), table, req)
    got = flash_decoding(*args, seq, bound)
    # probabilities and the result are rounded to the storage type: half a unit each, on values of up to about 4
    assert (got.double() - reference(q, pool[:, :hkv], pool[:, hkv:], 2.0 / math.sqrt(d), table, seq)).abs().max().item() < 4 * 2.0 ** -10
    for _ in range(3):
        assert torch.equal(flash_decoding(*args, seq, bound), got)
    empty = seq.clone()
    empty[0] = 0
    again = flash_decoding(*args, empty, bound)
    assert again[0].isnan().all() and torch.equal(again[1:], got[1:])
    assert all(int(c.abs().sum()) == 0 for c in _fd_counters.values())


@pytest.mark.parametrize("b,longest", [(1, 513), (7, 900), (27, 1024)])
def test_planes_at_middle_contexts(b, longest):
    """q | k | v as split-K planes == the finished projection where several workgroups share a row, bit for bit, output and written cache rows."""
    from lite_llama_amd.kernels.attention import decode_attention, decode_attention_partials

    parts, hq, hkv, d, cos, sin, pos, sel, pool, table, req, seq = _planes(b, longest, b)
    pool_a, pool_b = pool.clone(), pool.clone()
    got = decode_attention_partials(parts, None, hq, hkv, d, cos, sin, pos, sel, pool_a, 0.1, table, req, seq, longest)
    sums = parts.parts[0].clone()
    for p in parts.parts[1:]:
        sums = sums + p                                               # (planes are added in order, in 32 bits)
    rows = sums.to(torch.bfloat16)
    q, kv = rows[:, :hq * d].view(b, hq, d), rows[:, hq * d:].view(b, 2 * hkv, d)
    want = decode_attention(q.contiguous(), kv.contiguous(), cos, sin, pos, sel, pool_b, 0.1, table, req, seq, longest)
    assert torch.equal(pool_a, pool_b) and torch.equal(got.reshape(-1), want.reshape(-1))


# every form of the launch; heads of one and two column tiles, and of an odd last round of the merge; five, six and eight partitions; rows at the edges of a
# partition, of what is not spread (384) and of one workgroup's share
@pytest.mark.parametrize("kind,hkv,rep,bound", [("rows", 2, 7, 1024), ("rows", 1, 20, 1024), ("rows", 4, 1, 640), ("rows bf16", 2, 16, 768), ("fp8", 2, 4, 1024),
                                                ("fused", 2, 6, 1024), ("fused norm", 2, 4, 900), ("planes", 2, 7, 1024), ("planes norm", 4, 16, 640),
                                                ("planes int32", 2, 4, 1024)])
def test_the_bits_of_one_workgroup(kind, hkv, rep, bound):
    """Rows whose pairs leave compute units idle are spread over several workgroups; beside so many others that the launch keeps one workgroup to a pair,
    they are not: the same bits, in the result and in the written cache rows."""
    from lite_llama_amd.kernels import flash_decoding
    from lite_llama_amd.kernels.attention import decode_attention, decode_attention_partials, flash_decoding_fp8kv
    from lite_llama_amd.kernels.norm_act import PartialSums, ScaledInt32Partials

    d, hq = 128, hkv * rep
    dt = torch.float16 if kind in ("rows", "fp8", "planes int32") else torch.bfloat16
    g = torch.Generator(device=DEV).manual_seed(hq + bound)
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV)  # noqa: E731
    splits, groups = -(-bound // 256), -(-rep // 16)
    lens = [n for n in (bound, 1, 128, 129, 383, 384, 385, 512, 513, 640, 641, 700, 768, 897) if n <= bound]
    few = len(lens)
    assert few * hkv * groups * splits <= 256
    lens += [(37 * i) % bound + 1 for i in range(256 // (hkv * groups * splits) + 1)]
    rows = len(lens)
    pool = (rand(sum(lens), 2 * hkv, d) * (0.5 if kind == "fp8" else 1.0)).to(torch.float8_e4m3fn if kind == "fp8" else dt)
    pool = pool.view(torch.uint8) if kind == "fp8" else pool
    table = torch.zeros(rows, bound, dtype=torch.int32, device=DEV)
    for i, at in enumerate(torch.randperm(sum(lens), generator=g, device=DEV).to(torch.int32).split(lens)):
        table[i, :lens[i]] = at
    seq, req = torch.tensor(lens, dtype=torch.int64, device=DEV), torch.arange(rows, dtype=torch.int64, device=DEV)
    pos, sel = seq - 1, table[req, seq - 1].contiguous()
    ang = torch.arange(bound, device=DEV)[:, None] * torch.rand(d // 2, generator=g, device=DEV)[None]
    cos, sin = (torch.cat([f(ang)] * 2, -1).to(dt) for f in (torch.cos, torch.sin))
    norm = (1 + rand(d).to(dt) * 0.1, 1 + rand(d).to(dt) * 0.1, 1e-6) if kind.endswith("norm") else None
    width = (hq + 2 * hkv) * d
    q, kv, planes = rand(rows, hq, d).to(dt), rand(rows, 2 * hkv, d).to(dt), rand(5, rows, width)
    counts = torch.randint(-3000, 3000, (5, rows, width), generator=g, device=DEV, dtype=torch.int32)
    a_scale, w_scale = rand(rows).abs() * 0.01 + 0.001, rand(width).abs() * 0.01 + 0.001

    def call(n):
        own = pool.clone()
        k, v, tail = own[:, :hkv], own[:, hkv:], (0.1, table[:n], req[:n], seq[:n], bound)
        if kind.startswith("rows"):
            return flash_decoding(q[:n], k, v, *tail), own
        if kind == "fp8":
            return flash_decoding_fp8kv(q[:n], k, v, *tail), own
        at = (cos, sin, pos[:n].contiguous(), sel[:n].contiguous(), own, *tail)
        if kind.startswith("fused"):
            return decode_attention(q[:n], kv[:n], *at, qk_norm=norm), own
        if kind == "planes int32":
            parts = ScaledInt32Partials(counts[:, :n].contiguous(), (n, width), a_scale[:n].contiguous(), w_scale)
        else:
            parts = PartialSums(planes[:, :n].contiguous(), (n, width), dt)
        return decode_attention_partials(parts, None, hq, hkv, d, *at, qk_norm=norm), own

    (alone, pool_a), (all_rows, pool_b) = call(few), call(rows)
    assert torch.isfinite(alone.float()).all() and torch.equal(alone, all_rows[:few])
    written = sel[:few].long()
    assert torch.equal(pool_a[written], pool_b[written])
    if not kind.startswith("rows") and kind != "fp8":
        assert not torch.equal(pool_a[written], pool[written])
