"""Split-K planes of narrow projections (csrc/gemm_split.hip): every tile width, more slices than units, shares of unequal length, rows
that end inside a 32-row block, rows of a wider tensor."""

import pytest
import torch

from lite_llama_amd import _lib as L

DEV = "cuda"
FP8, I8, I8I8, F16, BF16 = 1, 2, 3, 4, 5


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", [FP8, I8, I8I8, F16, BF16])
@pytest.mark.parametrize("m,n,k,cap", [(1, 32, 128, 12), (64, 96, 128, 12), (33, 64, 384, 2), (32, 1120, 1152, 12), (31, 4096, 640, 8),
                                       (64, 5120, 2048, 8), (7, 8192, 256, 3), (45, 896, 4864, 12)])
def test_planes_add_up_to_the_product(fmt, m, n, k, cap):
    g = torch.Generator().manual_seed(n + k + fmt)
    pad = 64   # rows of x and w are column ranges of wider tensors
    if fmt in (F16, BF16):
        dt = torch.float16 if fmt == F16 else torch.bfloat16
        w = torch.randn(n, k + pad, generator=g).to(dt)
        x = torch.randn(m, k + pad, generator=g).to(dt)
        wide, scales, gk = w[:, :k].double(), None, k
    else:
        w = torch.randint(-127, 128, (n, k + pad), generator=g, dtype=torch.int8)
        x = torch.randint(-127, 128, (m, k + pad), generator=g, dtype=torch.int8) if fmt == I8I8 else torch.randn(m, k + pad, generator=g).half()
        gk = 64 if k % 128 else 128
        # (powers of two: a widened weight is exact in fp16, what remains is the sums)
        scales = None if fmt == I8I8 else 2.0 ** torch.randint(-4, 3, ((n + 31) // 32, (k + gk - 1) // gk), generator=g).float()
        wide = w[:, :k].double()
        if fmt == FP8:
            w = torch.randn(n, k + pad, generator=g).to(torch.float8_e4m3fn)
            wide, w = w[:, :k].double(), w.view(torch.uint8)
        if scales is not None:
            wide = wide * scales.double().repeat_interleave(32, 0)[:n].repeat_interleave(gk, 1)[:, :k]
    ref = x[:, :k].double() @ wide.T
    size = x[:, :k].double().abs() @ wide.abs().T
    x, w, scales = x.to(DEV), w.to(DEV), None if scales is None else scales.to(DEV)
    count = L.lib().ll_dense_partials_count(m, n, k, fmt, cap)
    assert 1 <= count <= cap
    guard = 64
    planes = torch.full((count * m * n + guard,), 7777, dtype=torch.int32, device=DEV)
    got = L.lib().ll_dense_partials(planes.data_ptr(), x.data_ptr(), w.data_ptr(), L.ptr(scales), m, n, k, 32, gk, fmt, x.stride(0), w.stride(0),
                                    scales.stride(0) if scales is not None else 0, scales.stride(1) if scales is not None else 0, cap,
                                    L.stream_ptr())
    assert got == count
    assert (planes[count * m * n:] == 7777).all()   # nothing past the last plane
    body = planes[:count * m * n].view(count, m, n)
    if fmt == I8I8:
        assert torch.equal(body.sum(0, dtype=torch.int64).cpu(), ref.long())
        return
    total = body.view(torch.float32).double().sum(0).cpu()
    # fp32 sums of k exact products, in whatever order: k * 2^-24 of the sum of their sizes bounds them from far above
    assert ((total - ref).abs() <= k * 2.0 ** -24 * size + 1e-30).all()


@pytest.mark.parametrize("fmt", [FP8, I8, I8I8, F16, BF16])
@pytest.mark.parametrize("n,k", [(1536, 8960), (4096, 14336), (5120, 2048), (896, 896), (36, 128), (32, 64)])
def test_plane_count_does_not_depend_on_the_rows(fmt, n, k):
    for cap in (1, 3, 12):
        counts = {L.lib().ll_dense_partials_count(m, n, k, fmt, cap) for m in (1, 31, 32, 33, 64)}
        assert len(counts) == 1 and max(counts) <= cap
    assert L.lib().ll_dense_partials_count(65, n, k, fmt, 12) == 0


@pytest.mark.parametrize("fmt", [FP8, I8])
def test_contractions_of_whole_64_columns_leave_planes(fmt):
    for n, k in ((2048, 4160), (1024, 2112), (4096, 1088)):
        assert 1 <= L.lib().ll_dense_partials_count(33, n, k, fmt, 12) <= 12


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", [FP8, I8])
@pytest.mark.parametrize("m,n,k", [(64, 2048, 4160), (7, 2048, 4160), (33, 1024, 2112), (33, 2048, 4096), (64, 5120, 2048), (9, 4096, 2432), (32, 96, 640)])
@pytest.mark.parametrize("group_n", [1, 32, 128])
@pytest.mark.parametrize("group_k", [64, 128, 192, 0])
def test_scales_of_a_block_meet_its_columns_alone(fmt, m, n, k, group_n, group_k):
    """Blocks of half a unit of the contraction, of one, of one and a half and of all of it (0); the last block of 192 columns is a partial one."""
    gk = group_k or k
    g = torch.Generator(device=DEV).manual_seed(n + k + group_n + gk)
    x = torch.randn(m, k, generator=g, device=DEV).half()
    if fmt == FP8:
        w = torch.randn(n, k, generator=g, device=DEV).to(torch.float8_e4m3fn)
        wide, w = w.double(), w.view(torch.uint8)
    else:
        w = torch.randint(-127, 128, (n, k), generator=g, device=DEV, dtype=torch.int8)
        wide = w.double()
    blocks = (-(-n // group_n), -(-k // gk))
    scales = 2.0 ** torch.randint(-6, 5, blocks, generator=g, device=DEV).float()   # (powers of two: a widened weight is exact in fp16)
    wide *= scales.double().repeat_interleave(group_n, 0)[:n].repeat_interleave(gk, 1)[:, :k]
    count = L.lib().ll_dense_partials_count(m, n, k, fmt, 12)
    assert 1 <= count <= 12
    planes = torch.full((count, m, n), float("nan"), device=DEV)
    got = L.lib().ll_dense_partials(planes.data_ptr(), x.data_ptr(), w.data_ptr(), scales.data_ptr(), m, n, k, group_n, gk, fmt, k, k, scales.stride(0),
                                    scales.stride(1), 12, L.stream_ptr())
    assert got == count
    # fp32 sums of k exact products, in whatever order
    bound = k * 2.0 ** -24 * (x.double().abs() @ wide.abs().T) + 1e-30
    assert ((planes.double().sum(0) - x.double() @ wide.T).abs() <= bound).all()


# tiles of one, two, three, four and eight row groups; slices of one unit, of many, a short last one
@pytest.mark.gpu
@pytest.mark.parametrize("fmt,m,n,k,cap", [(f, *s) for f in (F16, BF16) for s in (
    (27, 1536, 8960, 12), (64, 1536, 1536, 12), (27, 2048, 1536, 8), (37, 896, 4864, 12), (37, 896, 896, 12), (33, 1024, 4096, 12), (5, 2048, 2048, 12),
    (7, 256, 2048, 12), (1, 128, 64, 12), (64, 4096, 4096, 12), (32, 4096, 1216, 12))] + [(f, *s) for f in (FP8, I8) for s in (
        (64, 5120, 2048, 8), (7, 5120, 2048, 12), (31, 4096, 14336, 12), (64, 4096, 14336, 12), (9, 1536, 8960, 12), (33, 1024, 12288, 8), (64, 2048, 8192, 8))])
def test_sums_are_formed_in_one_order(fmt, m, n, k, cap):
    """The same planes, bit for bit, where four weight rows less put the call on the kernel of gemm_w8_skinny.hip: as many slices, and every sum in its order."""
    g = torch.Generator(device=DEV).manual_seed(n + k + m)
    scales, gk = None, k
    if fmt in (F16, BF16):
        dt = torch.float16 if fmt == F16 else torch.bfloat16
        w, x = torch.randn(n, k, generator=g, device=DEV).to(dt), torch.randn(m, k, generator=g, device=DEV).to(dt)
    else:
        x, gk = torch.randn(m, k, generator=g, device=DEV).half(), 64
        w = (torch.randn(n, k, generator=g, device=DEV).to(torch.float8_e4m3fn).view(torch.uint8) if fmt == FP8 else
             torch.randint(-127, 128, (n, k), generator=g, device=DEV, dtype=torch.int8))
        scales = 0.5 + torch.rand(-(-n // 32), k // gk, generator=g, device=DEV)
    got = []
    for rows in (n, n - 4):
        count = L.lib().ll_dense_partials_count(m, rows, k, fmt, cap)
        planes = torch.full((count, m, rows), float("nan"), device=DEV)
        assert L.lib().ll_dense_partials(planes.data_ptr(), x.data_ptr(), w.data_ptr(), L.ptr(scales), m, rows, k, 32, gk, fmt, k, k,
                                         0 if scales is None else scales.stride(0), 0 if scales is None else 1, cap, L.stream_ptr()) == count
        got.append(planes[:, :, :n - 4])
    assert torch.equal(*got)
