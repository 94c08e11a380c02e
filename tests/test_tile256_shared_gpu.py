"""Products of many rows whose tiles behind the last full round are cut along the contraction (csrc/gemm_tile256.hip): against 64-bit products of
the dequantised operands, and against the same call without scratch memory.  Last slices shorter than the others, slices that begin inside a
scale block, one tile, tiles whose rows and columns end early, a sliver behind a full round."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def near(got, want):
    """fp32 sums of fp16 products of unit size, rounded once to fp16: half a unit of the result plus the sums' own rounding."""
    bar = 2.0 ** -11 * want.abs() + 2.0 ** -13 * want.abs().amax()
    assert ((got.double() - want).abs() <= bar).all(), ((got.double() - want).abs() - bar).max()


def shared(m, n, k, wf):
    from lite_llama_amd import _lib as L
    return L.lib().ll_tile256_split_bytes(m, n, k, wf) > 0


@pytest.mark.parametrize("m,n,k", [(65, 2560, 1536), (300, 3584, 3584), (500, 2560, 1920), (2300, 8192, 1920)])
def test_int4(m, n, k):
    import lite_llama_amd.kernels.quantization as Q

    assert shared(m, n, k, 0)
    g = gen(m)
    q = torch.randint(0, 16, (n, k // 8, 8), generator=g, device=DEV, dtype=torch.int32)
    words = sum(q[..., j] << (4 * j) for j in range(8)).to(torch.int32)
    scale = torch.rand(n, k // 128, generator=g, device=DEV) * 0.01 + 0.01
    zero = torch.randint(0, 16, (n, k // 128), generator=g, device=DEV).float()
    x = torch.randn(m, k, generator=g, device=DEV).half()
    bias = torch.randn(n, generator=g, device=DEV).half()
    pw, ps = Q.pack_w4a16_weights(words), Q.pack_w4a16_scales(scale, zero)
    s16, nzs = scale.half().double(), (-zero * scale).half().double()
    w = (q.view(n, k // 128, 128).double() * s16[..., None] + nzs[..., None]).half().double().view(n, k)   # one rounding, as the kernel's fma
    want = x.double() @ w.T
    near(Q.w4a16_matmul_prepacked_rows(x, pw, ps, bias=bias), want + bias.double())
    pairs = want.half().double()
    act = Q.w4a16_matmul_prepacked_rows(x, pw, ps, gate_up_swiglu=True)
    ref = torch.nn.functional.silu(pairs[:, 0::2]) * pairs[:, 1::2]
    # gate and up are rounded to fp16 first: a unit of each, times the other
    bar = 2.0 ** -9 * (ref.abs() + pairs[:, 0::2].abs() + pairs[:, 1::2].abs() + 1)
    assert ((act.double() - ref).abs() <= bar).all()


@pytest.mark.parametrize("m,n,k", [(65, 32, 4224), (129, 5120 + 96, 2304), (4300, 4096, 1920)])
@pytest.mark.parametrize("fmt,gn,gk", [("fp8", 128, 128), ("fp8", 1, 384), ("int8", 1, 1 << 30)])
def test_8bit_weights(m, n, k, fmt, gn, gk):
    from lite_llama_amd import kernels as K

    if k % gk and gk < k:
        gk = 128
    gk = min(gk, k)
    assert shared(m, n, k, 1 if fmt == "fp8" else 2)
    g = gen(n)
    if fmt == "fp8":
        w = (torch.randn(n, k, generator=g, device=DEV) * 60).clamp(-448, 448).to(torch.float8_e4m3fn)
        codes, wide, unit = w.view(torch.uint8), w.double(), 1 / 60
    else:
        codes = torch.randint(-127, 128, (n, k), generator=g, device=DEV, dtype=torch.int8)
        wide, unit = codes.double(), 1 / 64
    scale = ((torch.rand(-(-n // gn), k // gk, generator=g, device=DEV) + 0.5) * unit).half().float()
    x = torch.randn(m, k, generator=g, device=DEV).half()
    bias = torch.randn(n, generator=g, device=DEV).half()

    def spread(s):
        return s.repeat_interleave(gn, 0)[:n].repeat_interleave(gk, 1)

    # weight times scale is rounded to fp16 once (fp8: the widened value, 2^-8 of it, times 256 scales)
    w16 = (wide * spread(scale.double())).half().double() if fmt == "int8" else (
        (wide / 256).half().double() * spread((scale * 256).half().double())).half().double()
    near(K.w8a16_matmul(x, codes, scale, group_n=gn, group_k=gk, bias=bias), x.double() @ w16.T + bias.double())


@pytest.mark.parametrize("m,n,k", [(65, 32, 3072), (300, 4096 + 32, 4352), (1300, 6144, 3072), (4200, 4096, 3840)])
@pytest.mark.parametrize("with_bias", [False, True])
def test_int8_by_int8(m, n, k, with_bias):
    from lite_llama_amd import kernels as K
    from lite_llama_amd import _lib as L

    assert shared(m, n, k, 3) or m == 1300
    g = gen(k)
    w = torch.randint(-127, 128, (n, k), generator=g, device=DEV, dtype=torch.int8)
    scale = torch.rand(n, generator=g, device=DEV) * 0.01
    bias = torch.randn(n, generator=g, device=DEV).half() if with_bias else None
    x = torch.randn(m, k, generator=g, device=DEV).half()
    got, sums, qa, a = K.smoothquant_matmul(x, w, scale, bias=bias, _return_int32=True)
    assert torch.equal(sums.double(), qa.double() @ w.double().T)
    plain = torch.empty_like(got)     # the same call without scratch memory: the same bits
    ws, cnt = L.gemm_workspace(x.device, m, n, k)
    L.check(L.lib().ll_w8a8_matmul(plain.data_ptr(), qa.data_ptr(), a.data_ptr(), w.data_ptr(), scale.data_ptr(), L.ptr(bias), m, n, k,
                                   w.stride(0), 0, ws.data_ptr(), cnt.data_ptr(), L.stream_ptr()), "plain")
    assert torch.equal(got, plain)
