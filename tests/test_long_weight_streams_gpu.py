"""Row-group products over weight streams long enough to be staggered (csrc/gemm_w16_rows.hip) against products of the same operands in fp32 / int64."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
# (rows a multiple of 4 KB: every workgroup of its own column; the last two, 256 MB as well, are of other rows: all from column 0)
@pytest.mark.parametrize("n,k", [(65536 + 32, 2048), (32768 + 96, 4096), (8192, 16384), (32768, 4224), (262144 * 4, 128)])
@pytest.mark.parametrize("m", [1, 33])
def test_staggered_rows(dtype, n, k, m):
    from lite_llama_amd.kernels.quantization import dense16_rows_linear

    g = torch.Generator(device=DEV).manual_seed(n + k)
    w = (torch.randn(n, k, generator=g, device=DEV, dtype=torch.float32) * k ** -0.5).to(dtype)
    x = torch.randn(m, k, generator=g, device=DEV).to(dtype)
    got = dense16_rows_linear(x, w)
    want = torch.cat([x.float() @ part.float().T for part in w.split(65536)], dim=1)
    # one rounding to the storage dtype; fp32 sums of k products of size ~ k^-1/2 in another order: far below 2^-14
    unit = 2.0 ** (-11 if dtype == torch.float16 else -8)
    assert ((got.float() - want).abs() <= unit * want.abs() + 2.0 ** -14).all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n,k", [(65536 + 32, 2048), (33792 + 32, 4096)])
def test_a_rows_sums_do_not_depend_on_how_many_rows_there_are(dtype, n, k):
    """Tiles of four and of eight row groups (up to 32 rows, more) begin a staggered weight's rows at the same column."""
    from lite_llama_amd.kernels.quantization import dense16_rows_linear

    g = torch.Generator(device=DEV).manual_seed(n)
    w = (torch.randn(n, k, generator=g, device=DEV) * k ** -0.5).to(dtype)
    x = torch.randn(64, k, generator=g, device=DEV).to(dtype)
    every = dense16_rows_linear(x, w)
    for m in (1, 32, 33):
        assert torch.equal(dense16_rows_linear(x[:m], w), every[:m])


def test_staggered_int8_rows():
    from lite_llama_amd.kernels.quantization import smoothquant_rows_matmul

    n, k, m = 16384 + 32, 4096, 30
    g = torch.Generator(device=DEV).manual_seed(7)
    w = torch.randint(-127, 128, (n, k), generator=g, device=DEV, dtype=torch.int8)
    scale = torch.rand(n, generator=g, device=DEV) * 1e-3
    x = torch.randn(m, k, generator=g, device=DEV).half()
    out = smoothquant_rows_matmul(x, w, scale)
    head = smoothquant_rows_matmul(x, w[:8192], scale[:8192])   # (32 MB: not staggered; sums of whole numbers have one value)
    assert torch.equal(out[:, :8192], head)


# more than four row groups per CU: tiles of eight for more than 32 rows; runs of 4 and 5, 8 and 9, 17 groups; one unit of the contraction
@pytest.mark.parametrize("n", [32 * 1025, 32 * 2049, 32 * 4352])
@pytest.mark.parametrize("k", [128, 512])
@pytest.mark.parametrize("m", [32, 33, 64])
@pytest.mark.parametrize("swiglu", [False, True])
def test_row_group_runs(n, k, m, swiglu):
    from lite_llama_amd.kernels.quantization import dense16_rows_linear, quantize_activations_int8, smoothquant_rows_matmul

    g = torch.Generator(device=DEV).manual_seed(n + k)
    w = (torch.randn(n, k, generator=g, device=DEV) * k ** -0.5).half()
    x = torch.randn(m, k, generator=g, device=DEV).half()
    want = x.float() @ w.float().T
    got = dense16_rows_linear(x, w, gate_up_swiglu=swiglu)
    if swiglu:
        gate, up = want[:, 0::2].half().float(), want[:, 1::2].half().float()
        want = torch.nn.functional.silu(gate) * up
        # gate and up are rounded to fp16 first: a unit of each, times the other (and |silu'| <= 1.1)
        bar = 2.0 ** -9 * (want.abs() + gate.abs() + up.abs() + 2.0 ** -4)
    else:
        bar = 2.0 ** -11 * want.abs() + 2.0 ** -14
    assert ((got.float() - want).abs() <= bar).all()
    if not swiglu and k % 256 == 0:
        codes = torch.randint(-127, 128, (n, k), generator=g, device=DEV, dtype=torch.int8)
        scale = torch.rand(n, generator=g, device=DEV) * 1e-3
        qa, a = quantize_activations_int8(x)
        sums = qa.float() @ codes.float().T                 # (whole numbers below 2^24: exact)
        assert torch.equal(smoothquant_rows_matmul(x, codes, scale), ((sums * a.view(-1, 1)) * scale.view(1, -1)).half())


# 64 to 256 MB: six and seven row groups per CU (tiles of up to four, of up to eight for more than 32 rows), one and two
MIDDLE = [(49152 + 32, 2048), (8192 + 32, 8192), (14336, 4096)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n,k", MIDDLE)
def test_sums_of_streams_of_middle_length(dtype, n, k):
    """In the order of columns, as those of short streams: 32 MB of the same weights give the same bits."""
    from lite_llama_amd.kernels.quantization import dense16_rows_linear

    g = torch.Generator(device=DEV).manual_seed(n + k)
    w = (torch.randn(n, k, generator=g, device=DEV) * k ** -0.5).to(dtype)
    x = torch.randn(64, k, generator=g, device=DEV).to(dtype)
    every, want = dense16_rows_linear(x, w), x.float() @ w.float().T
    unit = 2.0 ** (-11 if dtype == torch.float16 else -8)   # as above
    assert ((every.float() - want).abs() <= unit * want.abs() + 2.0 ** -14).all()
    for m in (1, 32, 33):
        assert torch.equal(dense16_rows_linear(x[:m], w), every[:m])
    part = (1 << 24) // k
    assert torch.equal(dense16_rows_linear(x, w[:part]), every[:, :part])


@pytest.mark.parametrize("m", [30, 33, 64])
@pytest.mark.parametrize("n,k", [(40960 + 32, 4096), (16384, 8192)])
def test_staggered_int8_rows_in_all_tiles(m, n, k):
    from lite_llama_amd.kernels.quantization import quantize_activations_int8, smoothquant_rows_matmul

    g = torch.Generator(device=DEV).manual_seed(n + m)
    w = torch.randint(-127, 128, (n, k), generator=g, device=DEV, dtype=torch.int8)
    scale = torch.rand(n, generator=g, device=DEV) * 1e-3
    x = torch.randn(m, k, generator=g, device=DEV).half()
    qa, each = quantize_activations_int8(x)
    sums = torch.cat([qa.double() @ part.double().T for part in w.split(8192)], dim=1).float()   # (whole numbers: one value, whatever the order)
    assert torch.equal(smoothquant_rows_matmul(x, w, scale), ((sums * each.view(-1, 1)) * scale.view(1, -1)).half())


# (rows of weights, contraction): half a group at the end, runs dealt in halves (a CU with three), both, one workgroup
@pytest.mark.parametrize("n,k", [(48, 128), (8208, 128), (8224, 256), (12080, 384), (17936, 128), (4112, 640)])
@pytest.mark.parametrize("m", [1, 32, 33, 64])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_halves_of_row_groups(n, k, m, dtype):
    from lite_llama_amd.kernels.quantization import dense16_rows_linear

    g = torch.Generator(device=DEV).manual_seed(n + m)
    x = torch.randn(m, k, generator=g, device=DEV).to(dtype)
    w = (torch.randn(n, k, generator=g, device=DEV) * k ** -0.5).to(dtype)
    bias = torch.randn(n + 16, generator=g, device=DEV).to(dtype)[:n]
    # exact 16-bit products summed in fp32 (k 2^-24 of their magnitudes' sum, which stays below 40 deviations), rounded once
    unit, slack = 2.0 ** (-11 if dtype == torch.float16 else -8), k * 2.0 ** -24 * 40 + 2.0 ** -24
    want = x.double() @ w.double().T + bias.double()
    got = dense16_rows_linear(x, w, bias)
    assert ((got.double() - want).abs() <= unit * want.abs() + slack).all()
    plain = dense16_rows_linear(x, w)
    pairs = dense16_rows_linear(x, w, gate_up_swiglu=True)
    gate, up = plain[:, 0::2].double(), plain[:, 1::2].double()
    act = torch.nn.functional.silu(gate) * up
    assert ((pairs.double() - act).abs() <= unit * act.abs() + 2.0 ** -20 * (gate * up).abs() + 2.0 ** -24).all()
