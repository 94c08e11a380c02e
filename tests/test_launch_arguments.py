"""What the host side of a launch decides and hands its kernel, without a GPU: the source is compiled for the host alone and without
optimisation -- where a field that nobody assigned is whatever lay on the stack -- and the runtime's calls are replaced."""

import ctypes
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lite_llama_amd", "csrc")

# The calls that hipcc's launch stubs and the entry points make, so that the library needs no GPU runtime.
RUNTIME = r"""
#include <string.h>
static int launches = 0;
static dim3 cfg_grid, cfg_block;
static size_t cfg_lds = 0;
extern "C" {
void** __hipRegisterFatBinary(void*) { static void* h; return &h; }
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*, void*, int*) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void**) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t s, hipStream_t) { cfg_grid = g; cfg_block = b; cfg_lds = s; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* s, hipStream_t* st) {
  *g = cfg_grid; *b = cfg_block; *s = cfg_lds; *st = nullptr;
  return hipSuccess;
}
static int on_device = 0, asked_on[4];
hipError_t hipGetDevice(int* d) { *d = on_device; return hipSuccess; }
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { ++asked_on[on_device]; return hipSuccess; }
void use_device(int d) { on_device = d; }
int attributes_asked(int d) { return asked_on[d]; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipPeekAtLastError() { return hipSuccess; }
}
"""

SCAN = r"""
static ScanArgs kept[8];
extern "C" {
hipError_t hipLaunchKernel(const void*, dim3, dim3, void** args, size_t, hipStream_t) {
  if (launches < 8) memcpy(&kept[launches++], args[0], sizeof(ScanArgs));
  return hipSuccess;
}
// what an earlier call may have left on the stack
__attribute__((noinline)) void dirty_stack() {
  volatile unsigned char junk[1 << 16];
  for (int i = 0; i < (int)sizeof(junk); ++i) junk[i] = 0xA5;
  launches = 0;
}
int launch_count() { return launches; }
void launch_pointers(int i, const void** out) {
  const void* p[4] = {kept[i].seq_start, kept[i].seq_first_pos, kept[i].seq_slot, kept[i].state};
  memcpy(out, p, sizeof(p));
}
int launch_tokens_per_pass(int i) { return kept[i].tb; }
}
"""

PLAN = r"""
extern "C" {
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) { return hipSuccess; }
void decode_plan(int64_t max_len, int64_t pairs, int heads, int d, int planes, int* out) {
  const FdPlan p = fd_plan(max_len, pairs, heads, d, planes != 0);
  out[0] = p.waves;
  out[1] = p.splits;
}
void decode_plan_merged(int64_t max_len, int64_t pairs, int heads, int d, int* out) {
  const FdPlan p = fd_plan(max_len, pairs, heads, d, true, true);
  out[0] = p.waves;
  out[1] = p.splits;
}
int decode_alone() { return FD_ALONE * FD_PART; }
}
"""

TILES = r"""
extern "C" {
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) { return hipSuccess; }
int wants(int64_t m, int64_t n, int64_t k, int wf) { return tile256_wants(m, n, k, wf); }
}
"""


def _host_library(where, source, extra):
    from lite_llama_amd import build

    src, lib = where / "host.hip", where / "host.so"
    src.write_text(f'#include "{source}"\n' + RUNTIME + extra)
    subprocess.run([build._hipcc(), "--offload-host-only", "--offload-arch=" + build.ARCH, "-O0", "-std=c++17", "-fPIC", "-I", CSRC, "-c",
                    str(src), "-o", str(where / "host.o")], check=True, capture_output=True, text=True)
    # the device code that the object would register: an address that nothing looks at
    names = subprocess.run(["nm", "-u", str(where / "host.o")], check=True, capture_output=True, text=True).stdout.split()
    defs = [f"-Wl,--defsym,{n}=0" for n in names if n.startswith("__hip_fatbin")]
    subprocess.run(["g++", "-shared", str(where / "host.o"), *defs, "-o", str(lib)], check=True, capture_output=True, text=True)
    return ctypes.CDLL(str(lib))


@pytest.fixture(scope="module")
def linear_mix(tmp_path_factory):
    return _host_library(tmp_path_factory.mktemp("host_linear_mix"), "linear_mix.hip", SCAN)


@pytest.fixture(scope="module")
def flash_decoding(tmp_path_factory):
    return _host_library(tmp_path_factory.mktemp("host_flash_decoding"), "flash_decoding.hip", PLAN)


BATCH, HEADS, DK, DV = 2, 4, 64, 32


def _call(lib, name, kind, longest, scratch):
    """One linear_scan of ``longest`` tokens per sequence over made-up addresses (nothing reads them): the addresses given."""
    p = {k: 0x10000 * (i + 1) for i, k in enumerate(["q", "k", "v", "head_decay", "gate", "gate_bias", "dt", "dt_bias", "a_log", "skip", "o",
                                                     "seq_start", "seq_first_pos", "seq_slot", "state", "scratch"])}
    P, L, F, I = ctypes.c_void_p, ctypes.c_int64, ctypes.c_float, ctypes.c_int
    fn = getattr(lib, name)
    fn.restype = I
    fn.argtypes = [P, L, P, L, P, L, L, L, L, L, I, I, F, P, P, L, P, F, P, L, P, P, P, P, L, P, P, P, P, P, L, L, I, P]
    rc = fn(p["q"], HEADS * DK, p["k"], HEADS * DK, p["v"], HEADS * DV, HEADS, DK, DV, 1, kind, 0, 1.0, p["head_decay"], p["gate"], HEADS * DK,
            p["gate_bias"], 1.0, p["dt"], HEADS, p["dt_bias"], p["a_log"], p["skip"], p["o"], BATCH, p["seq_start"], p["seq_first_pos"],
            p["seq_slot"], p["state"], p["scratch"] if scratch else None, BATCH * longest, longest, 1, None)
    assert rc == 0
    return [p[k] for k in ("seq_start", "seq_first_pos", "seq_slot", "state")]


@pytest.mark.parametrize("kind", [0, 1, 2])
@pytest.mark.parametrize("name,longest,launches", [("ll_linear_scan_walk", 24, 2), ("ll_linear_scan_walk", 1000, 2), ("ll_linear_scan", 1000, 1),
                                                   ("ll_linear_scan", 1, 1)])
def test_linear_scan_hands_over_its_runs_and_state(linear_mix, name, longest, launches, kind):
    linear_mix.dirty_stack()
    want = _call(linear_mix, name, kind, longest, scratch=name.endswith("walk"))
    assert linear_mix.launch_count() == launches
    for i in range(launches):
        got = (ctypes.c_void_p * 4)()
        linear_mix.launch_pointers(i, got)
        assert list(got) == want
    assert 1 <= linear_mix.launch_tokens_per_pass(launches - 1) <= 16


def _plan(lib, tokens, pairs, heads=4, d=128, planes=False):
    out = (ctypes.c_int * 2)()
    lib.decode_plan(ctypes.c_int64(tokens), ctypes.c_int64(pairs), heads, d, int(planes), out)
    return tuple(out)


@pytest.mark.parametrize("tokens", [1025, 1500, 2048, 3000, 4096, 6000, 8192, 16384, 32768])
@pytest.mark.parametrize("heads", [1, 4, 8, 16])
def test_a_long_row_is_spread_whatever_stands_beside_it(flash_decoding, tokens, heads):
    """The launch knows the longest row's bound only: beside short rows it must still have waves enough of its own (one workgroup per CU in
    all left a row of 32 768 tokens beside 49 short ones to 16 waves: 94 -> 233 us), and few pairs must reach many CUs."""
    np_ = -(-tokens // 128)
    for pairs in (1, 2, 8, 24, 32, 33, 40, 64, 65, 80, 96, 100, 127):
        waves, splits = _plan(flash_decoding, tokens, pairs, heads)
        assert waves in (2, 4, 8) and 1 <= splits <= min(np_, 32)
        assert waves * splits * 8 >= np_ * 0.75                       # at most about ten partitions a wave
        assert pairs * splits >= min(160, pairs * min(32, np_ // 2))  # .. and most CUs have a workgroup
        planes = _plan(flash_decoding, tokens, pairs, heads, planes=True)
        assert planes[0] >= 4 and planes[1] >= 1                      # (18 rows of a head fit the planes' two pieces per lane)


def test_more_lds_than_a_launch_has_is_asked_for_on_every_device(flash_decoding):
    """Eight waves of decode attention hold 74 KB: granted to a kernel on the device that is current, and no other."""
    P, L, I, F = ctypes.c_void_p, ctypes.c_int64, ctypes.c_int, ctypes.c_float
    flash_decoding.ll_flash_decoding.argtypes = [P] * 9 + [I, I, I, I, L, F] + [L] * 9 + [I, I, I, P, P]
    for device in (0, 1, 1, 0):
        flash_decoding.use_device(device)
        before = flash_decoding.attributes_asked(device)
        assert flash_decoding.ll_flash_decoding(*[4096] * 9, 2, 16, 1, 128, 1024, 0.1, *[2048, 128] * 4, 64, 1, 0, 0, 4096, None) == 0
        assert flash_decoding.attributes_asked(device) >= 1 and before <= flash_decoding.attributes_asked(device) <= 1
    flash_decoding.use_device(0)


def test_decode_plans_of_other_calls(flash_decoding):
    for d in (32, 64, 128, 256):
        for tokens in (0, 1, 128):
            assert _plan(flash_decoding, tokens, 5, d=d) == (0, 0)
        for tokens in (129, 700, 1024):                              # a wave per partition
            for pairs in (1, 500):
                assert _plan(flash_decoding, tokens, pairs, d=d) == (-(-tokens // 128), 1)
        assert _plan(flash_decoding, 5000, 128, d=d) == (8, 1)       # the pairs fill the chip
        assert _plan(flash_decoding, 32769, 500, d=d) == (0, 0)
    for pairs in (1, 16, 40, 127):                                   # heads of 256 spill in a grouped workgroup
        assert _plan(flash_decoding, 1025, pairs, d=256) == (0, 0)
        assert (_plan(flash_decoding, 32768, pairs, d=256)[0] == 8) == (pairs <= 16)


@pytest.mark.parametrize("heads", range(1, 17))
def test_rows_of_five_to_eight_partitions_in_several_workgroups(flash_decoding, heads):
    """Every lane of the workgroup that merges has a float4 of the result, in one round; a row that is not spread has a wave for every partition."""
    out = (ctypes.c_int * 2)()
    alone = flash_decoding.decode_alone()
    assert alone == 384
    for tokens, splits in ((513, 3), (640, 3), (641, 3), (768, 3), (769, 4), (1024, 4)):
        for pairs in (1, 64, 256 // splits, 256 // splits + 1):
            flash_decoding.decode_plan_merged(ctypes.c_int64(tokens), ctypes.c_int64(pairs), heads, 128, out)
            if pairs * splits > 256:
                assert tuple(out) == (-(-tokens // 128), 1)
                continue
            assert out[1] == splits and 64 * out[0] >= heads * 128 // 4 and 128 * out[0] >= alone and out[0] <= 8
            assert 128 * out[0] >= (heads + 2) * 128 // 4             # (the planes' two pieces per lane)
    flash_decoding.decode_plan_merged(ctypes.c_int64(1024), ctypes.c_int64(8), heads, 64, out)
    assert tuple(out) == (8, 1)


def test_the_switch_back_to_a_workgroup_per_partition(flash_decoding, tmp_path, monkeypatch):
    copy = tmp_path / "host.so"
    shutil.copy(flash_decoding._name, copy)   # (read once per library)
    monkeypatch.setenv("LL_FD_NO_LOOP", "1")
    lib = ctypes.CDLL(str(copy))
    for pairs in (1, 40, 500):
        assert _plan(lib, 1025, pairs) == _plan(lib, 32768, pairs) == (0, 0)
        assert _plan(lib, 1024, pairs) == (8, 1)


@pytest.fixture(scope="module")
def wants(tmp_path_factory):
    fn = _host_library(tmp_path_factory.mktemp("host_tile256"), "gemm_tile256.hip", TILES).wants
    fn.argtypes, fn.restype = [ctypes.c_int64] * 3 + [ctypes.c_int], ctypes.c_int
    return fn


MTILED = r"""
static unsigned threads = 0;
extern "C" {
hipError_t hipLaunchKernel(const void*, dim3, dim3 b, void**, size_t, hipStream_t) { threads = b.x; return hipSuccess; }
unsigned launched_threads() { return threads; }
}
"""


@pytest.mark.parametrize("source,knob", [("gemm_w4_prefill.hip", "LL_PF_WMH"), ("gemm_w8_prefill.hip", "LL_P8_WMH")])
def test_a_forced_tile_height_is_the_128_row_engines(tmp_path, monkeypatch, source, knob):
    monkeypatch.setenv(knob, "1")
    lib = _host_library(tmp_path, source, '#include "gemm_tile256.hip"\n' + MTILED)
    P, L, I = ctypes.c_void_p, ctypes.c_int64, ctypes.c_int
    m, n, k = 8192, 5120, 2048   # (on the 256 x 256 tiles by their rule)
    if knob == "LL_PF_WMH":
        lib.ll_w4a16_matmul_prepacked_mtiled.argtypes = [P] * 5 + [L, L, L, I, L, I, P]
        assert lib.ll_w4a16_matmul_prepacked_mtiled(*[4096] * 4, None, m, n, k, 128, k, 0, None) == 0
    else:
        lib.ll_w8_mtiled_try.argtypes = [P] * 7 + [L, L, L, I, L, I, L, L, L, L, P, L, P]
        assert lib.ll_w8_mtiled_try(*[4096] * 4, None, None, None, m, n, k, n, k, 1, k, k, 1, 1, None, 0, None) == 1
    assert lib.launched_threads() == 256


# (rows, columns, contraction): which engine was faster, alone on the GPU; 0 int4, 1 fp8, 2 int8 weights, 3 int8 x int8
@pytest.mark.parametrize("fmt,shape,tiles", [
    (0, (8144, 37888, 3584), 1), (0, (1024, 5120, 3584), 1), (0, (4096, 3584, 3584), 1), (0, (10700, 3584, 3584), 1), (0, (16384, 2048, 1024), 1),
    (0, (4096, 4352, 3584), 0), (0, (6144, 4096, 3584), 0), (0, (9300, 3584, 1024), 0), (0, (2048, 12288, 1024), 0), (0, (1024, 3584, 3584), 0),
    (0, (8192, 4096, 1024), 0), (0, (300, 4352, 512), 0), (0, (16384, 28672, 1024), 0), (0, (512, 5120, 640), 1),
    (1, (8192, 5120, 2048), 1), (1, (96, 5120, 2048), 1), (1, (96, 4096, 4096), 1), (1, (1024, 4096, 1024), 1), (1, (4096, 1024, 512), 1),
    (1, (256, 4096, 2048), 0), (1, (65, 32, 512), 0), (1, (512, 256, 2048), 0), (1, (2048, 12288, 512), 0), (1, (2048, 12288, 256), 0),
    (2, (8192, 5120, 2048), 1), (2, (4096, 4096, 4096), 1), (2, (1024, 12288, 768), 1),
    (2, (1024, 4096, 1024), 0), (2, (256, 2048, 2560), 0), (2, (2048, 4352, 768), 0), (2, (4096, 4096, 512), 0),
    (3, (5000, 28672, 4096), 1), (3, (65, 28672, 512), 1), (3, (256, 4096, 2048), 1), (3, (1000, 4096, 1024), 1),
    (3, (65, 4096, 2048), 0), (3, (192, 1024, 1024), 0), (3, (300, 256, 512), 0), (3, (600, 32, 1024), 0)])
def test_the_256_tiles_are_taken_where_they_are_faster(wants, fmt, shape, tiles):
    assert wants(*shape, fmt) == tiles
    assert wants(shape[0], shape[1], shape[2] + 64, fmt) == 0      # an odd number of steps


@pytest.mark.parametrize("experts,top,hidden,inter,tokens,int8,pays", [
    (128, 8, 2048, 768, 8192, False, True), (64, 8, 1024, 512, 1024, True, True), (8, 2, 4096, 14336, 1024, True, True),
    (8, 2, 2048, 768, 2048, False, True), (8, 2, 2048, 768, 1024, False, False), (4, 2, 1024, 512, 512, False, False),
    (4, 2, 4096, 14336, 512, True, False), (16, 4, 256, 384, 1024, False, False)])
def test_expert_blocks_of_256_are_taken_where_they_fill_the_chip(experts, top, hidden, inter, tokens, int8, pays):
    import torch

    from lite_llama_amd.kernels.fused_moe import _tiles_256_pay

    w1, w2 = (torch.empty(experts, *s, dtype=torch.int8, device="meta") for s in ((2 * inter, hidden), (hidden, inter)))
    assert _tiles_256_pay(tokens * top, experts, w1, w2, int8) == pays


ROUTER = r"""
static unsigned most_lds = 0;
bool moe_stream_wants(const MoeStreamParams&, int, int, int, int64_t, int64_t) { return false; }
int moe_stream_launch(const MoeStreamParams&, int, int, int, int64_t, hipStream_t) { return LL_OK; }
extern "C" {
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t lds, hipStream_t) {
  if (lds > most_lds) most_lds = lds;
  return hipSuccess;
}
unsigned router_lds() { const unsigned n = most_lds; most_lds = 0; return n; }
}
"""


def test_every_router_that_is_accepted_fits_the_lds_of_a_launch(tmp_path):
    lib = _host_library(tmp_path, "moe_sparse.hip", ROUTER)
    P, L, I, F = ctypes.c_void_p, ctypes.c_int64, ctypes.c_int, ctypes.c_float
    lib.ll_group_router.argtypes = [P, L, P, P, L, L, L, L, L, L, F, I, P, P, P, P, P, L, I, P]
    for scoring in range(5):
        for experts, groups, top in [(4096, 4096, 64), (4096, 1, 64), (4096, 2048, 64), (513, 513, 64), (512, 512, 64), (511, 511, 64), (64, 64, 64)]:
            groups = 1 if scoring in (1, 2) else groups
            for tokens in (1, 300):
                assert lib.ll_group_router(4096, 64, 4096, None, tokens, 64, experts, top, groups, groups, 1.0, scoring, *[4096] * 4, None, 0, 1, None) == 0
                assert 0 < lib.router_lds() <= 64 * 1024, (scoring, experts, groups, tokens)
    # ... and where the choices are sorted in the same launch, which holds 128 bytes of its own beside what it is given
    lib.ll_group_router_sorted.argtypes = [P, L, P, P, L, L, L, L, L, L, F, I, P, P, P, P, P, L, L, L, I, P, P, P, P, I, P]
    for scoring in range(5):
        for experts in (34, 128, 129, *range(466, 514)):
            for tokens, top in ((1, 8), (16, 8), (12, 12), (16, 64), (1, 64)):
                assert lib.ll_group_router_sorted(4096, 64, 4096, None, tokens, 64, experts, min(top, experts), 1, 1, 1.0, scoring, *[4096] * 4, None, 0,
                                                  experts, 128, 0, *[4096] * 4, 1, None) == 0
                assert 0 < lib.router_lds() <= 64 * 1024 - 128, (scoring, experts, tokens, top)


# (tokens, heads, key heads, key width, value width, kind): the longest steps, a little below 2^28 floats of pairs, decays and steps
@pytest.mark.parametrize("n,heads,qk_heads,dk,dv,kind", [(65000, 16, 16, 128, 128, 0), (43000, 8, 8, 256, 256, 1), (130000, 8, 8, 128, 256, 0),
                                                         (64000, 32, 16, 128, 64, 2), (500000, 8, 4, 64, 64, 2), (24, 4096, 4096, 256, 512, 1)])
def test_long_steps_keep_the_walk_in_two_kernels(linear_mix, n, heads, qk_heads, dk, dv, kind):
    fn = linear_mix.ll_linear_scan_walk_floats
    fn.argtypes, fn.restype = [ctypes.c_int64] * 6 + [ctypes.c_int, ctypes.c_int64], ctypes.c_int64
    terms = qk_heads * dk * 2 + (heads * dk if kind == 1 else 0) + (heads * 2 if kind == 2 else 0)
    assert 0.7 * 2 ** 28 < n * terms <= 2 ** 28 or n == 24
    assert fn(n, 4, heads, dk, dv, heads // qk_heads, kind, n // 4 + 24) == (n + 8) * (terms + heads * -(-dv // 32) * 32)
    assert fn(2 ** 28 // terms + 1, 4, heads, dk, dv, heads // qk_heads, kind, 1000) == 0
    assert fn(n, 4, heads, dk, dv, heads // qk_heads, kind, 23) == 0


MOE = r"""
#include "gemm_tile256.h"
static int64_t asked[2];
int tile256_grouped_launch(T2Params&, int, void*) { return LL_OK; }
bool moe_stream_wants(const MoeStreamParams&, int, int, int, int64_t experts, int64_t runs) { asked[0] = experts; asked[1] = runs; return false; }
int moe_stream_launch(const MoeStreamParams&, int, int, int, int64_t, hipStream_t) { return LL_OK; }
extern "C" {
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) { return hipSuccess; }
void stream_asked(int64_t* out) { out[0] = asked[0]; out[1] = asked[1]; asked[0] = asked[1] = 0; }
}
"""


@pytest.fixture(scope="module")
def moe_gemm(tmp_path_factory):
    """Experts and runs that a call of ll_moe_gemm names to the streaming form, or ``(0, 0)`` where it does not ask."""
    lib = _host_library(tmp_path_factory.mktemp("host_moe"), "moe.hip", MOE)
    P, L, I = ctypes.c_void_p, ctypes.c_int64, ctypes.c_int
    lib.ll_moe_gemm.argtypes = [P] * 8 + [L, L, I, L, L, I, I, I, I, L, L, L, L, L, L, L, I, P]

    def call(fmt, experts, slots, block, n, k, spare=0):
        em = slots + experts * (block - 1) + spare
        wf = {"f16": 0, "fp8": 1, "int8": 2}[fmt]
        assert lib.ll_moe_gemm(*[4096] * 8, slots, em, block, n, k, 1, 0, wf, 128, 128, k, n * k, k, 1, 1, 1, 0, None) == 0
        out = (ctypes.c_int64 * 2)()
        lib.stream_asked(out)
        return tuple(out)

    return call


@pytest.mark.parametrize("experts", [1, 2, 4, 8, 34, 128, 300])
@pytest.mark.parametrize("block", [16, 32, 64])
@pytest.mark.parametrize("fmt", ["f16", "fp8"])
def test_the_streaming_form_counts_the_experts(moe_gemm, experts, block, fmt):
    """Not the blocks of their lists, which grow with the slots: the rows per expert from which tiles are faster are rows per expert."""
    for rows in (1, 5, 10):
        slots = rows * experts
        asked, runs = moe_gemm(fmt, experts, slots, block, 1536, 2048)
        assert asked == experts
        assert runs >= min(experts, slots) and runs * block >= slots + experts * (block - 1)   # (blocks that the lists can hold)


# (format, experts, n, k, rows per expert): which form was faster, both products of fused_moe on the GPU
@pytest.mark.parametrize("fmt,experts,n,k,rows,stream", [
    ("fp8", 128, 1536, 2048, 18, True), ("fp8", 128, 1536, 2048, 20, False), ("int8", 128, 1536, 2048, 28, False), ("fp8", 128, 3072, 4096, 18, True),
    ("fp8", 128, 1024, 1024, 12, True), ("fp8", 128, 1024, 1024, 14, False), ("fp8", 200, 1024, 2048, 18, True), ("fp8", 64, 1536, 2048, 22, True),
    ("fp8", 64, 1536, 2048, 28, False), ("fp8", 32, 1536, 2048, 24, True), ("fp8", 32, 1536, 2048, 32, False), ("int8", 8, 28672, 4096, 24, True),
    ("int8", 8, 28672, 4096, 40, False), ("f16", 128, 1536, 2048, 20, True), ("f16", 128, 1536, 2048, 28, False),
    ("f16", 64, 2048, 2048, 32, True), ("f16", 64, 2048, 2048, 64, False), ("f16", 4, 1024, 1024, 80, True), ("f16", 34, 2048, 704, 80, True),
    ("fp8", 4, 1024, 1024, 32, True), ("fp8", 4, 1024, 1024, 100, False), ("f16", 48, 2816, 2048, 24, True),
    ("f16", 48, 2816, 2048, 40, False), ("f16", 34, 1408, 2048, 56, True), ("f16", 16, 2048, 2048, 56, True), ("f16", 16, 2048, 2048, 64, False),
    ("f16", 8, 28672, 4096, 56, True), ("f16", 8, 28672, 4096, 64, False)])
def test_the_streaming_form_is_asked_where_it_is_faster(moe_gemm, fmt, experts, n, k, rows, stream):
    assert (moe_gemm(fmt, experts, rows * experts, 64, n, k)[0] == experts) == stream
