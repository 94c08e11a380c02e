"""Linear attention with a decay over runs of many tokens (csrc/linear_mix.hip: the tokens' terms ahead of the walk) and decoded tokens in
64-column workgroups, against 64 bits and bit for bit against the walk in one kernel, which serves a step whose longest run is not known."""

import dataclasses

import pytest
import torch

from tests.test_layered_gpu import _step

pytestmark = pytest.mark.gpu
DEV, F64 = "cuda", torch.float64


def _inputs(kind, heads, qk_heads, dk, dv, n, dtype, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)

    def r(*s):
        return torch.randn(*s, generator=g, device=DEV).to(dtype)

    # (rows of a fused projection: column ranges, starts off every 16-byte border)
    rows = r(n, 2 * qk_heads * dk + heads * dv + 3)
    q, k, v = rows[:, 1:1 + qk_heads * dk], rows[:, 2 + qk_heads * dk:2 + 2 * qk_heads * dk], rows[:, 3 + 2 * qk_heads * dk:]
    if kind == "fixed":
        kw = dict(act=True, head_decay=torch.linspace(1.0, 0.25, heads, device=DEV))
    elif kind == "entry":
        kw = dict(q_scale=dk ** -0.5, gate=r(n, heads * dk), gate_bias=r(heads * dk), tau=4.0)
    else:
        kw = dict(dt=r(n, heads), dt_bias=r(heads), a_log=r(heads), skip=r(heads))
    return q, k, v, dict(kw, qk_heads=qk_heads)


def _exact(q, k, v, heads, dk, dv, runs, state, kw):
    qk_heads = kw["qk_heads"]
    q, k, v = q.to(F64).reshape(-1, qk_heads, dk), k.to(F64).reshape(-1, qk_heads, dk), v.to(F64).reshape(-1, heads, dv)
    b = torch.ones(v.shape[0], heads, 1, dtype=F64, device=DEV)
    if "head_decay" in kw:
        q, k, v = (torch.nn.functional.silu(t) for t in (q, k, v))
        a = kw["head_decay"].to(F64).view(1, heads, 1).expand(v.shape[0], heads, dk)
    elif "gate" in kw:
        q = q * float(torch.tensor(kw["q_scale"], dtype=torch.float32))
        a = torch.exp(torch.nn.functional.logsigmoid(kw["gate"].to(F64) + kw["gate_bias"].to(F64)) / kw["tau"]).view(-1, heads, dk)
    else:
        b = torch.nn.functional.softplus(kw["dt"].to(F64) + kw["dt_bias"].to(F64)).unsqueeze(-1)
        a = torch.exp(-torch.exp(kw["a_log"].to(F64)).view(1, heads, 1) * b).expand(-1, heads, dk)
    q, k = q.repeat_interleave(heads // qk_heads, 1), k.repeat_interleave(heads // qk_heads, 1)
    out, state, at = torch.empty_like(v), state.to(F64).clone(), 0
    for i, (first, count) in enumerate(runs):
        s = state[i] if first else torch.zeros_like(state[i])
        for t in range(at, at + count):
            s = a[t].unsqueeze(-1) * s + k[t].unsqueeze(-1) * (b[t] * v[t]).unsqueeze(1)
            out[t] = torch.einsum("hkv,hk->hv", s, q[t])
        state[i], at = s, at + count
    if "skip" in kw:
        out += kw["skip"].to(F64).view(1, heads, 1) * v
    return out.reshape(-1, heads * dv), state


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("kind,heads,qk_heads,dk,dv", [("fixed", 3, 3, 64, 17), ("fixed", 2, 1, 128, 64), ("entry", 2, 2, 128, 40),
                                                     ("entry", 4, 2, 256, 9), ("token", 34, 2, 64, 4), ("token", 3, 1, 256, 80), ("entry", 20, 20, 64, 272)])
@pytest.mark.parametrize("runs", [[(0, 24)], [(5, 1), (9, 79), (0, 16), (3, 17), (0, 1)], [(2, 95), (0, 33)]])
def test_runs_of_many_tokens(dtype, kind, heads, qk_heads, dk, dv, runs):
    """Runs that end on and off eight tokens, beside single tokens; carried and fresh states; values off every tile of columns; one column
    per thread (two below)."""
    from lite_llama_amd import _lib
    from lite_llama_amd.kernels.recurrent import linear_scan

    n = sum(c for _, c in runs)
    q, k, v, kw = _inputs(kind, heads, qk_heads, dk, dv, n, dtype, dk + dv)
    step = _step([(i, f, c, 0) for i, (f, c) in enumerate(runs)], None)
    assert _lib.lib().ll_linear_scan_walk_floats(n, len(runs), heads, dk, dv, heads // qk_heads, ["fixed", "entry", "token"].index(kind),
                                                  step.longest_run) > 0
    start = torch.randn(len(runs), heads, dk, dv, device=DEV)
    want, want_state = _exact(q, k, v, heads, dk, dv, runs, start, kw)
    states = [start.clone(), start.clone()]
    outs = [linear_scan(q, k, v, heads, dk, dv, dataclasses.replace(step, longest_run=m), s, **kw) for m, s in zip((step.longest_run, 0), states)]
    # fp32 throughout: a few units of rounding per token of a run and per entry of a sum, against the largest result
    for x, y in ((outs[0], want), (states[0], want_state)):
        assert (x.to(F64) - y).abs().max() <= 64 * 2.0 ** -24 * y.abs().max()
    assert torch.equal(outs[0], outs[1]) and torch.equal(states[0], states[1])


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("kind,heads,qk_heads,dk,dv", [("fixed", 64, 64, 64, 200), ("entry", 48, 24, 128, 258), ("token", 112, 7, 256, 98)])
@pytest.mark.parametrize("runs", [[(0, 24)], [(5, 1), (9, 79), (0, 16), (3, 17), (0, 1)]])
def test_runs_of_many_tokens_in_two_columns_per_thread(dtype, kind, heads, qk_heads, dk, dv, runs):
    """Three workgroups of 16 columns per CU and more; a last slice of 2, 8 and 32 columns."""
    n, longest = sum(c for _, c in runs), max(c for _, c in runs)
    assert -(-n // longest) * heads * -(-dv // 16) >= 768   # (where the walk takes two)
    test_runs_of_many_tokens(dtype, kind, heads, qk_heads, dk, dv, runs)


def test_a_step_whose_scratch_passes_a_gigabyte():
    """Terms below 2^28 floats, terms and values above: the same bits as the walk in one kernel, at the far end of the scratch too."""
    from lite_llama_amd import _lib
    from lite_llama_amd.kernels.recurrent import linear_scan

    heads, dk, dv, runs = 16, 128, 128, [(0, 47000), (3, 24), (9, 1), (0, 975)]
    n = sum(c for _, c in runs)
    q, k, v, kw = _inputs("fixed", heads, heads, dk, dv, n, torch.bfloat16, 3)
    step = _step([(i, f, c, 0) for i, (f, c) in enumerate(runs)], None)
    assert _lib.lib().ll_linear_scan_walk_floats(n, len(runs), heads, dk, dv, 1, 0, step.longest_run) > 2 ** 28
    start = torch.randn(len(runs), heads, dk, dv, device=DEV)
    states = [start.clone(), start.clone()]
    outs = [linear_scan(q, k, v, heads, dk, dv, dataclasses.replace(step, longest_run=m), s, **kw) for m, s in zip((step.longest_run, 0), states)]
    assert torch.equal(outs[0], outs[1]) and torch.equal(states[0], states[1])


@pytest.mark.parametrize("heads,dv,columns", [(8, 16, 1), (8, 320, 1), (24, 320, 2)])   # state columns per thread
def test_a_run_without_tokens_leaves_the_state_it_started_from(heads, dv, columns):
    """Zeros where it starts at position 0, whatever an earlier owner of the slot left; as in the walk in one kernel."""
    from lite_llama_amd.kernels.recurrent import linear_scan

    runs, dk = [(0, 30), (0, 0), (7, 0), (3, 24)], 64
    n = sum(c for _, c in runs)
    assert (-(-n // 30) * heads * -(-dv // 16) >= 768) == (columns == 2)
    q, k, v, kw = _inputs("fixed", heads, heads, dk, dv, n, torch.bfloat16, 5)
    step = _step([(i, f, c, 0) for i, (f, c) in enumerate(runs)], None)
    start = torch.randn(len(runs), heads, dk, dv, device=DEV)
    states = [start.clone(), start.clone()]
    outs = [linear_scan(q, k, v, heads, dk, dv, dataclasses.replace(step, longest_run=m), s, **kw) for m, s in zip((step.longest_run, 0), states)]
    for s in states:
        assert (s[1] == 0).all() and torch.equal(s[2], start[2]) and not torch.equal(s[0], start[0])
    assert torch.equal(outs[0], outs[1]) and torch.equal(states[0], states[1])


@pytest.mark.parametrize("kind,heads,qk_heads,dk,dv", [("fixed", 5, 5, 64, 68), ("entry", 4, 4, 24, 40), ("token", 64, 2, 136, 4)])
def test_decoded_tokens_are_bit_equal_in_either_workgroup(kind, heads, qk_heads, dk, dv):
    from lite_llama_amd.kernels.recurrent import linear_scan

    for batch in (1, 40):   # 16-column and 64-column workgroups; the walk where the longest run is not known
        q, k, v, kw = _inputs(kind, heads, qk_heads, dk, dv, batch, torch.bfloat16, batch)
        step = _step([(i, i % 3, 1, 0) for i in range(batch)], None)
        start = torch.randn(batch, heads, dk, dv, device=DEV)
        states = [start.clone(), start.clone()]
        outs = [linear_scan(q, k, v, heads, dk, dv, dataclasses.replace(step, longest_run=m), s, **kw) for m, s in zip((1, 0), states)]
        assert torch.equal(outs[0], outs[1]) and torch.equal(states[0], states[1])
