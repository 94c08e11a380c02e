"""The router in one launch and the two-launch form of many experts (csrc/moe_sparse.hip) against 64-bit scores: one token and one past a workgroup's
tokens, experts off the waves' shares and past one and two per lane, widths off the pieces, every scoring."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, F64 = "cuda", torch.float64


@pytest.mark.parametrize("n,width,experts", [(1, 40, 5), (3, 2048, 34), (256, 136, 40), (257, 72, 41), (33, 3080, 65), (9, 100, 130), (600, 264, 68),
                                             (5, 520, 511), (7, 520, 513)])
@pytest.mark.parametrize("scoring", ["sigmoid", "softmax_chosen", "softmax_all", "sigmoid_plain", "softmax_groups"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_choice(n, width, experts, scoring, dtype):
    from lite_llama_amd.kernels.fused_moe import group_router

    g = torch.Generator(device=DEV).manual_seed(n + width + experts)
    top, route_scale, identity = min(4, experts), 1.5, 1
    h = torch.randn(n, width, generator=g, device=DEV).to(dtype)
    w = (torch.randn(experts, width, generator=g, device=DEV) * 2 * width ** -0.5).to(dtype)
    z = h.to(F64) @ w.to(F64).T
    kw, extra = {"scoring": scoring}, None
    if scoring == "softmax_all":
        kw.update(correction=(torch.randn(experts, generator=g, device=DEV) * 0.02).to(dtype), identity=identity)
    else:
        extra = torch.randn(width, generator=g, device=DEV).to(dtype) * width ** -0.5
        kw.update(extra_weight=extra)
    ids, weights, own = group_router(h, w, top, route_scale=route_scale, **kw)
    score = z if scoring == "softmax_chosen" else torch.sigmoid(z) if scoring.startswith("sigmoid") else torch.softmax(z, -1)
    rank = score + kw["correction"].to(F64) if scoring == "softmax_all" else score
    best, want = rank.topk(min(top + 1, experts), -1)
    # logits are fp32 sums of up to 3080 products of unit deviation (about 1e-6 off); a softmax's scores are off by that share of
    # themselves, the correction's sum by an fp32 unit: scores closer than ten times as much may change places
    close = 1e-5 * (best[:, :1].abs() if scoring.startswith("softmax_") and scoring != "softmax_chosen" else 1.0) + 1e-7
    clear = (best[:, :-1] - best[:, 1:] > close).all(-1)
    assert clear.float().mean() > 0.8
    want = want[:, :top]
    assert torch.equal(ids[clear].long(), want[clear])
    chosen = score.gather(1, want)
    weight = {"sigmoid": chosen / chosen.sum(-1, keepdim=True), "softmax_chosen": torch.softmax(chosen, -1), "softmax_all": chosen,
              "sigmoid_plain": chosen, "softmax_groups": chosen / chosen.sum(-1, keepdim=True)}[scoring] * route_scale
    assert (weights[clear].to(F64) - weight[clear]).abs().max() <= 2e-5
    if extra is not None:
        assert (own.to(F64) - torch.sigmoid(h.to(F64) @ extra.to(F64))).abs().max() <= 2e-5
    else:
        mine = torch.where(want >= experts - identity, chosen, torch.zeros_like(chosen)).sum(-1) * route_scale
        assert (own[clear].to(F64) - mine[clear]).abs().max() <= 2e-5


@pytest.mark.parametrize("scoring", ["sigmoid", "softmax_chosen", "softmax_all", "sigmoid_plain", "softmax_groups"])
@pytest.mark.parametrize("experts,top", [(4096, 64), (513, 4)])
def test_the_largest_choices(scoring, experts, top):
    """As many experts, groups of one and slots as are accepted: their tables are as large as a launch's LDS allows."""
    from lite_llama_amd.kernels.fused_moe import group_router

    g = torch.Generator(device=DEV).manual_seed(experts)
    h = torch.randn(3, 64, generator=g, device=DEV)
    w = torch.randn(experts, 64, generator=g, device=DEV) * 0.25
    groups = 1 if scoring in ("softmax_chosen", "softmax_all") else experts
    ids, weights, own = group_router(h, w, top, groups, groups, scoring=scoring, **({"identity": 1000 if experts > 1000 else 5} if scoring == "softmax_all" else {}))
    z = h.to(F64) @ w.to(F64).T
    score = z if scoring == "softmax_chosen" else torch.sigmoid(z) if scoring.startswith("sigmoid") else torch.softmax(z, -1)
    best, want = z.topk(top, -1)                 # (every score rises with its logit)
    clear = (z.topk(top + 1, -1).values.diff(dim=-1).abs() > 1e-5).all(-1)
    assert clear.any() and torch.equal(ids[clear].long(), want[clear])
    chosen = score.gather(1, want)
    weight = {"softmax_chosen": torch.softmax(best, -1), "softmax_all": chosen, "sigmoid_plain": chosen}.get(scoring, chosen / chosen.sum(-1, keepdim=True))
    assert (weights[clear].to(F64) - weight[clear]).abs().max() <= 2e-5
    if scoring == "softmax_all":
        mine = torch.where(want >= experts - (1000 if experts > 1000 else 5), chosen, torch.zeros_like(chosen)).sum(-1)
        assert (own[clear].to(F64) - mine[clear]).abs().max() <= 2e-5


@pytest.mark.parametrize("n,width,experts,top", [(1, 40, 5, 1), (1, 3072, 68, 8), (4, 2048, 34, 4), (5, 520, 34, 4), (31, 136, 130, 3), (32, 3080, 65, 4),
                                                 (33, 264, 40, 4), (2, 520, 512, 9), (8, 72, 513, 2), (32, 64, 511, 64)])
@pytest.mark.parametrize("scoring", ["sigmoid", "softmax_chosen", "softmax_all", "sigmoid_plain", "softmax_groups"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_choices_sorted_for_the_products_are_those_of_two_calls(n, width, experts, top, scoring, dtype):
    """Bit for bit; slots in their order, every list's tail.  Up to 16 tokens every expert's workgroup makes the choices, beyond them a launch of its own."""
    _the_same_as_two_calls(n, width, experts, top, scoring, dtype)


# the waves of the one launch and the largest step that takes it; the end of the choice in registers; the LDS of a launch
@pytest.mark.parametrize("n,width,experts,top", [(9, 520, 34, 4), (16, 3072, 68, 8), (17, 3072, 68, 8), (16, 264, 64, 16), (3, 264, 64, 17), (16, 264, 128, 16),
                                                 (7, 264, 128, 17), (13, 264, 129, 16), (16, 64, 482, 8), (16, 64, 483, 8), (12, 64, 480, 12), (1, 64, 491, 8)])
@pytest.mark.parametrize("scoring", ["sigmoid", "softmax_chosen", "softmax_all", "sigmoid_plain", "softmax_groups"])
def test_choices_at_the_edges_of_the_one_launch_are_those_of_two_calls(n, width, experts, top, scoring):
    _the_same_as_two_calls(n, width, experts, top, scoring, torch.bfloat16)


@pytest.mark.parametrize("n,width,experts,top,groups,keep", [(1, 520, 64, 4, 8, 2), (9, 264, 32, 5, 4, 3), (16, 264, 256, 8, 8, 4), (17, 264, 64, 4, 8, 2)])
@pytest.mark.parametrize("scoring", ["sigmoid", "softmax_groups"])
def test_choices_from_groups_sorted_for_the_products_are_those_of_two_calls(n, width, experts, top, groups, keep, scoring):
    _the_same_as_two_calls(n, width, experts, top, scoring, torch.bfloat16, group_count=groups, group_keep=keep)


def _the_same_as_two_calls(n, width, experts, top, scoring, dtype, **kw):
    from lite_llama_amd.kernels.fused_moe import _sort_slots, group_router

    g = torch.Generator(device=DEV).manual_seed(n + width + experts)
    h = torch.randn(n, width + 8, generator=g, device=DEV).to(dtype)[:, :width]
    w = (torch.randn(experts, width, generator=g, device=DEV) * 2 * width ** -0.5).to(dtype)
    identity = 2 if scoring == "softmax_all" and experts > 5 else 0
    served = experts - identity
    kw.update(scoring=scoring, route_scale=1.25)
    if scoring == "softmax_all":
        kw.update(correction=(torch.randn(experts, generator=g, device=DEV) * 0.02).to(dtype), identity=identity)
    elif n % 2:
        kw.update(extra_weight=(torch.randn(width, generator=g, device=DEV) * width ** -0.5).to(dtype))
    ids, weights, extra = group_router(h, w, top, **kw)
    block, srt, owner, post = _sort_slots(ids, n * top, served, width, 24, dtype, identity > 0)
    got = group_router(h, w, top, sort_for=torch.empty(served, width, 24, dtype=dtype, device=DEV), skipped=identity > 0, **kw)
    assert torch.equal(got[0], ids) and torch.equal(got[1], weights)
    assert (extra is None and got[2] is None) or torch.equal(got[2], extra)
    used = int(post)
    assert got[3][0] == block and int(got[3][3]) == used
    assert torch.equal(got[3][1][:used], srt[:used]) and torch.equal(got[3][2][:used // block], owner[:used // block])


@pytest.mark.parametrize("scoring", range(5))
def test_an_extra_scale_that_nothing_makes_is_left(scoring):
    """The C entry with ``extra_scale`` and no row of weights for it: as the entry without the sort leaves it (softmax_all writes the identity
    experts' sum, none here)."""
    from lite_llama_amd import _lib as L

    n, width, experts, top, block = 5, 64, 12, 3, 128
    h, w = (torch.randn(r, width, device=DEV).to(torch.bfloat16) for r in (n, experts))
    i32, f32 = (lambda *s: torch.zeros(*s, dtype=torch.int32, device=DEV)), (lambda *s: torch.zeros(*s, device=DEV))
    runs = n * top + experts * (block - 1)
    out = []
    for name in ("ll_group_router", "ll_group_router_sorted"):
        ids, weights, extra, logits = i32(n, top), f32(n, top), f32(n) + 7.0, f32(n, experts)
        args = (h.data_ptr(), width, w.data_ptr(), 0, n, width, experts, top, 1, 1, 1.0, scoring, ids.data_ptr(), weights.data_ptr(), extra.data_ptr(),
                logits.data_ptr(), 0, 0)
        lists = [i32(experts), i32(runs), i32(-(-runs // block)), i32(1)]
        sort = (experts, block, 0, *(t.data_ptr() for t in lists)) if name.endswith("sorted") else ()
        L.check(getattr(L.lib(), name)(*args, *sort, L.LL_BF16, L.stream_ptr()), name)
        out.append((ids, weights, extra))
    assert all(torch.equal(a, b) for a, b in zip(*out))
    assert (out[1][2] == (0.0 if scoring == 2 else 7.0)).all()
