"""Head norms, rotation and cache scatter in one launch: the bits of the launches they replace."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("tokens,heads,kv_heads", [(1, 1, 1), (37, 32, 4), (300, 7, 2), (65, 64, 32)])
@pytest.mark.parametrize("cs", [torch.float16, torch.float32])
@pytest.mark.parametrize("by_position", [False, True])
def test_head_norms_ride_in_the_rope_launch(dtype, tokens, heads, kv_heads, cs, by_position):
    from lite_llama_amd import kernels as K
    from lite_llama_amd.kernels.norm_act import norm_rope_and_cache_supported, rope_and_cache

    g = torch.Generator(device=DEV).manual_seed(tokens)
    rows = (torch.randn(tokens, (heads + 2 * kv_heads) * 128 + 8, generator=g, device=DEV) * 3).to(dtype)   # (a wider, strided projection)
    view = lambda r: (r[:, :heads * 128].view(tokens, heads, 128),  # noqa: E731
                      r[:, heads * 128:(heads + 2 * kv_heads) * 128].view(tokens, 2 * kv_heads, 128))
    weights = [torch.randn(128, generator=g, device=DEV).to(dtype) for _ in range(2)]
    pool = torch.zeros(2, tokens + 5, 2 * kv_heads, 128, dtype=dtype, device=DEV)
    select = torch.randperm(tokens + 5, generator=g, device=DEV)[:tokens].int()
    table = torch.rand(2, 1, tokens + 9, 128, generator=g, device=DEV).to(cs)
    positions = torch.randint(0, tokens + 9, (tokens,), generator=g, device=DEV) if by_position else None
    cos, sin = (table[0, 0], table[1, 0]) if by_position else (table[0, :, :tokens], table[1, :, :tokens])
    one, two = rows.clone(), rows.clone()
    q, kv = view(one)
    assert norm_rope_and_cache_supported(q, kv, pool[0], *weights)
    rope_and_cache(q, kv, cos, sin, 1, tokens, select, pool[0], positions=positions, qk_norm=(*weights, 1e-6))
    q2, kv2 = view(two)
    q2.copy_(K.skip_rmsnorm(q2, None, weights[0], 1e-6)[0])
    kv2[:, :kv_heads].copy_(K.skip_rmsnorm(kv2[:, :kv_heads], None, weights[1], 1e-6)[0])
    rope_and_cache(q2, kv2, cos, sin, 1, tokens, select, pool[1], positions=positions)
    assert torch.equal(one, two) and torch.equal(pool[0], pool[1])


def test_other_heads_keep_their_own_launches():
    from lite_llama_amd.kernels.norm_act import norm_rope_and_cache_supported, rope_and_cache

    q, kv, pool = (torch.zeros(4, h, 64, dtype=torch.float16, device=DEV) for h in (2, 4, 4))
    w = torch.ones(64, dtype=torch.float16, device=DEV)
    assert not norm_rope_and_cache_supported(q, kv, pool, w, w)
    with pytest.raises(ValueError):
        rope_and_cache(q, kv, pool[:1], pool[:1], 1, 4, torch.arange(4, device=DEV), pool, qk_norm=(w, w, 1e-6))
