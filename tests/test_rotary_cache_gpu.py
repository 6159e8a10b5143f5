"""Rotation and cache write in one launch against the two of their own: the same bits."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens", [1, 2, 33, 300])
@pytest.mark.parametrize(("heads", "kv_heads", "dim"), [(32, 8, 128), (32, 8, 64), (3, 1, 48),
                                                        (4, 4, 256)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.uint8])
@pytest.mark.parametrize("sliced", [True, False])
def test_same_as_apart(tokens, heads, kv_heads, dim, dtype, sliced):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from vllm_tgis_adapter_amd import ops

    gen = torch.Generator("cuda").manual_seed(tokens + dim)
    sizes = [heads * dim, kv_heads * dim, kv_heads * dim]
    qkv = torch.randn((tokens, sum(sizes)), generator=gen, device="cuda").bfloat16()
    parts = qkv.split(sizes, dim=-1)
    if not sliced:
        parts = [p.contiguous() for p in parts]
    angle = torch.rand((500, dim // 2), generator=gen, device="cuda") * 6.3
    cos_sin = torch.cat([angle.cos(), angle.sin()], dim=1).contiguous()
    positions = torch.randint(0, 500, (tokens,), generator=gen, device="cuda")
    slots = torch.randperm(320, generator=gen, device="cuda")[:tokens]
    slots[tokens // 2] = -1          # a row of padding

    def cache():
        return [torch.full((20, 16, kv_heads, dim), 3, dtype=dtype, device="cuda") for _ in "kv"]

    kc, vc = cache()
    got = ops.rotary_and_cache(positions, *[p.clone() if not sliced else p for p in parts], dim,
                               cos_sin, kc, vc, slots)
    q, k, v = [p.clone() for p in parts]
    want_k, want_v = cache()
    q, k = ops.rotary_embedding(positions, q, k, dim, cos_sin)
    ops.reshape_and_cache(k.view(tokens, kv_heads, dim), v.view(tokens, kv_heads, dim), want_k,
                          want_v, slots)
    assert got.is_contiguous() and torch.equal(got, q)
    assert torch.equal(kc, want_k) and torch.equal(vc, want_v)
