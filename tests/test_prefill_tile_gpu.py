"""Prompt attention over the paged cache (attention_prefill_tile.hip) against float64:
edges of the 32-row waves, of the workgroup's tokens and of the 64-key tiles, every split
of the waves into heads and tokens, prompts that earlier steps have begun."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

# heads, key heads: 8, 4, 2 heads of a group in a workgroup, one of three, one of one
HEADS = [(16, 2), (8, 2), (12, 2), (3, 1), (2, 2)]
# new tokens and those of earlier steps
SHAPES = [
    [(1, 0)], [(1, 63), (2, 64), (31, 1)], [(32, 0), (33, 31), (64, 64)],
    [(63, 65), (65, 127)], [(128, 0), (129, 700)], [(255, 3), (256, 0), (257, 64)],
    [(300, 1000), (7, 2049), (40, 0)], [(1100, 0)],
]


def _need():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


@pytest.mark.parametrize("shape", SHAPES, ids=str)
@pytest.mark.parametrize(("heads", "kv_heads"), HEADS)
@pytest.mark.parametrize(("dim", "dtype", "block"), [
    (128, torch.bfloat16, 16), (64, torch.bfloat16, 16), (128, torch.uint8, 16),
    (128, torch.bfloat16, 12), (64, torch.bfloat16, 1)])
def test_prefill(shape, heads, kv_heads, dim, dtype, block):
    _need()
    from vllm_tgis_adapter_amd import ops

    gen = torch.Generator("cuda").manual_seed(heads * 17 + dim + len(shape))
    new = [n for n, _ in shape]
    lens = [n + past for n, past in shape]
    need = [-(-n // block) for n in lens]
    ids = torch.randperm(sum(need), generator=torch.Generator().manual_seed(3)).tolist()
    tables, at = [], 0
    for n in need:
        tables.append(ids[at:at + n])
        at += n
    cache = [torch.randn((at + 1, block, kv_heads, dim), generator=gen, device="cuda")
             for _ in "kv"]
    if dtype == torch.uint8:
        cache = [c.to(torch.float8_e4m3fn) for c in cache]
        kc, vc = (c.view(torch.uint8) for c in cache)
    else:
        kc, vc = cache = [c.bfloat16() for c in cache]
    # what no sequence owns must not be looked at
    q = torch.randn((sum(new) + 2, heads, dim), generator=gen, device="cuda").bfloat16()
    start = [0]
    for n in new:
        start.append(start[-1] + n)

    def ints(v):
        return torch.tensor(v, dtype=torch.int32, device="cuda")

    scale = 1.3 * dim ** -0.5
    got = ops.paged_attention_prefill(
        q, kc, vc, ints([t + [0] * (max(need) - len(t)) for t in tables]), ints(start),
        ints(lens), scale, max(new), max(lens))
    for i, (n, past) in enumerate(shape):
        rows = slice(start[i], start[i] + n)
        k, v = (c[ints(tables[i]).long()].double().reshape(-1, kv_heads, dim)[:lens[i]]
                .repeat_interleave(heads // kv_heads, 1).transpose(0, 1).contiguous()
                for c in cache)
        s = q[rows].double().transpose(0, 1).contiguous() @ k.transpose(1, 2).contiguous() * scale
        pos = torch.arange(lens[i], device="cuda")
        s = s.masked_fill(pos[None, :] > pos[past:past + n, None], float("-inf"))
        p = s.softmax(-1)
        want = (p @ v).transpose(0, 1)
        terms = (p @ v.abs()).transpose(0, 1)
        # probabilities and the result are rounded to bf16 once each, which is off by half a
        # unit in the last of 8 bits: by 2**-8 of the value just above a power of two
        err = (got[rows].double() - want).abs()
        assert (err <= 1.01 * 2 ** -7 * terms + 1e-6).all(), (i, err.max().item())
