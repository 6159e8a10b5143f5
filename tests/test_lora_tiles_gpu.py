"""Multi-LoRA products in bf16 (lora_bgmv.hip) against float64: edges of the 16-token
tiles and of the 256 columns of a workgroup, every padded rank, K of a single tile, of a
quarter of one and cut over workgroups, tokens and adapters without a partner."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

TOKENS = [1, 2, 15, 16, 17, 61, 64, 65, 257, 300]
# rank, K, widths of the projections, columns before and after each
SHAPES = [
    (8, 8, [1], 0), (8, 40, [256, 8], 3), (16, 4096, [4096, 1024, 1024], 0),
    (32, 1024, [257, 255, 1], 16), (64, 264, [300], 16), (64, 2048, [512, 512, 40], 1),
    (16, 14336, [264], 0), (32, 512, [64, 64], 0),
]


def _need():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


@pytest.mark.parametrize("t", TOKENS)
@pytest.mark.parametrize(("rank", "k", "widths", "gap"), SHAPES)
def test_delta(t, rank, k, widths, gap):
    _need()
    from vllm_tgis_adapter_amd import ops

    gen = torch.Generator("cpu").manual_seed(t * 131 + k)
    adapters, p = 5, len(widths)
    spans, at = [], gap
    for w in widths:
        spans.append((at, at + w))
        at += w + gap
    a = torch.randn(adapters, p * rank, k, generator=gen).bfloat16()
    b = torch.randn(adapters, sum(widths), rank, generator=gen).bfloat16()
    x = torch.randn(t, k, generator=gen).bfloat16()
    base = torch.randn(t, at, generator=gen).bfloat16()
    # runs of one adapter, single tokens, none; the last adapter has no token
    slots = torch.randint(-1, adapters - 1, (t,), generator=gen, dtype=torch.int32)
    slots[t // 3: 2 * t // 3] = 1
    scales = torch.linspace(0.5, 2.0, adapters)
    got = base.cuda()
    ops.lora_delta(got, x.cuda(), a.cuda(), b.cuda(), slots.cuda(), scales.cuda(), spans)
    want, terms = base.double(), base.double().abs()
    for i, s in enumerate(slots.tolist()):
        v = 0
        for j, (lo, hi) in enumerate(spans):
            if s >= 0:
                aa, bb = a[s, j * rank:(j + 1) * rank].double(), b[s, v: v + hi - lo].double()
                scale = scales[s].double()
                want[i, lo:hi] += scale * (bb @ (aa @ x[i].double()))
                terms[i, lo:hi] += scale * (bb.abs() @ (aa.abs() @ x[i].double().abs()))
            v += hi - lo
    # one rounding to bf16, and float32 sums: 2**-20 of the size of their terms
    err = (got.cpu().double() - want).abs()
    assert (err <= 2 ** -8 * want.abs() + 2 ** -20 * terms).all(), err.max().item()
    still = torch.ones(t, at, dtype=torch.bool)
    for lo, hi in spans:
        still[slots >= 0, lo:hi] = False
    assert torch.equal(got.cpu()[still], base[still])


@pytest.mark.parametrize("t", [0, 1, 255, 256, 257])
def test_slots(t):
    _need()
    from vllm_tgis_adapter_amd import ops

    ids = (3, 7, 8, 40)
    tokens = torch.randint(0, 45, (t,), generator=torch.Generator().manual_seed(t),
                           dtype=torch.int32)
    want = [ids.index(i) if i in ids else -1 for i in tokens.tolist()]
    got = ops.lora_slots(tokens.cuda(), ids)
    assert got.dtype == torch.int32 and got.tolist() == want
    assert ops.lora_slots(tokens.cuda(), ()).tolist() == [-1] * t
