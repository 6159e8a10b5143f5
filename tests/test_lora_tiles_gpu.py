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


def _gpu_check(t, adapters, rank, k, widths, pick):
    """ops.lora_delta of random stacks against float64, tokens' slots as given."""
    from vllm_tgis_adapter_amd import ops

    g = torch.Generator("cuda").manual_seed(t + k + rank)

    def normal(*shape):
        return torch.randn(shape, generator=g, device="cuda").bfloat16()

    p, width = len(widths), sum(widths)
    ends = [sum(widths[:i]) for i in range(p + 1)]
    a, b, x, base = (normal(adapters, p * rank, k), normal(adapters, width, rank), normal(t, k),
                     normal(t, width))
    scales = torch.linspace(0.5, 2.0, adapters, device="cuda")
    got = base.clone()
    ops.lora_delta(got, x, a, b, pick, scales, list(zip(ends, ends[1:])))
    want, terms = base.double(), base.double().abs()
    for s in range(adapters):
        rows = (pick == s).nonzero().view(-1)
        xs = x[rows].double()
        for j in range(p):
            at = slice(ends[j], ends[j + 1])
            aa, bb = a[s, j * rank:(j + 1) * rank].double().t(), b[s, at].double().t()
            want[rows, at] += scales[s].double() * ((xs @ aa) @ bb)
            terms[rows, at] += scales[s].double() * ((xs.abs() @ aa.abs()) @ bb.abs())
    # one rounding to bf16, and float32 sums: 2**-20 of the size of their terms
    err = (got.double() - want).abs()
    assert (err <= 2 ** -8 * want.abs() + 2 ** -20 * terms).all(), err.max().item()
    assert torch.equal(got[pick < 0], base[pick < 0])


@pytest.mark.parametrize("rank", [8, 16, 32, 64])
# columns in tiles of 256 times tokens on both sides of the lines at 2560, 8192 and 98304
# that choose the tokens of a workgroup, the last one with a few
@pytest.mark.parametrize(("t", "widths"), [(51, [12800]), (61, [10752]), (301, [6912]),
                                           (301, [7168, 1]), (877, [14336, 14336]),
                                           (1037, [14336, 14336])])
def test_tokens_of_a_workgroup(rank, t, widths):
    _need()
    # runs, neighbours with different adapters, neighbours that take turns, none
    pick = torch.randint(-1, 4, (t,), generator=torch.Generator().manual_seed(t),
                         dtype=torch.int32)
    pick[t // 4: t // 2] = 2
    pick[t // 2: t // 2 + 20] = torch.arange(20, dtype=torch.int32) % 2
    pick[t // 2 + 20: t // 2 + 40] = -1
    _gpu_check(t, 4, rank, 64, widths, pick.cuda())


@pytest.mark.parametrize("t", [16, 255, 256, 257, 500, 513])
@pytest.mark.parametrize("rank", [8, 64])
def test_many_adapters(rank, t):
    """Groups of 16 tokens of one adapter in windows of 256: none, one and several of them,
    with one token and with all."""
    _need()
    g = torch.Generator().manual_seed(t)
    pick = torch.randint(-1, 33, (t,), generator=g, dtype=torch.int32)
    _gpu_check(t, 33, rank, 264, [300], pick.cuda())
    pick[torch.randperm(t, generator=g)[: t // 2]] = 5
    _gpu_check(t, 33, rank, 264, [300], pick.cuda())
    _gpu_check(t, 33, rank, 264, [300], torch.full((t,), 32, dtype=torch.int32).cuda())


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
