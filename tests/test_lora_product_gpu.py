"""Products made together with their LoRA deltas and their gate (lora_bgmv.hip), against
float64: from weights, with and without parts of K, and from a product that is given; every
padded rank, tokens and columns without an adapter, edges of the 256 columns of a workgroup."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


# tokens, K, columns, spans of the projections
SHAPES = [
    (1, 64, 128, [(0, 128)]), (17, 8192, 768, [(0, 512), (512, 640), (640, 768)]),
    (61, 4096, 4096, [(0, 4096)]), (61, 256, 512, [(0, 256), (256, 512)]),
    (64, 4096, 1792, [(128, 300), (1700, 1792)]), (300, 1024, 512, [(256, 512)]),
    (2050, 128, 2304, [(0, 1152), (1152, 2304)]),
]


@pytest.mark.parametrize(("t", "k", "width", "spans"), SHAPES)
@pytest.mark.parametrize("rank", [8, 16, 32, 64])
@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("given", [False, True])
def test_product(t, k, width, spans, rank, gated, given):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from vllm_tgis_adapter_amd.ops import _C

    g = torch.Generator("cuda").manual_seed(t + k + rank)

    def normal(*shape, by=1.0):
        return (torch.randn(shape, generator=g, device="cuda") * by).bfloat16()

    adapters, cols = 5, sum(hi - lo for lo, hi in spans)
    x, w = normal(t, k), normal(width, k, by=k ** -0.5)
    a, b = normal(adapters, len(spans) * rank, k, by=k ** -0.5), normal(adapters, cols, rank)
    slots = torch.randint(-1, adapters - 1, (t,), generator=g, device="cuda").int()
    slots[t // 3: 2 * t // 3] = 1
    scales = torch.linspace(0.5, 2.0, adapters, device="cuda")
    out = torch.full((t, width // 2 if gated else width), float("nan"), device="cuda").bfloat16()
    y = (x.double() @ w.double().t()).bfloat16() if given else None
    _C.lora_product(out, x, None if given else w, y, a, b, slots, scales, spans, gated)

    want = y.double() if given else x.double() @ w.double().t()
    # a product that is one part is rounded to bf16 before its deltas
    off = torch.zeros_like(want) if given else 2 ** -8 * want.abs() + 2 ** -20 * (
        x.double().abs() @ w.double().abs().t())
    for s in range(adapters):
        rows, v = (slots == s).nonzero().view(-1), 0
        for p, (lo, hi) in enumerate(spans):
            aa, bb = a[s, p * rank:(p + 1) * rank].double(), b[s, v:v + hi - lo].double()
            xr, scale = x[rows].double(), scales[s].double()
            want[rows, lo:hi] += scale * (xr @ aa.t()) @ bb.t()
            off[rows, lo:hi] += 2 ** -20 * scale * (xr.abs() @ aa.abs().t()) @ bb.abs().t()
            v += hi - lo
    if gated:
        (gate, up), (og, ou) = want.chunk(2, 1), off.chunk(2, 1)
        want = torch.nn.functional.silu(gate) * up
        # silu' is at most 1.1; exp and the division in float32
        off = 1.1 * (og * (up.abs() + ou)) + ou * gate.abs() + 1e-5 * want.abs()
    err = (out.double() - want).abs()
    assert (err <= 2 ** -8 * want.abs() + off + 1e-7).all(), err.max().item()


# rows, adapters, K, rank: edges of the 16 tokens of a group and the 256 of a window, more adapters
# than rows, K that its parts do not divide; up to 256 workgroups go beside the product
@pytest.mark.parametrize(("t", "adapters", "k", "rank"), [
    (1, 40, 4096, 16), (15, 1, 4160, 8), (16, 16, 1024, 64), (17, 3, 14336, 32), (63, 60, 4096, 8),
    (64, 4, 64, 64), (255, 2, 2048, 64), (256, 1, 4096, 8), (257, 3, 1088, 16), (272, 30, 1024, 8),
    (513, 1, 4096, 32), (600, 2, 4096, 8), (600, 9, 4096, 64),
])
@pytest.mark.parametrize("some", [False, True])
def test_adapters_beside_the_product(t, adapters, k, rank, some):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from vllm_tgis_adapter_amd.ops import _C

    g = torch.Generator("cuda").manual_seed(t + k + rank)

    def normal(*shape, by=1.0):
        return (torch.randn(shape, generator=g, device="cuda") * by).bfloat16()

    width, spans = 384, [(0, 256), (256, 384)]
    x, w = normal(t, k), normal(width, k, by=k ** -0.5)
    a, b = normal(adapters, 2 * rank, k, by=k ** -0.5), normal(adapters, width, rank)
    slots = torch.randint(-1, adapters, (t,), generator=g, device="cuda").int()
    if not some:   # the last one alone, then a row without
        slots[:] = adapters - 1
        slots[t - 1] = -1
    scales = torch.linspace(0.5, 2.0, adapters, device="cuda")
    out = torch.full((t, width), float("nan"), device="cuda").bfloat16()
    _C.lora_product(out, x, w, None, a, b, slots, scales, spans, False)

    x, w, a, b = x.double(), w.double(), a.double(), b.double()
    want = x @ w.t()
    # a product of one part is rounded to bf16, sums are in float32
    off = 2 ** -8 * want.abs() + 2 ** -20 * (x.abs() @ w.abs().t())
    for s in slots.unique().tolist():
        rows = (slots == s).nonzero().view(-1)
        for p, (lo, hi) in enumerate(spans if s >= 0 else []):
            aa, bb, scale = a[s, p * rank:(p + 1) * rank], b[s, lo:hi], scales[s].double()
            want[rows, lo:hi] += scale * (x[rows] @ aa.t()) @ bb.t()
            off[rows, lo:hi] += 2 ** -20 * scale * (x[rows].abs() @ aa.abs().t()) @ bb.abs().t()
    err = (out.double() - want).abs()
    assert (err <= 2 ** -8 * want.abs() + off + 1e-7).all(), err.max().item()
