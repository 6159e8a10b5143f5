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
    _beside_the_product(t, adapters, k, rank, some, 384, [(0, 256), (256, 384)])


# every form of tile, weights that stay in the caches and that go past them, K whole and in parts
@pytest.mark.parametrize(("t", "width", "k", "form", "parts"), [
    (61, 28672, 4096, 4, 1), (9, 5120, 4096, 4, 3), (61, 1408, 28672, 3, 8), (65, 15360, 512, 3, 1),
    (129, 2688, 8192, 3, 4), (120, 28672, 4096, 2, 1), (65, 5120, 8192, 2, 6),
    (129, 11264, 2048, 2, 1), (200, 2816, 14336, 2, 5)])
def test_adapters_beside_every_form_of_product(t, width, k, form, parts):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from vllm_tgis_adapter_amd.ops import _C

    plan = _C.gemm_ring_plan(t, width, k, False)
    assert plan == form << 4 | parts and _C.gemm_ring_lora_cuts(t, k, 3, 32, plan) > 0
    _beside_the_product(t, 3, k, 16, True, width, [(0, 256), (256, width)])


# sizes at which the tiles take a product for its adapters' sake only
@pytest.mark.parametrize(("t", "width", "k"), [
    (1, 2048, 2048), (2, 28672, 4096), (8, 384, 64), (16, 6144, 4096), (17, 768, 768),
    (64, 2048, 2048), (65, 16384, 2048), (128, 28672, 4096), (256, 3072, 2048), (320, 4096, 4096),
    (512, 1536, 4096)])
@pytest.mark.parametrize("rank", [8, 64])
def test_products_that_adapters_bring(t, width, k, rank):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from vllm_tgis_adapter_amd import ops

    assert ops._lora_tiles_take(t, width, k) and not ops._tiles_take(t, width, k)
    _beside_the_product(t, 3, k, rank, True, width, [(0, 256), (256, width)])


def _beside_the_product(t, adapters, k, rank, some, width, spans):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from vllm_tgis_adapter_amd.ops import _C

    g = torch.Generator("cuda").manual_seed(t + k + rank)

    def normal(*shape, by=1.0):
        return (torch.randn(shape, generator=g, device="cuda") * by).bfloat16()

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


# deltas by the matrix unit: spans off its 32 columns, columns without an adapter, ragged windows
TILES = [(257, 64, 2048, [(3, 700), (701, 2043)], 5, 64), (1000, 128, 5792, [(0, 5792)], 1, 8),
         (520, 64, 4800, [(1000, 1033), (1050, 2400), (2600, 4800)], 9, 32),
         (450, 64, 5376, [(0, 2688), (2688, 5376)], 3, 16), (130, 2048, 8192, [(0, 8192)], 2, 32),
         (900, 64, 2064, [(0, 2064)], 2, 32)]   # (half a tile of columns: a column a thread)


@pytest.mark.parametrize(("t", "k", "width", "spans", "adapters", "rank"), TILES)
@pytest.mark.parametrize("way", ["product", "gated", "in place"])
def test_deltas_by_the_matrix_unit(t, k, width, spans, adapters, rank, way):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from vllm_tgis_adapter_amd.ops import _C

    g = torch.Generator("cuda").manual_seed(t + rank)

    def normal(*shape, by=1.0):
        return (torch.randn(shape, generator=g, device="cuda") * by).bfloat16()

    cols = sum(hi - lo for lo, hi in spans)
    assert _C.lora_tiles_win(t, adapters, rank, cols)   # (the gate of rank 64: a column a thread)
    x, y = normal(t, k), normal(t, width)
    a, b = normal(adapters, len(spans) * rank, k, by=k ** -0.5), normal(adapters, cols, rank)
    # tokens 0 and 1, alone in rank 0: a sum past float32 and one just inside it
    x[:2], a[:, :, 0] = 0, 0
    x[0, 0], x[1, 0] = 3e38, 3e38
    a[:, ::rank, 0] = 1.0625
    a[0, ::rank, 0] = 16
    slots = torch.randint(-1, adapters, (t,), generator=g, device="cuda").int()
    slots[0], slots[1] = 0, adapters - 1
    scales = torch.linspace(0.5, 1.0, adapters, device="cuda")
    scales[0] = 0.5
    if way == "in place":
        out = y.clone()
        _C.lora_delta(out, x, a, b, slots, scales, spans)
    else:
        out = torch.full((t, width // (1 + (way == "gated"))), float("nan"), device="cuda").bfloat16()
        _C.lora_product(out, x, None, y, a, b, slots, scales, spans, way == "gated")

    want = y.double()
    off = torch.zeros_like(want)
    for s in range(adapters):
        rows, v = (slots == s).nonzero().view(-1), 0
        for p, (lo, hi) in enumerate(spans):
            aa, bb = a[s, p * rank:(p + 1) * rank].double(), b[s, v:v + hi - lo].double()
            xr, scale = x[rows].double(), scales[s].double()
            want[rows, lo:hi] += scale * (xr @ aa.t()) @ bb.t()
            off[rows, lo:hi] += 2 ** -20 * scale * (xr.abs() @ aa.abs().t()) @ bb.abs().t()
            v += hi - lo
    # 16 * 3e38 is infinite in float32, whatever B makes of it
    past = torch.zeros_like(want, dtype=torch.bool)
    for lo, hi in spans:
        past[0, lo:hi] = True
        if adapters == 1:
            past[1, lo:hi] = True
    if way == "gated":
        (gate, up), (og, ou) = want.chunk(2, 1), off.chunk(2, 1)
        want = torch.nn.functional.silu(gate) * up
        off = 1.1 * (og * (up.abs() + ou)) + ou * gate.abs() + 1e-5 * want.abs()
        p0, p1 = past.chunk(2, 1)
        past = p0 | p1
        past[:2] = True   # (products of two sums of that size)
        assert not out[2:].isnan().any()
    else:
        assert not out.isnan().any()
        assert (out.double()[past] == float("inf") * want[past].sign()).all()
    past |= want.abs() + off > 2.0 ** 127   # (rounded to what is infinite in bf16)
    err = (out.double() - want).abs()
    assert (err <= 2 ** -8 * want.abs() + off + 1e-7)[~past].all(), err[~past].max().item()


def test_infinite_adapters_by_the_matrix_unit():
    """An infinity in B times a sum is one, of the sum's sign, whatever terms the sum enters in."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from vllm_tgis_adapter_amd.ops import _C

    t, k, width, rank = 1000, 128, 5792, 8
    g = torch.Generator("cuda").manual_seed(4)
    x, a = (torch.randn(s, generator=g, device="cuda").bfloat16() for s in ((t, k), (1, rank, k)))
    b = torch.randn((1, width, rank), generator=g, device="cuda").bfloat16()
    # sums that are 0, that bf16 holds, one that is infinite itself
    x[:3] = 0
    x[1, 3], x[2, 5], a[0, :, 5], a[0, 2, 5] = 1, 3e38, 0.25, 4
    b[0, 7, 2], b[0, 40, 5], b[0, 41, 0] = float("inf"), -float("inf"), float("nan")
    b[0, 40, 2] = -1
    slots = torch.zeros(t, dtype=torch.int32, device="cuda")
    assert _C.lora_tiles_win(t, 1, rank, width)
    out = torch.zeros((t, width), device="cuda").bfloat16()
    _C.lora_delta(out, x, a, b, slots, torch.ones(1, device="cuda"), [(0, width)])
    s = x.double() @ a[0].double().t()
    assert (s[1:, [2, 5]].abs() > 1e-3).all()   # (no sum of float32 is of another sign)
    assert torch.equal(out[1:, 7].double(), float("inf") * s[1:, 2].sign())
    assert torch.equal(out[1:, 40].double(), -float("inf") * s[1:, 5].sign())
    assert out[0, [7, 40]].isnan().all() and out[:, 41].isnan().all()
    rest = [v for v in range(width) if v not in (7, 40, 41)]
    assert out[:2, rest].isfinite().all() and out[3:, rest].isfinite().all()


def test_many_adapters_of_few_tokens_take_a_column_a_thread():
    """Groups of 16 tokens are mostly empty there, and each looks through all adapters."""
    from vllm_tgis_adapter_amd.ops import _C

    if _C is None:
        pytest.skip("the extension is not built")
    for t, adapters, rank, width in [(200, 60, 32, 6144), (599, 60, 32, 2048), (150, 60, 64, 4096),
                                     (1197, 32, 16, 2048), (300, 32, 32, 4096), (291, 16, 16, 6144)]:
        assert not _C.lora_tiles_win(t, adapters, rank, width)
        assert _C.lora_tiles_win(t, 1, rank, 4 * width)
