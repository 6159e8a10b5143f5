"""Expert products and what surrounds them: every way the products are cut, empty and
uneven segments, rows through a list, against float64 and the reference ops."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


def _segments(counts):
    seg = torch.zeros(len(counts) + 1, dtype=torch.int32)
    seg[1:] = torch.tensor(counts).cumsum(0)
    return seg


# rows per expert: one pair, means at and around each line of the rule (9, 18, 52, 250),
# empty experts, one expert with everything, more experts than lanes of a wave
COUNTS = [
    [0, 1, 0], [9, 9], [16, 1, 0, 17, 11], [18, 20, 16], [19, 19, 40, 0], [52, 52], [53, 130, 0],
    [64, 65, 127, 1], [249, 250], [250, 250], [300, 1, 513, 256], [0, 0, 700],
    [3] * 70, [0] * 65 + [40, 0, 2],
]


@pytest.mark.parametrize("mode", ["plain", "silu", "relu2", "clamped"])
@pytest.mark.parametrize("counts", COUNTS, ids=str)
@pytest.mark.parametrize(("n", "k"), [(128, 64), (256, 320)])
@pytest.mark.parametrize("listed", [False, True])
def test_products(mode, counts, n, k, listed):
    from vllm_tgis_adapter_amd import ops

    g = torch.Generator("cuda").manual_seed(len(counts) + n)
    seg = _segments(counts)
    total, experts = int(seg[-1]), len(counts)
    gated = mode in ("silu", "clamped")
    w = torch.randn((experts, (2 if gated else 1) * n, k), generator=g,
                    device="cuda").bfloat16() / k ** 0.5
    rows = None
    if listed:
        x = torch.randn((max(total // 2, 1), k), generator=g, device="cuda").bfloat16()
        rows = torch.randint(len(x), (total,), generator=g, device="cuda", dtype=torch.int32)
        xs = x[rows.long()]
    else:
        x = xs = torch.randn((total, k), generator=g, device="cuda").bfloat16()
    act = {"relu2": "relu2", "clamped": "clamped"}.get(mode)
    got = ops.moe_gemm(x, w, seg.cuda(), gated, act=act, limit=1.5, rows=rows)
    assert got.shape == (total, n)
    for e in range(experts):
        lo, hi = int(seg[e]), int(seg[e + 1])
        s = xs[lo:hi].double() @ w[e].double().t()
        if gated:
            a, u = s.chunk(2, dim=1)
            if mode == "clamped":
                a, u = a.clamp(max=1.5), u.clamp(-1.5, 1.5)
                s = a * torch.sigmoid(1.702 * a) * (u + 1)
            else:
                s = torch.nn.functional.silu(a) * u
        elif mode == "relu2":
            s = s.clamp(min=0).square()
        # one rounding to bf16; float32 sums of up to 320 terms and exp below 1e-5
        err = (got[lo:hi].double() - s).abs()
        assert (err <= 2 ** -8 * s.abs() + 1e-4).all(), (e, err.max().item())


@pytest.mark.parametrize("tokens", [1, 3, 4, 5, 33, 1030])
@pytest.mark.parametrize(("experts", "top", "k"), [(8, 2, 4096), (1, 1, 64), (9, 3, 200),
                                                   (64, 8, 512)])
def test_router_grouping_and_sum(tokens, experts, top, k):
    from vllm_tgis_adapter_amd import ops

    g = torch.Generator("cuda").manual_seed(tokens)
    x = torch.randn((tokens, k), generator=g, device="cuda").bfloat16()
    gate = torch.randn((experts, k), generator=g, device="cuda").bfloat16() / k ** 0.5
    ids, weights = ops.moe_topk(x, gate, top)
    logits = x.double() @ gate.double().t()
    assert (ids.sort(dim=1).values.diff(dim=1) > 0).all()       # no expert twice
    chosen = logits.gather(1, ids.long())
    # float32 sums: what was chosen is the largest up to their error
    assert (chosen - logits.topk(top, dim=1).values).abs().max() <= 1e-5 * k ** 0.5
    torch.testing.assert_close(weights.double(), chosen.softmax(dim=1), atol=1e-5, rtol=1e-4)

    rows, pos, seg = ops.moe_group(ids, experts)
    count = torch.bincount(ids.view(-1).long(), minlength=experts)
    assert torch.equal(seg[1:].long(), count.cumsum(0)) and seg[0] == 0
    flat = pos.view(-1).long()
    assert torch.equal(flat.sort().values, torch.arange(tokens * top, device="cuda"))
    assert torch.equal(rows[flat].long(),
                       torch.arange(tokens, device="cuda").repeat_interleave(top))
    e = ids.view(-1).long()
    assert (flat >= seg[e]).all() and (flat < seg[e + 1]).all()

    ye = torch.randn((tokens * top, 264), generator=g, device="cuda").bfloat16()
    got = ops.moe_sum(ye, pos, weights)
    want = (ye[pos.long()].double() * weights.double()[..., None]).sum(dim=1)
    assert ((got.double() - want).abs() <= 2 ** -8 * want.abs() + 1e-5).all()


def test_router_of_equal_and_undefined_scores_names_experts():
    from vllm_tgis_adapter_amd import ops

    gate = torch.ones((8, 64), device="cuda").bfloat16()
    x = torch.ones((3, 64), device="cuda").bfloat16()
    x[1, 0] = float("nan")
    x[2, 0] = float("inf")
    ids, weights = ops.moe_topk(x, gate, 2)
    assert ids.tolist() == [[0, 1]] * 3
    assert weights[0].tolist() == [0.5, 0.5] and weights[1].isnan().all()


@pytest.mark.parametrize("layout", ["dense", "slice", "turned", "odd offset", "odd gate"])
@pytest.mark.parametrize("rows", [1, 33, 700])
def test_mixture_of_rows_in_any_layout(layout, rows):
    """The whole block, for rows as callers may have them, against float64."""
    from vllm_tgis_adapter_amd.engine.config import ModelConfig
    from vllm_tgis_adapter_amd.models.mixtral import MoEBlock

    mc = ModelConfig(model="m", architecture="mixtral", vocab_size=64, hidden_size=256,
                     intermediate_size=384, num_layers=1, num_heads=2, num_kv_heads=1,
                     head_dim=128, max_model_len=64, dtype=torch.bfloat16, num_experts=8,
                     num_experts_per_tok=2)
    torch.manual_seed(rows)
    with torch.device("cuda"):
        block = MoEBlock(mc)
    for w in (block.gate, block.w13, block.w2):
        w.data.normal_(0, 0.06)
    x = torch.randn((rows, 256), device="cuda").bfloat16()
    if layout == "slice":
        given = torch.zeros((rows, 300), dtype=x.dtype, device="cuda")[:, 16:272]
    elif layout == "turned":
        given = torch.zeros((256, rows), dtype=x.dtype, device="cuda").t()
    elif layout == "odd offset":
        given = torch.zeros(rows * 256 + 1, dtype=x.dtype, device="cuda")[1:].view(rows, 256)
    else:
        given = x.clone()
    if layout == "odd gate":
        wide = torch.zeros((8, 257), dtype=x.dtype, device="cuda")
        wide[:, 1:] = block.gate.data
        block.gate.data = wide[:, 1:]
    given.copy_(x)
    with torch.inference_mode():
        got = block(given)
    logits = x.double() @ block.gate.double().t()
    score, pick = logits.topk(2, dim=1)
    # f32 router sums: only rows whose second and third scores they cannot swap
    third = logits.topk(3, dim=1).values[:, 2]
    clear = score[:, 1] - third > 1e-3
    score = score.softmax(1)
    want, terms = (torch.zeros((rows, 256), dtype=torch.float64, device="cuda") for _ in "wt")
    for j in range(2):
        for e in range(8):
            at = (pick[:, j] == e).nonzero().view(-1)
            a, u = (x[at].double() @ block.w13[e].double().t()).chunk(2, dim=1)
            h = torch.nn.functional.silu(a) * u
            want[at] += score[at, j, None] * (h @ block.w2[e].double().t())
            terms[at] += score[at, j, None] * (h.abs() @ block.w2[e].double().abs().t())
    # roundings to bf16 of h, of an expert's result and of the sum
    err = (got.double() - want).abs()[clear]
    assert (err <= 3 * 2 ** -8 * terms[clear] + 1e-4).all(), err.max().item()


def test_router_keeps_an_undefined_score():
    """One expert's score is NaN: so is every weight, as a softmax over all experts says."""
    from vllm_tgis_adapter_amd import ops

    g = torch.Generator("cuda").manual_seed(0)
    x = torch.randn((5, 64), generator=g, device="cuda").bfloat16()
    gate = torch.randn((8, 64), generator=g, device="cuda").bfloat16()
    gate[3, 10] = float("nan")
    ids, weights = ops.moe_topk(x, gate, 2)
    assert weights.isnan().all() and ((ids >= 0) & (ids < 8)).all()


@pytest.mark.parametrize("mode", ["plain", "relu2"])
# widths that fill whole rounds of streaming workgroups and ones that do not, short and long K
@pytest.mark.parametrize(("experts", "n", "k"), [(16, 4096, 128), (16, 4096, 2112), (8, 4096, 2048),
                                                 (8, 4096, 2112), (16, 3712, 192), (15, 2048, 64)])
@pytest.mark.parametrize("mean", [9, 10, 30, 53])
def test_products_that_fill_whole_rounds(mode, experts, n, k, mean):
    """Uneven loads on both ways of cutting a plain product."""
    from vllm_tgis_adapter_amd import ops

    g = torch.Generator("cuda").manual_seed(n + k + mean)
    counts = [0, 3 * mean - 1 + mean // 2, mean - mean // 2, 1] + [mean] * (experts - 4)
    seg = _segments(counts)
    assert int(seg[-1]) == experts * mean
    w = torch.randn((experts, n, k), generator=g, device="cuda").bfloat16() / k ** 0.5
    x = torch.randn((int(seg[-1]), k), generator=g, device="cuda").bfloat16()
    got = ops.moe_gemm(x, w, seg.cuda(), False, act="relu2" if mode == "relu2" else None)
    for e in range(experts):
        lo, hi = int(seg[e]), int(seg[e + 1])
        s = x[lo:hi].double() @ w[e].double().t()
        if mode == "relu2":
            s = s.clamp(min=0).square()
        err = (got[lo:hi].double() - s).abs()
        # one rounding to bf16; float32 sums of up to 2112 terms of size 1 / sqrt(k)
        assert (err <= 2 ** -8 * s.abs() + 1e-4).all(), (e, err.max().item())


# a token a workgroup up to 2048 tokens, then four
@pytest.mark.parametrize("tokens", [2048, 2049])
def test_router_of_many_tokens(tokens):
    test_router_grouping_and_sum(tokens, 9, 2, 1000)


# results of the weighted sum: less than a wave's, a workgroup's, more
@pytest.mark.parametrize("width", [8, 520, 8192, 8200])
@pytest.mark.parametrize("top", [1, 2, 3])
def test_sums_of_any_width(width, top):
    from vllm_tgis_adapter_amd.ops import _C

    g = torch.Generator("cuda").manual_seed(width)
    ye = torch.randn((5 * top, width), generator=g, device="cuda").bfloat16()
    pos = torch.randperm(5 * top, generator=g, device="cuda").int().view(5, top)
    weights = torch.rand((5, top), generator=g, device="cuda")
    out = torch.full((5, width), float("nan"), device="cuda").bfloat16()
    _C.moe_sum(out, ye, pos, weights)
    want = (weights.double()[..., None] * ye.double()[pos.long()]).sum(dim=1)
    # one rounding to bf16 of a float32 sum of three
    assert ((out.double() - want).abs() <= 2 ** -8 * want.abs() + 1e-6).all()


# parts of a wave and of a round of pairs, all of one expert
@pytest.mark.parametrize(("tokens", "top", "experts"), [
    (3, 2, 1), (40, 2, 8), (700, 3, 64), (1024, 1, 5), (1025, 1, 33), (2100, 2, 9), (5000, 3, 1)])
def test_pairs_without_an_expert(tokens, top, experts):
    from vllm_tgis_adapter_amd.ops import _C

    g = torch.Generator("cuda").manual_seed(tokens)
    ids = torch.randint(-2, experts + 2, (tokens, top), generator=g, device="cuda").int()
    rows, pos = torch.full((tokens * top,), -7).int().cuda(), torch.full_like(ids, -7)
    seg = torch.empty(experts + 1, dtype=torch.int32, device="cuda")
    _C.moe_group(rows, pos, seg, ids)
    real = (ids >= 0) & (ids < experts)
    count = torch.bincount(ids[real].long(), minlength=experts)
    assert torch.equal(seg[1:].long(), count.cumsum(0)) and seg[0] == 0
    at, e = pos[real].long(), ids[real].long()
    assert (at >= seg[e]).all() and (at < seg[e + 1]).all()
    assert torch.equal(at.sort().values, torch.arange(len(at), device="cuda"))
    token = torch.arange(tokens, device="cuda")[:, None].expand(-1, top)
    assert torch.equal(rows[at].long(), token[real])
    assert (pos[~real] == -7).all() and (rows[len(at):] == -7).all()
