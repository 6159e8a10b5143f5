"""Expert products by large tiles: rows an expert at each line of the rule that chooses them,
uneven and empty segments, against float64."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


# means below and above 52, 110, 150, 220, with edges of 128 and 256 rows
COUNTS = [[52, 53], [53, 53], [129, 91], [111, 111], [0, 255, 45], [256, 45, 0], [151, 151],
          [300, 140], [221, 221], [257, 0, 511]]


@pytest.mark.parametrize("mode", ["plain", "silu", "relu2"])
@pytest.mark.parametrize("counts", COUNTS, ids=str)
@pytest.mark.parametrize(("n", "k"), [(128, 192), (512, 64), (256, 4096)])
def test_tiles(mode, counts, n, k):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from vllm_tgis_adapter_amd import ops

    g = torch.Generator("cuda").manual_seed(sum(counts) + n)
    seg = torch.zeros(len(counts) + 1, dtype=torch.int32)
    seg[1:] = torch.tensor(counts).cumsum(0)
    total, gated = int(seg[-1]), mode == "silu"
    w = (torch.randn((len(counts), (1 + gated) * n, k), generator=g, device="cuda")
         / k ** 0.5).bfloat16()
    x = torch.randn((total // 2, k), generator=g, device="cuda").bfloat16()
    rows = torch.randint(len(x), (total,), generator=g, device="cuda", dtype=torch.int32)
    got = ops.moe_gemm(x, w, seg.cuda(), gated, act="relu2" if mode == "relu2" else None,
                       rows=rows)
    for e in range(len(counts)):
        lo, hi = int(seg[e]), int(seg[e + 1])
        s = x[rows[lo:hi].long()].double() @ w[e].double().t()
        if gated:
            a, u = s.chunk(2, dim=1)
            s = torch.nn.functional.silu(a) * u
        elif mode == "relu2":
            s = s.clamp(min=0).square()
        # one rounding to bf16; float32 sums of up to 4096 terms and exp below 1e-4
        err = (got[lo:hi].double() - s).abs()
        assert (err <= 2 ** -8 * s.abs() + 2e-4).all(), (e, err.max().item())


# what has enough of them for 256 x 256 (short and long K, gated) and for 128 x 256: segments of one
# row more and less than tiles, of none, and of several tiles
@pytest.mark.parametrize(("mode", "counts", "n", "k", "tile"), [
    ("plain", [511, 0, 257, 256, 255, 1, 700, 512] * 3, 2048, 64, 0),
    ("relu2", [513, 300, 257, 256, 255, 129, 400, 512] * 3, 2048, 192, 0),
    ("plain", [257, 200, 256, 255, 222, 129, 213, 255] * 2, 4096, 2112, 0),
    ("silu", [257, 0, 256, 255, 1, 129, 127, 255] * 2, 1536, 192, 0),
    ("silu", [256, 100, 129, 128, 127, 70, 1, 257] * 2, 1536, 4096, 0),
    ("plain", [129, 128, 127, 1, 0, 257, 160, 110] * 2, 2048, 64, 1),
    ("relu2", [129, 128, 127, 1, 0, 257, 160, 110] * 2, 2048, 128, 1)])
def test_many_large_tiles(mode, counts, n, k, tile):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from vllm_tgis_adapter_amd import ops

    gated = mode == "silu"
    assert ops._C.moe_tile(sum(counts) // len(counts), len(counts), n * (1 + gated), k, gated) == tile
    test_tiles(mode, counts, n, k)


@pytest.mark.parametrize("module", ["_C", "_C_seq"])
@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("counts", [[5, 3], [60, 70], [300, 0, 141]], ids=str)
def test_results_at_any_address(module, mode, counts):
    """Results that start off a 16-byte boundary, rows past the last segment left as they are."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import importlib

    moe_gemm = importlib.import_module(f"vllm_tgis_adapter_amd.{module}").moe_gemm
    g = torch.Generator("cuda").manual_seed(len(counts))
    n, k, total = 256, 128, sum(counts)
    seg = torch.zeros(len(counts) + 1, dtype=torch.int32)
    seg[1:] = torch.tensor(counts).cumsum(0)
    w = torch.randn((len(counts), (1 + (mode == 1)) * n, k), generator=g, device="cuda")
    w = (w / k ** 0.5).bfloat16()
    x = torch.randn((total + 2, k), generator=g, device="cuda").bfloat16()
    got = torch.full(((total + 2) * n + 1,), 7.0, dtype=torch.bfloat16, device="cuda")
    moe_gemm(got[1:].view(total + 2, n), x, w, seg.cuda(), mode)
    assert (got[:1] == 7).all() and (got[1 + total * n:] == 7).all()
    for e in range(len(counts)):
        lo, hi = int(seg[e]), int(seg[e + 1])
        s = x[lo:hi].double() @ w[e].double().t()
        if mode == 1:
            a, u = s.chunk(2, dim=1)
            s = torch.nn.functional.silu(a) * u
        elif mode == 2:
            s = s.clamp(min=0).square()
        # as in test_tiles
        err = (got[1:].view(-1, n)[lo:hi].double() - s).abs()
        assert (err <= 2 ** -8 * s.abs() + 2e-4).all(), (e, err.max().item())


# tiles of 256 x 256 behind whole rounds of 256 whose K is cut: 16 by 8 with one row in the last,
# 32, 128 by 2 with an odd last part, one alone; 144 and none stay whole, and 120, as long in two parts
@pytest.mark.parametrize(("mode", "counts", "n", "k"), [
    ("plain", [400] * 7 + [513], 4096, 8192), ("relu2", [400] * 7 + [513], 4096, 8256),
    ("plain", [256] * 16 + [257], 4096, 8192), ("plain", [600] * 8, 4096, 8256),
    ("relu2", [600, 0] + [700] * 7, 4096, 8320), ("plain", [256] * 257, 256, 8192),
    ("plain", [600] * 7 + [769], 4096, 8192), ("plain", [400] * 8, 4096, 8192),
    ("plain", [256] * 47, 2048, 8192)])
def test_last_rounds_in_parts(mode, counts, n, k):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from vllm_tgis_adapter_amd import ops

    assert ops._C.moe_tile(sum(counts) // len(counts), len(counts), n, k, False) == 0
    test_tiles(mode, counts, n, k)


# the line between whole tiles and those whose K is cut (in 6, 8, 4 and 2) falls between the chunks of
# an expert's rows in one column tile: on the second of three, the fifth of six; and on the first
@pytest.mark.parametrize(("mode", "counts", "n", "k"), [
    ("plain", [700] * 9, 2560, 8192), ("relu2", [600] * 3 + [700] * 4 + [513], 2816, 8192),
    ("plain", [500] * 2 + [900] * 5 + [1300], 2560, 8192), ("plain", [600] * 8, 4096, 14336),
    ("plain", [400] * 9, 4096, 8192)])
def test_a_rows_results_do_not_depend_on_its_place(mode, counts, n, k):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from vllm_tgis_adapter_amd import ops

    assert ops._C.moe_tile(sum(counts) // len(counts), len(counts), n, k, False) == 0
    g = torch.Generator("cuda").manual_seed(n + len(counts))
    total = sum(counts)
    seg = torch.tensor([0, *counts]).cumsum(0).int().cuda()
    w = (torch.randn((len(counts), n, k), generator=g, device="cuda") / k ** 0.5).bfloat16()
    x = torch.randn((total, k), generator=g, device="cuda").bfloat16()
    order = torch.cat([lo + torch.randperm(m, generator=g, device="cuda")
                       for lo, m in zip(seg.tolist(), counts)])
    act = "relu2" if mode == "relu2" else None
    first = ops.moe_gemm(x, w, seg, False, act=act)
    assert torch.equal(ops.moe_gemm(x, w, seg, False, act=act, rows=order.int()), first[order])


# a whole round whatever the counts are; at most 6 chunks of rows by 32 tiles of columns, of which three
# (96 tiles) in two parts are the most
@pytest.mark.parametrize(("counts", "n", "parts"), [([300], 65536, 0), ([600, 600], 8192, 192)])
def test_room_for_parts(counts, n, parts):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from vllm_tgis_adapter_amd import ops

    assert ops._C.moe_tile(sum(counts) // len(counts), len(counts), n, 8192, False) == 0
    w = torch.zeros((len(counts), n, 8192), device="cuda").bfloat16()
    x = torch.zeros((sum(counts), 8192), device="cuda").bfloat16()
    seg = torch.tensor([0, *counts]).cumsum(0).int().cuda()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    out = ops.moe_gemm(x, w, seg, False)
    most = out.numel() * 2 + parts * 256 * 256 * 4
    assert torch.cuda.max_memory_allocated() - before <= most + (1 << 20)
