"""Products of few rows (gemm_stream.hip) against float64: every way of cutting them,
edges of the 16-row tiles, K that ends in half a tile."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

ROWS = [1, 15, 16, 17, 23, 32, 33, 61, 64]
# N, K: one workgroup's columns, K of a single tile and of half a last one, as many
# columns as the other cuts take
SHAPES = [(128, 64), (128, 128), (256, 192), (384, 1088), (5120, 256), (8192, 320), (256, 8192),
          (1152, 4160), (4096, 4224), (16384, 4096), (9216, 8192)]


def _need():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


def _x(m, k, seed):
    g = torch.Generator("cuda").manual_seed(seed)
    return torch.randn((m, k), generator=g, device="cuda").bfloat16()


def _check(got, want, terms):
    """Sums of `terms` products in float32, one rounding to bf16: half a unit in the
    last of 8 bits of the value, and 2**-20 of the terms' size for the sums."""
    assert got.dtype == torch.bfloat16
    err = (got.double() - want).abs()
    assert (err <= 2 ** -8 * want.abs() + 2 ** -20 * terms).all(), err.max().item()


@pytest.mark.parametrize("m", ROWS)
@pytest.mark.parametrize(("n", "k"), SHAPES)
def test_plain(m, n, k):
    _need()
    from vllm_tgis_adapter_amd import ops

    x, w = _x(m, k, 1), _x(n, k, 2)
    _check(ops.linear(x, w), x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t())


@pytest.mark.parametrize("m", ROWS)
@pytest.mark.parametrize(("n", "k"), SHAPES)
def test_gated(m, n, k):
    _need()
    from vllm_tgis_adapter_amd import ops

    x, w = _x(m, k, 3), _x(2 * n, k, 4) / k ** 0.5
    g, u = (x.double() @ w.double().t()).chunk(2, dim=1)
    got = ops.gated_mlp_up(x, w)
    # float32 sums are off by far less than the last rounding; exp and the division
    # are good to 1e-5
    want = torch.nn.functional.silu(g) * u
    _check(got, want, 30 * (1 + g.abs()) * (1 + u.abs()))


@pytest.mark.parametrize("qbits", [8, 4])
@pytest.mark.parametrize("m", ROWS)
@pytest.mark.parametrize(("n", "k"), [s for s in SHAPES if s[1] % 128 == 0])
def test_rounded(qbits, m, n, k):
    _need()
    from vllm_tgis_adapter_amd import ops

    x, w = _x(m, k, 5), _x(n, k, 6)
    w[0] = 0.0                      # a row of zeros has the smallest scale
    w[1, : k // 2] = 64.0           # one group or half of a row far above the rest
    wq, scale = ops.quantize_weight(w, qbits)
    if qbits == 8:
        exact = wq.double() * scale.double()[:, None]
    else:
        q = torch.stack([wq & 0xF, wq >> 4], dim=2).view(n, k // 128, 128).double() - 8.0
        exact = (q * scale.double()[:, :, None]).view(n, k)
    got = ops.linear_quant(x, wq, scale, qbits)
    # 4 bits: sums of 8 + n/2 in place of n - 8, up to five times their size
    _check(got, x.double() @ exact.t(), 5 * (x.double().abs() @ exact.abs().t()
                                             + 4 * x.double().abs().sum(1, keepdim=True)
                                             * exact.abs().amax(1) / 4))


@pytest.mark.parametrize("qbits", [8, 4])
@pytest.mark.parametrize("m", [65, 127, 128, 129, 301, 460, 900])
# blocks for the choices of tile: narrow, 64 wide, 128 wide, and many (more of them:
# test_rounded_largest_tiles)
@pytest.mark.parametrize(("n", "k"), [(128, 128), (512, 384), (4096, 256), (8192, 640),
                                      (36864, 256)])
def test_rounded_many_rows(qbits, m, n, k):
    _need()
    from vllm_tgis_adapter_amd import ops

    x, w = _x(m, k, 7), _x(n, k, 8)
    wq, scale = ops.quantize_weight(w, qbits)
    exact = ops.dequantize_weight(wq, scale, qbits, torch.float32).double()
    got = ops.linear_quant(x, wq, scale, qbits)
    terms = x.double().abs() @ exact.abs().t()
    # above the line of the product's own widening the weights are rounded to bf16
    wide = m > ops._quant_rows(qbits, n, k)
    err = (got.double() - x.double() @ exact.t()).abs()
    bound = 2 ** -8 * (x.double() @ exact.t()).abs() + (2 ** -9 if wide else 2 ** -17) * terms
    assert (err <= bound).all(), (err - bound).max().item()


@pytest.mark.parametrize("qbits", [8, 4])
def test_widened_weights_are_the_rounded_ones(qbits):
    _need()
    from vllm_tgis_adapter_amd import ops

    w = _x(384, 640, 9)
    wq, scale = ops.quantize_weight(w, qbits)
    x = _x(2100, 640, 10)
    got = ops.linear_quant(x, wq, scale, qbits)
    want = torch.nn.functional.linear(x, ops.dequantize_weight(wq, scale, qbits))
    assert torch.equal(got, want)


@pytest.mark.parametrize(("n", "k"), [(128, 28672), (128, 28800), (256, 6272), (33024, 2176)])
def test_one_row(n, k):
    """Rows as long as are kept in LDS, longer ones, and more rows of W than workgroups."""
    _need()
    from vllm_tgis_adapter_amd import ops

    x, w = _x(1, k, 11), _x(n, k, 12) / k ** 0.5
    terms = x.double().abs() @ w.double().abs().t()
    _check(ops.linear(x, w), x.double() @ w.double().t(), terms)
    g, u = (x.double() @ w.double().t()).chunk(2, dim=1)
    if n % 256 == 0:
        _check(ops.gated_mlp_up(x, w), torch.nn.functional.silu(g) * u,
               30 * (1 + g.abs()) * (1 + u.abs()))
    wq, scale = ops.quantize_weight(w, 4)
    exact = ops.dequantize_weight(wq, scale, 4, torch.float32).double()
    # sums of 8 + n/2 in place of n - 8 (see test_rounded)
    size = x.double().abs().sum(1, keepdim=True) * exact.abs().amax(1)
    _check(ops.linear_quant(x, wq, scale, 4), x.double() @ exact.t(),
           5 * (x.double().abs() @ exact.abs().t() + size))


@pytest.mark.parametrize(("n", "k"), [(128, 128), (768, 768), (4096, 1024), (128, 1152),
                                      (768, 28672), (128, 28800)])
def test_one_row_of_int8(n, k):
    """Both sides of the shortest and the longest rows of the kernel for one."""
    _need()
    from vllm_tgis_adapter_amd import ops

    x, w = _x(1, k, 28), _x(n, k, 29)
    wq, scale = ops.quantize_weight(w, 8)
    exact = (wq.double() * scale.double()[:, None]).t()
    _check(ops.linear_quant(x, wq, scale, 8), x.double() @ exact, x.double().abs() @ exact.abs())


def _at_odd_offset(t):
    flat = torch.zeros(t.numel() + 1, dtype=t.dtype, device=t.device)
    out = flat[1:].view(t.shape)
    return out.copy_(t)


@pytest.mark.parametrize("qbits", [8, 4])
@pytest.mark.parametrize("which", ["x", "codes", "scales"])
@pytest.mark.parametrize("m", [65, 300, 1200])
def test_rounded_many_rows_from_any_address(qbits, which, m):
    """Tensors that start off a 16-byte boundary, in both forms of the product."""
    _need()
    from vllm_tgis_adapter_amd import ops

    x, w = _x(m, 256, 13), _x(256, 256, 14)
    wq, scale = ops.quantize_weight(w, qbits)
    want = ops.linear_quant(x, wq, scale, qbits)
    if which == "x":
        x = _at_odd_offset(x)
    elif which == "codes":
        wq = _at_odd_offset(wq)
    else:
        scale = _at_odd_offset(scale)
    got = ops.linear_quant(x, wq, scale, qbits)
    exact = x.double() @ ops.dequantize_weight(wq, scale, qbits, torch.float32).double().t()
    terms = x.double().abs() @ ops.dequantize_weight(wq, scale, qbits, torch.float32).double(
        ).abs().t()
    # weights are rounded to bf16 on some of the ways
    for y in (want, got):
        assert ((y.double() - exact).abs() <= 2 ** -8 * exact.abs() + 2 ** -9 * terms).all()


@pytest.mark.parametrize("form", ["unsigned codes", "bf16 scales"])
def test_rounded_many_rows_of_other_types(form):
    """What dequantize_weight makes of codes and scales that quantize_weight does not make."""
    _need()
    from vllm_tgis_adapter_amd import ops

    x, w = _x(100, 256, 15), _x(384, 256, 16)
    wq, scale = ops.quantize_weight(w, 8)
    if form == "unsigned codes":
        wq = (wq.to(torch.int16) + 127).to(torch.uint8)
    else:
        scale = scale.bfloat16()
    want = torch.nn.functional.linear(x, ops.dequantize_weight(wq, scale, 8))
    assert torch.equal(ops.linear_quant(x, wq, scale, 8), want)


@pytest.mark.parametrize("qbits", [8, 4])
def test_rounded_many_rows_keep_the_gradient(qbits):
    _need()
    from vllm_tgis_adapter_amd import ops

    x = _x(100, 256, 17).requires_grad_()
    wq, scale = ops.quantize_weight(_x(256, 256, 18), qbits)
    back = _x(100, 256, 19)
    ops.linear_quant(x, wq, scale, qbits).backward(back)
    want = back @ ops.dequantize_weight(wq, scale, qbits)
    assert torch.equal(x.grad, want)


@pytest.mark.parametrize("m", [16, 17, 32, 33, 64])
# columns on both sides of every line of the cut, K of whole, half and uneven shares
@pytest.mark.parametrize(("n", "k"), [(128, 4096), (2048, 4160), (2176, 6464), (2176, 6528),
                                      (1024, 4032), (1280, 8192), (4096, 12288), (4096, 640),
                                      (4224, 640), (6016, 320), (6144, 320),
                                      (12160, 192), (12288, 192), (20480, 8192)])
def test_gated_cuts(m, n, k):
    _need()
    from vllm_tgis_adapter_amd import ops

    x, w = _x(m, k, 20), _x(2 * n, k, 21) / k ** 0.5
    g, u = (x.double() @ w.double().t()).chunk(2, dim=1)
    _check(ops.gated_mlp_up(x, w), torch.nn.functional.silu(g) * u,
           30 * (1 + g.abs()) * (1 + u.abs()))


@pytest.mark.parametrize("m", [17, 49])
# K over 1 to 8 workgroups, of equal and of unequal numbers of tiles
@pytest.mark.parametrize(("n", "k"), [(6144, 4096), (7168, 4224), (10240, 3200), (5120, 8192),
                                      (2560, 7040), (16384, 2048), (4096, 8320)])
def test_parts_of_k(m, n, k):
    _need()
    from vllm_tgis_adapter_amd import ops

    x, w = _x(m, k, 22), _x(n, k, 23)
    _check(ops.linear(x, w), x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t())
    if k % 128 == 0:
        wq, scale = ops.quantize_weight(w, 4)
        exact = ops.dequantize_weight(wq, scale, 4, torch.float32).double()
        size = x.double().abs().sum(1, keepdim=True) * exact.abs().amax(1)
        _check(ops.linear_quant(x, wq, scale, 4), x.double() @ exact.t(),
               5 * (x.double().abs() @ exact.abs().t() + size))


# what aligned tensors still reach of the cuts for more than 16 rows in bf16 (the rest of
# test_plain, test_gated_cuts and test_parts_of_k has the tiles of gemm_ring.hip): K over several
# workgroups, over one, and the gated cut for many columns
@pytest.mark.parametrize(("m", "n", "k", "gated"), [
    (33, 4096, 3072, False), (39, 5120, 2944, False), (33, 5120, 1792, False),
    (39, 12288, 1024, False), (17, 12288, 640, True), (49, 12288, 12288, True)])
def test_cuts_of_aligned_tensors(m, n, k, gated):
    _need()
    from vllm_tgis_adapter_amd import ops

    assert not ops._C.gemm_ring_wins(m, n, k, gated)
    x, w = _x(m, k, 30), _x(n * (1 + gated), k, 31) / k ** 0.5
    want, terms = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    if gated:
        g, u = want.chunk(2, dim=1)
        _check(ops.gated_mlp_up(x, w), torch.nn.functional.silu(g) * u,
               30 * (1 + g.abs()) * (1 + u.abs()))
    else:
        _check(ops.linear(x, w), want, terms)


# and the same cuts where the tiles refuse a tensor, which starts four bytes off their boundary
@pytest.mark.parametrize("which", ["x", "w"])
@pytest.mark.parametrize(("m", "n", "k", "gated"), [
    (17, 6144, 4096, False), (25, 7168, 4224, False), (17, 10240, 3200, False),
    (49, 5120, 8192, False), (49, 16384, 2048, False), (17, 20480, 8192, True),
    (25, 7168, 4096, True), (49, 14336, 4096, True)])
def test_cuts_of_tensors_off_a_boundary(which, m, n, k, gated):
    _need()
    from vllm_tgis_adapter_amd import ops

    assert ops._C.gemm_ring_wins(m, n, k, gated)
    x, w = _x(m, k, 32), _x(n * (1 + gated), k, 33) / k ** 0.5
    flat = torch.zeros((x if which == "x" else w).numel() + 2, dtype=x.dtype, device="cuda")[2:]
    if which == "x":
        x = flat.view(x.shape).copy_(x)
    else:
        w = flat.view(w.shape).copy_(w)
    want, terms = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    if gated:
        g, u = want.chunk(2, dim=1)
        _check(ops.gated_mlp_up(x, w), torch.nn.functional.silu(g) * u,
               30 * (1 + g.abs()) * (1 + u.abs()))
    else:
        _check(ops.linear(x, w), want, terms)


@pytest.mark.parametrize("m", [1025, 1041])
def test_rounded_largest_tiles(m):
    """Wide matrices of few inputs, past 4096 blocks of 64 x 128."""
    _need()
    from vllm_tgis_adapter_amd import ops

    n, k = 32768, 256
    assert m <= ops._quant_rows(8, n, k) and (m + 63) // 64 * (n // 128) >= 4096
    x, w = _x(m, k, 24), _x(n, k, 25)
    wq, scale = ops.quantize_weight(w, 8)
    exact = (wq.double() * scale.double()[:, None]).t()
    _check(ops.linear_quant(x, wq, scale, 8), x.double() @ exact, x.double().abs() @ exact.abs())


# every panel with whole K and with K cut over workgroups, evenly and unevenly, last panels
# with one row and nearly full
@pytest.mark.parametrize(("m", "n", "k", "panel", "parts"), [
    (321, 128, 128, 0, 1), (65, 128, 2176, 0, 4), (161, 1024, 4096, 0, 5), (65, 28672, 384, 1, 1),
    (65, 6144, 4096, 1, 5), (321, 8192, 128, 2, 1), (161, 2048, 4224, 2, 6), (511, 4096, 128, 3, 1),
    (127, 2048, 6272, 3, 7), (511, 16384, 128, 4, 1), (511, 4096, 14336, 4, 4),
    (97, 28672, 384, 5, 1), (97, 6144, 4096, 5, 5), (129, 28672, 384, 6, 1), (257, 4096, 8192, 6, 4),
    (1199, 8192, 128, 7, 1), (301, 6144, 8192, 7, 5)])
def test_int8_panels(m, n, k, panel, parts):
    _need()
    from vllm_tgis_adapter_amd import ops

    assert m <= ops._quant_rows(8, n, k)
    assert ops._C.gemm_panel_plan(m, n, k) == (panel + 1) << 8 | parts
    x, w = _x(m, k, 26), _x(n, k, 27)
    wq, scale = ops.quantize_weight(w, 8)
    exact = (wq.double() * scale.double()[:, None]).t().contiguous()
    _check(ops.linear_quant(x, wq, scale, 8), x.double() @ exact, x.double().abs() @ exact.abs())


def _exact4(wq, scale):
    q = torch.stack([wq & 0xF, wq >> 4], dim=2).view(wq.shape[0], -1, 128).double() - 8.0
    return (q * scale.double()[:, :, None]).view(wq.shape[0], -1).t().contiguous()


# the same for 4 bits, one group and parts of unequal numbers of groups among them
@pytest.mark.parametrize(("m", "n", "k", "panel", "parts"), [
    (257, 4096, 128, 0, 1), (65, 128, 2176, 0, 4), (65, 28672, 128, 1, 1), (65, 6144, 4224, 1, 5),
    (321, 8192, 128, 2, 1), (161, 2048, 6272, 2, 7), (161, 6144, 128, 3, 1), (161, 2048, 2176, 3, 4),
    (511, 16384, 384, 4, 1), (97, 8192, 8192, 4, 8), (129, 28672, 128, 5, 1), (129, 6144, 6272, 5, 5),
    (257, 6144, 2176, 6, 1), (161, 2048, 4224, 6, 5)])
def test_4_bit_panels(m, n, k, panel, parts):
    _need()
    from vllm_tgis_adapter_amd import ops

    assert m <= ops._quant_rows(4, n, k)
    assert ops._C.gemm_panel_plan(m, n, k, 4) == (panel + 1) << 8 | parts
    x, w = _x(m, k, 30), _x(n, k, 31)
    w[0], w[n // 2:n // 2 + 2] = 0.0, 8.0     # least scales; the largest weight
    wq, scale = ops.quantize_weight(w, 4)
    wq[n // 2 + 1] = 0                        # -8, which rounding to the nearest does not give
    exact = _exact4(wq, scale)
    _check(ops.linear_quant(x, wq, scale, 4), x.double() @ exact, x.double().abs() @ exact.abs())


@pytest.mark.parametrize(("m", "n", "k", "panel"), [
    (65, 4096, 128, 0), (65, 14336, 128, 1), (321, 4096, 384, 2), (161, 3072, 384, 3),
    (511, 8192, 384, 4), (301, 14336, 4096, 5), (257, 8192, 128, 5), (513, 3584, 4096, 6),
    (131, 4224, 128, 6), (65, 1024, 8192, None)])
def test_4_bit_gated_panels(m, n, k, panel):
    _need()
    from vllm_tgis_adapter_amd import ops

    plan = ops._C.gemm_panel_gated_plan(m, n, k, 4)
    assert plan == (0 if panel is None else (panel + 1) << 8 | 1)
    x, w = _x(m, k, 32), _x(2 * n, k, 33) / k ** 0.5
    wq, scale = ops.quantize_weight(w, 4)
    got = ops.gated_quant(x, wq, scale, 4)
    if panel is None:
        assert got is None
        return
    g, u = (x.double() @ _exact4(wq, scale)).chunk(2, dim=1)
    _check(got, torch.nn.functional.silu(g) * u, 30 * (1 + g.abs()) * (1 + u.abs()))


# panels of up to 64 rows, with whole K and with K cut evenly and unevenly, and with the gate
@pytest.mark.parametrize("qbits", [8, 4])
@pytest.mark.parametrize(("m", "n", "k", "panel", "parts"), [
    (2, 128, 16512, 0, 8), (32, 28672, 4096, 1, 1), (17, 4096, 14336, 1, 8), (33, 4096, 2048, 2, 4), (48, 16384, 1024, 2, 1),
    (33, 28672, 4096, 3, 1), (64, 2048, 2304, 4, 4), (49, 16384, 1024, 4, 1), (49, 6144, 14464, 5, 5),
    (64, 28672, 2048, 5, 1)])
def test_panels_of_few_rows(qbits, m, n, k, panel, parts):
    _need()
    from vllm_tgis_adapter_amd import ops

    assert ops._C.gemm_panel_few_plan(m, n, k, qbits) == (panel + 17) << 8 | parts
    x, w = _x(m, k, 34), _x(n, k, 35)
    wq, scale = ops.quantize_weight(w, qbits)
    exact = _exact4(wq, scale) if qbits == 4 else (
        wq.double() * scale.double()[:, None]).t().contiguous()
    want, terms = x.double() @ exact, x.double().abs() @ exact.abs()
    _check(ops.linear_quant(x, wq, scale, qbits), want, terms)
    # off a 16-byte boundary: the streaming kernels
    odd = torch.empty(m * k + 1, dtype=x.dtype, device="cuda")[1:].view(m, k).copy_(x)
    _check(ops.linear_quant(odd, wq, scale, qbits), want, 20 * (terms + 1))


@pytest.mark.parametrize("qbits", [8, 4])
@pytest.mark.parametrize(("m", "n", "k", "panel"), [
    (4, 8192, 2048, 0), (32, 8192, 2048, 0), (9, 14336, 4096, 1), (33, 128, 128, 2),
    (47, 14336, 1024, 3), (64, 4096, 128, 4), (49, 14336, 2048, 5),
    (2, 128, 2048, None)])
def test_gated_panels_of_few_rows(qbits, m, n, k, panel):
    _need()
    from vllm_tgis_adapter_amd import ops

    plan = ops._C.gemm_panel_gated_plan(m, n, k, qbits)
    if panel is None:
        assert plan == 0
        return
    assert plan == (panel + 17) << 8 | 1
    x, w = _x(m, k, 36), _x(2 * n, k, 37) / k ** 0.5
    wq, scale = ops.quantize_weight(w, qbits)
    exact = _exact4(wq, scale) if qbits == 4 else (
        wq.double() * scale.double()[:, None]).t().contiguous()
    g, u = (x.double() @ exact).chunk(2, dim=1)
    _check(ops.gated_quant(x, wq, scale, qbits), torch.nn.functional.silu(g) * u,
           30 * (1 + g.abs()) * (1 + u.abs()))


# every panel that takes the gate in, whole and with rows missing; the last is refused: K is cut
@pytest.mark.parametrize(("m", "n", "k", "panel"), [
    (511, 128, 128, 0), (511, 2048, 128, 3),
    (65, 14336, 384, 1), (321, 4096, 128, 2), (511, 8192, 128, 4), (97, 14336, 384, 5),
    (129, 14336, 384, 6), (301, 14336, 4096, 7), (1199, 4096, 128, 7), (301, 3072, 8192, None)])
def test_int8_gated_panels(m, n, k, panel):
    _need()
    from vllm_tgis_adapter_amd import ops

    plan = ops._C.gemm_panel_gated_plan(m, n, k)
    assert plan == (0 if panel is None else (panel + 1) << 8 | 1)
    x, w = _x(m, k, 28), _x(2 * n, k, 29) / k ** 0.5
    wq, scale = ops.quantize_weight(w, 8)
    got = ops.gated_quant(x, wq, scale, 8)
    if panel is None:
        assert got is None
        return
    exact = (wq.double() * scale.double()[:, None]).t().contiguous()
    g, u = (x.double() @ exact).chunk(2, dim=1)
    _check(got, torch.nn.functional.silu(g) * u, 30 * (1 + g.abs()) * (1 + u.abs()))
    # as by two launches, to the roundings in between
    two = ops.silu_and_mul(ops.linear_quant(x, wq, scale, 8))
    assert (got.float() - two.float()).norm() <= 2 ** -6 * two.float().norm()
