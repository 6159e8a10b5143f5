"""bf16 products of many rows by large tiles (gemm_ring.hip), plain and gated, against
float64: every tile's form at its edges in rows, K from one tile of 64 inputs on, odd counts
of them and uneven parts, and calls that take the tiles of their own accord."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

# rows and columns of W of a form's tile
FORMS = [(256, 256), (128, 256), (128, 128), (64, 128), (64, 64)]


@pytest.fixture(autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


def _inputs(m, n, k):
    g = torch.Generator("cuda").manual_seed(m + n + k)
    x, w = (torch.randn((r, k), generator=g, device="cuda").bfloat16() for r in (m, n))
    return x, (w / k ** 0.5).bfloat16()


def _check(got, x, w, gated):
    """float32 sums of K terms (2**-20 of their size) and one rounding to bf16; the gate
    passes a sum's error on by at most 1.1 times the other factor."""
    s, terms = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    off = 2 ** -20 * terms
    if gated:
        (g, u), (og, ou) = s.chunk(2, 1), off.chunk(2, 1)
        s = torch.nn.functional.silu(g) * u
        # and exp and the division in float32
        off = 1.1 * (og * u.abs() + ou * g.abs()) + 1e-5 * s.abs()
    err = (got.double() - s).abs()
    assert (err <= 2 ** -8 * s.abs() + off).all(), err.max().item()


@pytest.mark.parametrize("form", range(5))
@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("k", [64, 128, 448, 832])
def test_forms(form, gated, k):
    from vllm_tgis_adapter_amd.ops import _C

    bm, bn = FORMS[form]
    for m in (1, bm - 1, bm, bm + 1, 9 * bm + 17):      # nine tiles: a band and one more
        for cols in (1, 2, 3):
            n = bn * cols if not gated else bn * cols // 2
            if n % 128:
                continue
            x, w = _inputs(m, n * (1 + gated), k)
            y = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
            _C.gemm_ring(y, x, w, gated, form << 4 | 1)
            _check(y, x, w, gated)


@pytest.mark.parametrize("form", range(5))
@pytest.mark.parametrize(("parts", "k"), [(2, 128), (2, 192), (3, 448), (5, 2112), (8, 12352)])
def test_parts(form, parts, k):
    from vllm_tgis_adapter_amd.ops import _C

    x, w = _inputs(130, 512, k)
    y = torch.full((130, 512), float("nan"), dtype=torch.bfloat16, device="cuda")
    _C.gemm_ring(y, x, w, False, form << 4 | parts)
    _check(y, x, w, False)


# weights that one tile of rows reads go past the caches: tiles of 64 rows 20 million and more, larger
# ones 40
@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize(("form", "n"), [
    (0, 15872), (1, 15872), (2, 15872), (3, 15872), (4, 15872), (3, 8192), (4, 8192)])
def test_weights_read_once(form, n, gated):
    from vllm_tgis_adapter_amd.ops import _C

    n, k = n // (1 + gated), 2560
    for m in (FORMS[form][0] - 1, FORMS[form][0] + 1):   # read once, and twice
        assert _C.gemm_ring_reads_once(m, n, k, form << 4 | 1, gated) == (m < FORMS[form][0])
        x, w = _inputs(m, n * (1 + gated), k)
        y = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
        _C.gemm_ring(y, x, w, gated, form << 4 | 1)
        _check(y, x, w, gated)


@pytest.mark.parametrize("entry", ["gemm_block", "gemm_ring"])
def test_results_at_any_address(entry):
    """Results that start off a 16-byte boundary."""
    from vllm_tgis_adapter_amd.ops import _C

    x, w = _inputs(130, 384, 832)
    got = torch.full((130 * 384 + 1,), 7.0, dtype=torch.bfloat16, device="cuda")
    getattr(_C, entry)(got[1:].view(130, 384), x, w)
    assert got[0] == 7
    _check(got[1:].view(130, 384), x, w, False)


@pytest.mark.parametrize("parts", [4, 6, 7])
def test_counts_of_parts_that_are_added_at_once(parts):
    test_parts(4, parts, 64 * parts)


def test_plans_that_are_none():
    from vllm_tgis_adapter_amd.ops import _C

    x, w = _inputs(8, 128, 192)
    y = torch.empty((8, 128), dtype=torch.bfloat16, device="cuda")
    for plan in (-1, 0x51, 0x20, 0x29, 0x24, 0x01):   # form, parts, empty parts, columns
        with pytest.raises(RuntimeError):
            _C.gemm_ring(y, x, w, False, plan)


# first and last rows of the rule and the ones beside them: rows, N, K, whether it takes them
LINES = [(8, 16384, 2048, False), (9, 16384, 2048, True), (9, 2048, 8192, True),
         (16, 8192, 3584, False), (16, 4096, 4096, False), (17, 4096, 4096, True), (64, 4096, 4096, True),
         (33, 128, 8192, False), (17, 512, 4096, True), (39, 3072, 2048, False),
         (40, 3072, 2048, True), (64, 8192, 28672, True), (64, 28672, 4096, True),
         (17, 28672, 4096, True), (65, 28672, 4096, False), (256, 4096, 4096, True),
         (257, 4096, 4096, False), (128, 4096, 3520, False), (65, 2048, 8192, True),
         (1024, 2048, 8192, True), (1025, 2048, 8192, False)]


@pytest.mark.parametrize(("m", "n", "k", "own"), LINES)
def test_rule(m, n, k, own):
    from vllm_tgis_adapter_amd import ops

    assert ops._C.gemm_ring_wins(m, n, k, False) == own
    x, w = _inputs(m, n, k)
    _check(ops.linear(x, w), x, w, False)


@pytest.mark.parametrize(("m", "n", "k", "own"), [
    (17, 8192, 2048, True), (64, 14336, 4096, True), (24, 4096, 2048, True),
    (65, 8192, 2048, True), (512, 2048, 2048, True), (65, 3584, 8192, False)])
def test_gated_rule(m, n, k, own):
    from vllm_tgis_adapter_amd import ops

    x, w = _inputs(m, 2 * n, k)
    got = ops.gated_mlp_up(x, w)
    assert (got is not None) == own
    if own:
        _check(got, x, w, True)
    w.requires_grad_(True)
    if m > 64:      # products that are differentiated stay with the library
        assert ops.gated_mlp_up(x, w) is None
