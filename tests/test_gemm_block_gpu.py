"""bf16 products by large tiles with a cut K (gemm_ring.hip) against float64: rows around
the tiles of 128, a K of one tile, of uneven and of equal parts, and the rule that sends a
product there."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

# N, K: one part, parts of unequal length (193 tiles in 8), eight equal ones, two a CU
SHAPES = [(128, 64), (384, 960), (128, 12352), (2048, 8192), (4096, 14336), (10240, 8192)]


def _need():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


def _inputs(m, n, k):
    g = torch.Generator("cuda").manual_seed(m + n + k)
    return [torch.randn((r, k), generator=g, device="cuda").bfloat16() for r in (m, n)]


def _check(got, x, w):
    """float32 sums, one rounding to bf16: half a unit in the last of 8 bits of the
    value, and 2**-20 of the terms' size."""
    want = x.double() @ w.double().t()
    terms = x.double().abs() @ w.double().abs().t()
    err = (got.double() - want).abs()
    assert (err <= 2 ** -8 * want.abs() + 2 ** -20 * terms).all(), err.max().item()


@pytest.mark.parametrize("m", [1, 65, 127, 128, 129, 257, 512])
@pytest.mark.parametrize(("n", "k"), SHAPES)
def test_tiles(m, n, k):
    _need()
    from vllm_tgis_adapter_amd.ops import _C

    x, w = _inputs(m, n, k)
    y = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
    _C.gemm_block(y, x, w)
    _check(y, x, w)


# the last row below and the first row of the rule, the last row of it and the first above
LINES = [(4096, 14336, 65, 640), (8192, 8192, 65, 256), (2048, 8192, 129, 700),
         (1024, 8192, 257, 700), (2560, 8192, 200, 512), (12288, 8192, 65, 128)]


@pytest.mark.parametrize(("m", "n", "k", "own"), [
    (m, n, k, own) for n, k, lo, hi in LINES
    for m, own in ((lo - 1, False), (lo, True), (hi, True), (hi + 1, False))] + [
    (128, 12416, 8192, False), (128, 4096, 8128, False), (512, 57344, 8192, False)])
def test_rule(m, n, k, own, monkeypatch):
    """Which product a call gets, and that it is right."""
    _need()
    from vllm_tgis_adapter_amd import ops

    calls, run = [], ops._C.gemm_block
    monkeypatch.setattr(ops._C, "gemm_block", lambda *a: (calls.append(a), run(*a)))
    x, w = _inputs(m, n, k)
    y = ops.linear(x, w)
    assert bool(calls) == own
    _check(y, x, w)


@pytest.mark.parametrize("which", ["x", "w"])
def test_any_address(which):
    """Tensors that start off a 16-byte boundary."""
    _need()
    from vllm_tgis_adapter_amd import ops

    x, w = _inputs(200, 4096, 8192)

    def moved(t):
        flat = torch.zeros(t.numel() + 1, dtype=t.dtype, device="cuda")
        return flat[1:].view(t.shape).copy_(t)

    x, w = (moved(x), w) if which == "x" else (x, moved(w))
    _check(ops.linear(x, w), x, w)


@pytest.mark.parametrize("which", ["x", "w"])
def test_gradient(which):
    """A differentiated product has its gradient at every number of rows."""
    _need()
    from vllm_tgis_adapter_amd import ops

    x, w = _inputs(200, 4096, 8192)
    (x if which == "x" else w).requires_grad_()
    y = ops.linear(x, w)
    back = torch.ones_like(y)
    y.backward(back)
    if which == "x":
        want = back.float() @ w.float()
    else:
        want = back.float().t() @ x.float()
    got = (x if which == "x" else w).grad.float()
    # float32 sums, one rounding to bf16
    assert (got - want).norm() <= 2 ** -8 * want.norm()
