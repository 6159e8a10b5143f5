"""Steps of one row in fewer launches (norm ahead of a product, gate or rotation and cache
write behind it) against the same in 64 bits, and int8 products of one row."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

EPS = 1e-5


def _weights(rows, k, bits, gen):
    """(weight, scales, the values they stand for)."""
    from vllm_tgis_adapter_amd import ops

    w = torch.randn((rows, k), generator=gen, device="cuda").mul_(k ** -0.5)
    if bits == 16:
        return w.bfloat16(), None, w.bfloat16().double()
    wq, s = ops.quantize_weight(w, bits)
    if bits == 8:
        return wq, s, wq.double() * s.double()[:, None]
    q = torch.stack([wq & 15, wq >> 4], dim=2).view(rows, k).double() - 8
    return wq, s, (q.view(rows, -1, 128) * s.double()[..., None]).view(rows, k)


def _row(k, gen, with_residual):
    x = torch.randn((1, k), generator=gen, device="cuda").bfloat16()
    r = (torch.randn((1, k), generator=gen, device="cuda") * 3).bfloat16() if with_residual else None
    g = (1 + 0.1 * torch.randn(k, generator=gen, device="cuda")).bfloat16()
    total = x if r is None else (x.float() + r.float()).bfloat16()
    n = total.double()
    return x, r, g, total, n * torch.rsqrt(n.square().mean() + EPS) * g.double()


def _close(got, want, ulps=2.0):
    """The one rounding of a normed input (2^-9 each at most, at random over the sum: six
    times their root mean square) and those of the result: ulps of bf16 of the value, or of
    the results' root mean square."""
    bound = ulps * 2.0 ** -8 * torch.maximum(want.abs(), want.square().mean().sqrt())
    assert ((got.double() - want).abs() <= bound).all()


def _close_gated(got, gate, up):
    """The inputs' rounding goes into both factors (the gate's slope is 1.1 at most)."""
    own = 6 * 2.0 ** -9 * 3 ** -0.5
    silu = torch.nn.functional.silu(gate)
    bound = (own * gate.square().mean().sqrt() * 1.1 * up.abs()
             + own * up.square().mean().sqrt() * silu.abs() + 2.0 ** -8 * (silu * up).abs()
             + own ** 2)
    assert ((got.double() - silu * up).abs() <= bound).all()


@pytest.mark.parametrize("bits", [16, 8, 4])
@pytest.mark.parametrize(("k", "inter"), [(128, 128), (2048, 256), (4096, 4736), (6272, 128),
                                          (8192, 1024), (28672, 128)])
@pytest.mark.parametrize("with_residual", [True, False])
def test_norm_and_gate(bits, k, inter, with_residual):
    from vllm_tgis_adapter_amd import ops

    gen = torch.Generator("cuda").manual_seed(k + bits)
    x, r, g, total, n = _row(k, gen, with_residual)
    w, s, value = _weights(2 * inter, k, bits, gen)
    before = None if r is None else r.clone()
    out, rest = ops.row_norm_gated(x, r, g, EPS, w, s, bits)
    assert torch.equal(rest, total) and (r is None or torch.equal(r, before))
    _close_gated(out, *(n @ value.t()).chunk(2, dim=1))


@pytest.mark.parametrize("bits", [16, 8, 4])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize(("k", "heads", "kv_heads", "dim"),
                         [(2048, 32, 8, 64), (4096, 32, 8, 128), (128, 2, 1, 32), (8192, 2, 1, 256)])
def test_norm_and_rotation(bits, fp8, k, heads, kv_heads, dim):
    from vllm_tgis_adapter_amd import ops

    gen = torch.Generator("cuda").manual_seed(k + bits)
    x, r, g, total, n = _row(k, gen, True)
    w, s, value = _weights((heads + 2 * kv_heads) * dim, k, bits, gen)
    angle = torch.rand((500, dim // 2), generator=gen, device="cuda") * 6.3
    cos_sin = torch.cat([angle.cos(), angle.sin()], dim=1).contiguous()
    for slot in (37, -1):
        kc, vc = (torch.full((20, 16, kv_heads, dim), 3, device="cuda",
                             dtype=torch.uint8 if fp8 else torch.bfloat16) for _ in "kv")
        untouched = kc.clone()
        q, rest = ops.row_norm_qkv(
            x, r, g, EPS, w, s, bits, heads, torch.tensor([411], device="cuda"), cos_sin, kc, vc,
            torch.tensor([slot], device="cuda"))
        assert torch.equal(rest, total)
        y = (n @ value.t()).view(heads + 2 * kv_heads, dim)
        lo, hi = y[:heads + kv_heads].chunk(2, dim=1)
        c, si = cos_sin[411].double().chunk(2)
        turned = torch.cat([lo * c - hi * si, hi * c + lo * si], dim=1)
        # rounded ahead of the rotation and behind it
        _close(q.view(heads, dim), turned[:heads], ulps=4.0)
        for cache, want in ((kc, turned[heads:]), (vc, y[heads + kv_heads:])):
            rows = cache.view(-1, kv_heads, dim)
            others = torch.arange(320, device="cuda") != slot
            assert torch.equal(rows[others], untouched.view(-1, kv_heads, dim)[others])
            if slot < 0:
                continue
            if fp8:   # three bits of mantissa
                _close(rows[slot].view(torch.float8_e4m3fn).float(), want, ulps=2.0 ** 4 + 4)
            else:
                _close(rows[slot], want, ulps=4.0)


@pytest.mark.parametrize(("n", "k"), [(128, 128), (3072, 2048), (256, 2176), (4096, 14336),
                                      (128, 28672)])
def test_int8_products_of_one_row(n, k):
    from vllm_tgis_adapter_amd import ops

    gen = torch.Generator("cuda").manual_seed(n + k)
    w, s, value = _weights(n, k, 8, gen)
    x = torch.randn((1, k), generator=gen, device="cuda").bfloat16()
    _close(ops.linear_quant(x, w, s, 8), x.double() @ value.t())


@pytest.mark.parametrize("bits", [16, 8, 4])
@pytest.mark.parametrize(("n", "k"), [
    (128, 7168), (2048, 7296),       # a K that ends inside a wave's load
    (2176, 8320), (4096, 8192), (4096, 14464), (4224, 6400), (8192, 7168), (8320, 8320),
    (16512, 7168), (16512, 8320),    # more rows than the workgroups take at a time
    (256, 28672), (2688, 28672), (6144, 20480), (4608, 20480)])   # rows that fill LDS
def test_long_rows(bits, n, k):
    """Plain products of every form, on both sides of where workgroups of eight waves begin."""
    from vllm_tgis_adapter_amd import ops

    gen = torch.Generator("cuda").manual_seed(n + k + bits)
    w, s, value = _weights(n, k, bits, gen)
    x = torch.randn((1, k), generator=gen, device="cuda").bfloat16()
    got = ops.linear(x, w) if bits == 16 else ops.linear_quant(x, w, s, bits)
    _close(got, x.double() @ value.t())


@pytest.mark.parametrize("bits", [16, 8, 4])
@pytest.mark.parametrize(("k", "inter"), [
    (1024, 640), (1920, 640), (2048, 4224), (1280, 8320), (2176, 1152), (2176, 1280), (8320, 4224),
    (8192, 14336)])
def test_gates_of_long_rows(bits, k, inter):
    from vllm_tgis_adapter_amd import ops

    gen = torch.Generator("cuda").manual_seed(k + bits)
    x, r, g, total, n = _row(k, gen, True)
    w, s, value = _weights(2 * inter, k, bits, gen)
    out, rest = ops.row_norm_gated(x, r, g, EPS, w, s, bits)
    assert torch.equal(rest, total)
    _close_gated(out, *(n @ value.t()).chunk(2, dim=1))


@pytest.mark.parametrize("bits", [16, 8])
@pytest.mark.parametrize(("k", "heads", "kv_heads"), [(8192, 38, 2), (8192, 40, 2), (4096, 44, 2)])
def test_rotation_of_long_rows(bits, k, heads, kv_heads):
    """Heads of 128, around the widths where K is dealt to fewer of eight waves."""
    from vllm_tgis_adapter_amd import ops

    gen = torch.Generator("cuda").manual_seed(k + heads + bits)
    x, r, g, total, n = _row(k, gen, True)
    w, s, value = _weights((heads + 2 * kv_heads) * 128, k, bits, gen)
    cos_sin = torch.cat([torch.ones(500, 64), torch.zeros(500, 64)], dim=1).cuda()
    kc, vc = (torch.zeros((4, 16, kv_heads, 128), device="cuda", dtype=torch.bfloat16)
              for _ in "kv")
    q, rest = ops.row_norm_qkv(x, r, g, EPS, w, s, bits, heads, torch.tensor([7], device="cuda"),
                               cos_sin, kc, vc, torch.tensor([20], device="cuda"))
    assert torch.equal(rest, total)
    y = (n @ value.t()).view(heads + 2 * kv_heads, 128)
    _close(torch.cat([q.view(heads, 128), kc.view(-1, kv_heads, 128)[20],
                      vc.view(-1, kv_heads, 128)[20]]), y, ulps=4.0)


def test_what_stays_with_the_launches_apart(monkeypatch):
    from vllm_tgis_adapter_amd import ops

    gen = torch.Generator("cuda").manual_seed(5)
    x, r, g, _, _ = _row(256, gen, True)
    w = torch.randn((512, 256), generator=gen, device="cuda").bfloat16()
    assert ops.row_norm_gated(x, r, g, EPS, w, None) is not None
    assert ops.row_norm_gated(x.expand(2, -1).contiguous(), r, g, EPS, w, None) is None
    assert ops.row_norm_gated(x.half(), r, g, EPS, w, None) is None
    assert ops.row_norm_gated(x, r, g.float(), EPS, w, None) is None
    assert ops.row_norm_gated(x, r, g, EPS, w[:, ::2], None) is None
    assert ops.row_norm_gated(x, r, g, EPS, w[:256 + 128], None) is None
    x1 = torch.empty(257, device="cuda", dtype=torch.bfloat16)[1:].view(1, 256)   # off 16 bytes
    assert ops.row_norm_gated(x1, r, g, EPS, w, None) is None
    assert ops.row_norm_gated(x, r, g, EPS, w.clone().requires_grad_(), None) is None
    monkeypatch.setenv("VTA_GEMM_MAX_M", "0")
    assert ops.row_norm_gated(x, r, g, EPS, w, None) is None
