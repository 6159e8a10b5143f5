"""Projections with adapters as the layers call them: which launches make a product, its deltas
and its gate, and that they are right, against float64."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

HIDDEN, INTER, Q, KV = 4096, 512, 256, 128
QKV = [("q_proj", 0, Q), ("k_proj", Q, Q + KV), ("v_proj", Q + KV, Q + 2 * KV)]
GU = [("gate_proj", 0, INTER), ("up_proj", INTER, 2 * INTER)]
SIZES = {"q_proj": (HIDDEN, Q), "k_proj": (HIDDEN, KV), "v_proj": (HIDDEN, KV),
         "o_proj": (HIDDEN, 640), "gate_proj": (HIDDEN, INTER), "up_proj": (HIDDEN, INTER)}


@pytest.fixture(autouse=True)
def _fresh():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from vllm_tgis_adapter_amd.engine import lora

    lora._STACK_CACHE.clear()
    lora._RECENT_SETS.clear()
    yield
    lora.clear_context()
    lora._STACK_CACHE.clear()
    lora._RECENT_SETS.clear()


def _normal(g, *shape, by=1.0):
    return (torch.randn(shape, generator=g, device="cuda") * by).bfloat16()


def _adapters(g, rank):
    """All projections at the largest rank; a smaller one without keys and gate; one of up
    only, and one that has nothing in this layer."""
    from vllm_tgis_adapter_amd.engine.lora import LoRAAdapter

    def weights(r, names):
        return {(0, n): (_normal(g, r, SIZES[n][0], by=SIZES[n][0] ** -0.5),
                         _normal(g, SIZES[n][1], r, by=r ** -0.5)) for n in names}

    every = list(SIZES)
    made = [LoRAAdapter(3, rank, 1.5, weights(rank, every)),
            LoRAAdapter(5, 5, 0.5, weights(5, [n for n in every if n[0] not in "kg"])),
            LoRAAdapter(8, 8, 2.0, weights(8, ["up_proj"])), LoRAAdapter(9, 4, 1.0, {})]
    return {a.lora_int_id: a for a in made}


def _layer(g, kind, bits):
    from vllm_tgis_adapter_amd.parallel import layers

    if kind == "o":
        mod = layers.RowParallelLinear(HIDDEN, 640).cuda()
    else:
        mod = layers.MergedColumnParallelLinear(HIDDEN, [INTER] * 2 if kind == "gate" else
                                                [Q, KV, KV]).cuda()
    mod.weight.data.copy_(_normal(g, *mod.weight.shape, by=HIDDEN ** -0.5))
    weight = mod.weight.data.double()
    if bits < 16:
        from vllm_tgis_adapter_amd import ops

        layers.quantize_module_(mod, bits)
        weight = ops.dequantize_weight(mod.weight_q, mod.weight_scale, bits,
                                       torch.float32).double()
    return mod, weight, {"o": [("o_proj", 0, 640)], "gate": GU, "qkv": QKV}[kind]


def _want(x, weight, projs, adapters, ids):
    """(values, what the roundings may add up to)"""
    xd = x.double()
    want, off = xd @ weight.t(), 2 ** -20 * (xd.abs() @ weight.abs().t())
    off += 2 ** -8 * want.abs()    # a product may be rounded ahead of its deltas
    for number, a in adapters.items():
        rows = ids == number
        for name, lo, hi in projs:
            if (0, name) not in a.weights:
                continue
            wa, wb = (t.double() for t in a.weights[(0, name)])
            want[rows, lo:hi] += a.scaling * (xd[rows] @ wa.t()) @ wb.t()
            off[rows, lo:hi] += 2 ** -20 * a.scaling * (xd[rows].abs() @ wa.abs().t()) @ wb.abs().t()
    return want, off


@pytest.mark.parametrize("kind", ["qkv", "o", "gate"])
@pytest.mark.parametrize("bits", [16, 8, 4])
@pytest.mark.parametrize("rank", [8, 16, 32, 64])
# either side of the rows that gemm_ring.hip's tiles take, of the library's and of the gate's lines
@pytest.mark.parametrize("tokens", [1, 5, 17, 61, 64, 65, 300, 1500])
def test_layers(kind, bits, rank, tokens):
    from vllm_tgis_adapter_amd.engine import lora

    g = torch.Generator("cuda").manual_seed(tokens + rank + bits)
    adapters = _adapters(g, rank)
    mod, weight, projs = _layer(g, kind, bits)
    x = _normal(g, tokens, HIDDEN)
    ids = torch.tensor([0, 3, 5, 8, 9], device="cuda")[
        torch.randint(5, (tokens,), generator=g, device="cuda")].int()
    ids[tokens // 3: tokens // 2] = 3
    lora.set_context(ids, adapters)
    got = mod.gated(x, lora=(0, projs)) if kind == "gate" else mod(x, lora=(0, projs))
    want, off = _want(x, weight, projs, adapters, ids)
    if bits < 16:   # weights are rounded to bf16 on some of the ways, 4-bit sums are longer
        off += 2 ** -9 * (x.double().abs() @ weight.abs().t())
        off += 2 ** -18 * x.double().abs().sum(1, keepdim=True) * weight.abs().amax(1)
    if kind == "gate":
        # deltas may be added to a rounded product and rounded again ahead of the gate
        off += 2 ** -8 * want.abs()
        (gate, up), (og, ou) = want.chunk(2, 1), off.chunk(2, 1)
        want = torch.nn.functional.silu(gate) * up
        off = 1.1 * og * (up.abs() + ou) + ou * gate.abs() + 1e-5 * want.abs()
    err = (got.double() - want).abs()
    assert (err <= 2 ** -8 * want.abs() + off + 1e-7).all(), (err - off).max().item()


@pytest.mark.parametrize(("tokens", "rank", "columns", "taken"), [
    (1024, 8, 512, True), (33, 16, 28672, True), (292, 16, 28672, True), (293, 16, 28672, False),
    (36, 32, 28672, True), (37, 32, 28672, False), (512, 32, 28672, False), (9, 64, 28672, True),
    (10, 64, 28672, False), (2048, 64, 28672, False)])
def test_where_the_gate_is_taken(tokens, rank, columns, taken, monkeypatch):
    """In the launch of the deltas only up to the tokens where that is the faster way."""
    from vllm_tgis_adapter_amd import ops
    from vllm_tgis_adapter_amd.engine import lora

    monkeypatch.setitem(SIZES, "gate_proj", (128, columns // 2))
    monkeypatch.setitem(SIZES, "up_proj", (128, columns // 2))
    gates, product = [], ops._C.lora_product
    monkeypatch.setattr(ops._C, "lora_product", lambda *a: (gates.append(a[-1]), product(*a)))
    g = torch.Generator("cuda").manual_seed(1)
    projs = [("gate_proj", 0, columns // 2), ("up_proj", columns // 2, columns)]
    lora.set_context(torch.full((tokens,), 3, dtype=torch.int32, device="cuda"),
                     _adapters(g, rank))
    x, y = _normal(g, tokens, 128), _normal(g, tokens, columns)
    lora.lora_linear(0, projs, x, None, lambda: y, gated=True)
    assert any(gates) == taken


def test_the_switch_of_the_products_here(monkeypatch):
    """Few rows stay with the library where VTA_GEMM_MAX_M says so, with adapters too."""
    from vllm_tgis_adapter_amd import ops
    from vllm_tgis_adapter_amd.engine import lora

    g = torch.Generator("cuda").manual_seed(2)
    mod, _, projs = _layer(g, "qkv", 16)
    lora.set_context(torch.full((40,), 3, dtype=torch.int32, device="cuda"), _adapters(g, 16))
    calls, product = [], ops._C.lora_product
    monkeypatch.setattr(ops._C, "lora_product", lambda *a: (calls.append(a), product(*a)))
    x = _normal(g, 40, HIDDEN)
    near = mod(x, lora=(0, projs))
    assert calls
    calls.clear()
    monkeypatch.setenv("VTA_GEMM_MAX_M", "0")
    far = mod(x, lora=(0, projs))
    assert not calls
    assert (near.double() - far.double()).norm() <= 2 ** -7 * far.double().norm()
