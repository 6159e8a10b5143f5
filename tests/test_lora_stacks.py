"""Adapters of a batch side by side (engine/lora.py): how the stacks are laid out, and the
deltas of whole projection lists against float64."""

from __future__ import annotations

import pytest
import torch

from vllm_tgis_adapter_amd.engine import lora

SPANS = [("q_proj", 0, 40), ("k_proj", 40, 48), ("v_proj", 48, 56)]
MLP = [("gate_proj", 0, 264), ("up_proj", 264, 528)]
SIZE = 72


def _adapter(number, rank, seed, lacks=(), device="cpu", dtype=torch.float32):
    g = torch.Generator().manual_seed(seed)
    weights = {}
    for layer in range(2):
        for name, lo, hi in SPANS + MLP:
            if name in lacks or (layer, name) in lacks:
                continue
            weights[(layer, name)] = tuple(
                torch.randn(s, generator=g).to(device=device, dtype=dtype)
                for s in ((rank, SIZE), (hi - lo, rank)))
    return lora.LoRAAdapter(lora_int_id=number, rank=rank, scaling=0.5 + number % 7,
                            weights=weights)


def _adapters(**kw):
    """Ranks off and on the padded ones; one without keys, one without the second layer's
    feed-forward, one without that layer."""
    made = [_adapter(910001, 5, 1, **kw), _adapter(910004, 16, 2, lacks=("k_proj",), **kw),
            _adapter(910007, 40, 3, lacks=((1, "gate_proj"), (1, "up_proj")), **kw),
            _adapter(910009, 8, 4, lacks=[(1, n) for n, _, _ in SPANS + MLP], **kw)]
    return {a.lora_int_id: a for a in made}


@pytest.fixture(autouse=True)
def _fresh():
    lora.clear_context()
    yield
    for number in (910001, 910004, 910007, 910009):
        lora.invalidate_adapter(number)
    lora.clear_context()


@pytest.mark.parametrize(("layer", "projs", "present"), [
    (0, SPANS, [0, 1, 2]), (1, SPANS, [0, 1, 2]), (0, SPANS[1:2], [0]), (1, MLP, [0, 1]),
    (0, [("o_proj", 0, 72)], []), (1, [("o_proj", 0, 8)] + SPANS[2:], [1])])
def test_layout(layer, projs, present):
    adapters = _adapters()
    lora.set_context(torch.zeros(1, dtype=torch.int32), adapters)
    got = lora._get_stacks(layer, projs, SIZE, torch.float32, "cpu")
    assert lora._get_stacks(layer, projs, SIZE, torch.float32, "cpu") is got
    if not present:
        assert got is None
        return
    a, b, scales, spans = got
    have = [projs[i] for i in present]
    assert spans == [(lo, hi) for _, lo, hi in have]
    assert scales.tolist() == [adapters[i].scaling for i in sorted(adapters)]
    # padded to the largest rank among them, rounded up to what the kernels take
    rank = max(ad.weights[(layer, n)][0].shape[0] for ad in adapters.values()
               for n, _, _ in have if (layer, n) in ad.weights)
    padded = b.shape[2]
    assert padded == min(r for r in (8, 16, 32, 64) if r >= rank)
    assert a.shape == (4, len(have) * padded, SIZE)
    at = 0
    for p, (name, lo, hi) in enumerate(have):
        for s, number in enumerate(sorted(adapters)):
            rows, cols = a[s, p * padded:(p + 1) * padded], b[s, at: at + hi - lo]
            down, up = adapters[number].weights.get(
                (layer, name), (torch.zeros(0, SIZE), torch.zeros(hi - lo, 0)))
            r = down.shape[0]
            assert torch.equal(rows[:r], down) and not rows[r:].any()
            assert torch.equal(cols[:, :r], up) and not cols[:, r:].any()
        at += hi - lo
    assert at == b.shape[1]


def _check(adapters, ids, layer, projs, device):
    g = torch.Generator().manual_seed(len(ids) + layer)
    width = projs[-1][2]
    x = torch.randn(len(ids), SIZE, generator=g).bfloat16().to(device)
    base = torch.randn(len(ids), width, generator=g).bfloat16().to(device)
    out = base.clone()
    lora.set_context(torch.tensor(ids, dtype=torch.int32, device=device), adapters)
    lora.apply_lora(layer, projs, x, out)
    want, terms = base.double(), base.double().abs()
    for i, number in enumerate(ids):
        for name, lo, hi in projs:
            if number in adapters and (layer, name) in adapters[number].weights:
                down, up = (m.double() for m in adapters[number].weights[(layer, name)])
                s = adapters[number].scaling
                want[i, lo:hi] += s * (up @ (down @ x[i].double()))
                terms[i, lo:hi] += s * (up.abs() @ (down.abs() @ x[i].double().abs()))
    # one rounding to bf16, and float32 sums: 2**-20 of the size of their terms
    err = (out.double() - want).abs()
    assert (err <= 2 ** -8 * want.abs() + 2 ** -20 * terms).all(), err.max().item()


@pytest.mark.gpu
@pytest.mark.parametrize("layer", [0, 1])
@pytest.mark.parametrize("projs", [SPANS, MLP, SPANS[:1]], ids=["qkv", "mlp", "q"])
def test_deltas_of_a_mixed_batch(layer, projs):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    kw = dict(device="cuda", dtype=torch.bfloat16)
    adapters = _adapters(**kw)
    ids = [0, 910001, 910004, 910007, 910009, 910007, 910007, 5] * 5
    _check(adapters, ids, layer, projs, "cuda")
    # another adapter comes under a number that a batch has used
    lora.invalidate_adapter(910004)
    adapters[910004] = _adapter(910004, 7, 9, **kw)
    _check(adapters, ids, layer, projs, "cuda")
    _check({910009: adapters[910009]}, ids, layer, projs, "cuda")
