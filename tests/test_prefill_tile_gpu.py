"""Prompt attention over the paged cache (attention_prefill_tile.hip) against float64:
edges of the 32-row waves, of the workgroup's tokens and of the 64-key tiles, every split
of the waves into heads and tokens, prompts that earlier steps have begun."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

# heads, key heads: 8, 4, 2 heads of a group in a workgroup, one of three, one of one
HEADS = [(16, 2), (8, 2), (12, 2), (3, 1), (2, 2)]
# new tokens and those of earlier steps
SHAPES = [
    [(1, 0)], [(1, 63), (2, 64), (31, 1)], [(32, 0), (33, 31), (64, 64)],
    [(63, 65), (65, 127)], [(128, 0), (129, 700)], [(255, 3), (256, 0), (257, 64)],
    [(300, 1000), (7, 2049), (40, 0)], [(1100, 0)],
]


def _need():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


@pytest.mark.parametrize("shape", SHAPES, ids=str)
@pytest.mark.parametrize(("heads", "kv_heads"), HEADS)
@pytest.mark.parametrize(("dim", "dtype", "block"), [
    (128, torch.bfloat16, 16), (64, torch.bfloat16, 16), (128, torch.uint8, 16),
    (128, torch.bfloat16, 12), (64, torch.bfloat16, 1)])
def test_prefill(shape, heads, kv_heads, dim, dtype, block):
    _need()
    from vllm_tgis_adapter_amd import ops

    gen = torch.Generator("cuda").manual_seed(heads * 17 + dim + len(shape))
    new = [n for n, _ in shape]
    lens = [n + past for n, past in shape]
    need = [-(-n // block) for n in lens]
    ids = torch.randperm(sum(need), generator=torch.Generator().manual_seed(3)).tolist()
    tables, at = [], 0
    for n in need:
        tables.append(ids[at:at + n])
        at += n
    cache = [torch.randn((at + 1, block, kv_heads, dim), generator=gen, device="cuda")
             for _ in "kv"]
    if dtype == torch.uint8:
        cache = [c.to(torch.float8_e4m3fn) for c in cache]
        kc, vc = (c.view(torch.uint8) for c in cache)
    else:
        kc, vc = cache = [c.bfloat16() for c in cache]
    # what no sequence owns must not be looked at
    q = torch.randn((sum(new) + 2, heads, dim), generator=gen, device="cuda").bfloat16()
    start = [0]
    for n in new:
        start.append(start[-1] + n)

    def ints(v):
        return torch.tensor(v, dtype=torch.int32, device="cuda")

    scale = 1.3 * dim ** -0.5
    got = ops.paged_attention_prefill(
        q, kc, vc, ints([t + [0] * (max(need) - len(t)) for t in tables]), ints(start),
        ints(lens), scale, max(new), max(lens))
    for i, (n, past) in enumerate(shape):
        rows = slice(start[i], start[i] + n)
        k, v = (c[ints(tables[i]).long()].double().reshape(-1, kv_heads, dim)[:lens[i]]
                .repeat_interleave(heads // kv_heads, 1).transpose(0, 1).contiguous()
                for c in cache)
        s = q[rows].double().transpose(0, 1).contiguous() @ k.transpose(1, 2).contiguous() * scale
        pos = torch.arange(lens[i], device="cuda")
        s = s.masked_fill(pos[None, :] > pos[past:past + n, None], float("-inf"))
        p = s.softmax(-1)
        want = (p @ v).transpose(0, 1)
        terms = (p @ v.abs()).transpose(0, 1)
        # probabilities and the result are rounded to bf16 once each, which is off by half a
        # unit in the last of 8 bits: by 2**-8 of the value just above a power of two
        err = (got[rows].double() - want).abs()
        assert (err <= 1.01 * 2 ** -7 * terms + 1e-6).all(), (i, err.max().item())


def _paged(lens, kv_heads, dim, gen, block=16, fp8=False, unowned=None):
    """Caches and tables of sequences of these lengths; unowned: what the rows hold that
    no sequence has."""
    need = [-(-n // block) for n in lens]
    ids = torch.randperm(sum(need) + 1, generator=torch.Generator().manual_seed(7)).tolist()
    tables, at = torch.zeros((len(lens), max(need)), dtype=torch.int32), 0
    own = torch.zeros((sum(need) + 1, block), dtype=torch.bool)
    for i, n in enumerate(lens):
        tables[i, :need[i]] = torch.tensor(ids[at:at + need[i]])
        own[tables[i, :need[i]].long()] = torch.arange(need[i] * block).view(-1, block) < n
        at += need[i]
    cache = [torch.randn((len(own), block, kv_heads, dim), generator=gen, device="cuda")
             for _ in "kv"]
    cache = [c.to(torch.float8_e4m3fn) if fp8 else c.bfloat16() for c in cache]
    if unowned is not None:
        for c in cache:
            c.view(torch.uint8 if fp8 else torch.bfloat16)[~own.cuda()] = unowned
    return cache, tables


def _ints(v):
    return torch.tensor(v, dtype=torch.int32, device="cuda")


def _close(got, want, terms):
    """Probabilities and the result are rounded to bf16 once each (see above)."""
    err = (got.cpu().double() - want.double()).abs()
    assert (err <= 1.01 * 2 ** -7 * terms.double() + 1e-6).all(), err.max().item()


@pytest.mark.parametrize("scale", [-0.11, 0.0, -0.0, 1e-38, -1e-42, 1e-60, -1e-300])
@pytest.mark.parametrize(("kind", "dim"), [
    ("plain", 64), ("plain", 128), ("fp8", 128), ("windowed", 128), ("capped", 64),
    ("capped", 128), ("chunk", 128)])
def test_scale_of_any_sign(kind, dim, scale):
    """A row sees its own keys only, whatever the scale's sign."""
    _need()
    from vllm_tgis_adapter_amd import ops
    from vllm_tgis_adapter_amd.ops import reference as R

    gen = torch.Generator("cuda").manual_seed(dim)
    new, lens, heads, kv_heads = [70, 129], [135, 129], 8, 2
    (kc, vc), tables = _paged(lens, kv_heads, dim, gen, fp8=kind == "fp8")
    q = torch.randn((sum(new), heads, dim), generator=gen, device="cuda").bfloat16()
    start = [0, 70, 199]
    where = (tables.cuda(), _ints(start), _ints(lens))
    sinks = torch.linspace(-1, 1, heads)
    out = torch.full_like(q, float("nan"), dtype=torch.float32 if kind == "chunk" else None)
    if kind in ("plain", "fp8"):
        kb, vb = (c.view(torch.uint8) if kind == "fp8" else c for c in (kc, vc))
        out = ops.paged_attention_prefill(q, kb, vb, *where, scale, max(new), max(lens))
    elif kind == "windowed":
        ops.gqa_attention_prefill(q, kc, vc, *where, scale, max(new), out, window=40, sink=0.3)
    elif kind == "capped":
        ops.gqa_attention_prefill(q, kc, vc, *where, scale, max(new), out, window=40,
                                  sinks=sinks.cuda(), softcap=2.0)
    else:
        ops.chunk_attention_prefill(q, kc, vc, *where, scale, max(new), 48, out)

    def plain(v):
        args = (q.float().cpu(), kc.float().cpu(), v, tables, torch.tensor(start),
                torch.tensor(lens), scale)
        if kind == "chunk":
            return R.chunk_attention(*args, 48)
        if kind == "windowed":
            return R.paged_attention(*args, 40, 0.3)
        return R.paged_attention(*args, 40, sinks, 2.0) if kind == "capped" \
            else R.paged_attention(*args)

    _close(out, plain(vc.float().cpu()), plain(vc.float().abs().cpu()))


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("step", ["prompt", "decode", "decode into"])
def test_queries_and_results_in_any_order(step, dim):
    """Heads ahead of rows in memory: queries are read, and results written, by their
    strides."""
    _need()
    from vllm_tgis_adapter_amd import ops

    gen = torch.Generator("cuda").manual_seed(dim)
    lens = [33, 100, 7]
    (kc, vc), tables = _paged(lens, 2, dim, gen)
    new = [20, 100, 1] if step == "prompt" else [1] * 3
    q = torch.randn((sum(new), 8, dim), generator=gen, device="cuda").bfloat16()
    turned = q.transpose(0, 1).contiguous().transpose(0, 1)
    start = _ints([sum(new[:i]) for i in range(len(new) + 1)])

    def run(q, **kw):
        if step == "prompt":
            return ops.paged_attention_prefill(q, kc, vc, tables.cuda(), start, _ints(lens), 0.1,
                                               max(new), max(lens))
        return ops.paged_attention_decode(q, kc, vc, tables.cuda(), _ints(lens), 0.1, max(lens),
                                          **kw)

    want = run(q)
    if step == "decode into":
        out = torch.full_like(turned, float("nan"))
        assert not out.is_contiguous() and run(q, out=out) is out
        assert torch.equal(out, want)
    else:
        assert torch.equal(run(turned), want)
        out = torch.full_like(turned, float("nan"))
        if step == "prompt":
            ops.gqa_attention_prefill(turned, kc, vc, tables.cuda(), start, _ints(lens), 0.1,
                                      max(new), out)
        else:
            ops.gqa_attention_decode(turned, kc, vc, tables.cuda(), _ints(lens), 0.1, out)
        assert torch.equal(out, want)


@pytest.mark.parametrize(("dim", "fp8"), [(64, False), (128, False), (128, True)])
@pytest.mark.parametrize("step", ["prompt", "decode"])
def test_rows_that_no_sequence_owns(step, dim, fp8):
    """Free blocks, the rest of a last block and rows past the longest prompt's hold NaN."""
    _need()
    from vllm_tgis_adapter_amd import ops
    from vllm_tgis_adapter_amd.ops import reference as R

    gen = torch.Generator("cuda").manual_seed(dim)
    lens = [1, 17, 200, 65]
    new = [1, 3, 130, 65] if step == "prompt" else [1] * 4
    (kc, vc), tables = _paged(lens, 2, dim, gen, fp8=fp8, unowned=0x7f if fp8 else float("nan"))
    q = torch.randn((sum(new), 8, dim), generator=gen, device="cuda").bfloat16()
    start = [sum(new[:i]) for i in range(len(new) + 1)]
    kb, vb = (c.view(torch.uint8) if fp8 else c for c in (kc, vc))
    if step == "prompt":
        got = ops.paged_attention_prefill(q, kb, vb, tables.cuda(), _ints(start), _ints(lens),
                                          0.1, max(new), max(lens))
    else:
        got = ops.paged_attention_decode(q, kb, vb, tables.cuda(), _ints(lens), 0.1, max(lens))

    def plain(v):
        return R.paged_attention(q.float().cpu(), kc.float().cpu().nan_to_num(), v, tables,
                                 torch.tensor(start), torch.tensor(lens), 0.1)

    v = vc.float().cpu().nan_to_num()
    _close(got, plain(v), plain(v.abs()))


@pytest.mark.parametrize(("heads", "kv_heads", "dim", "fp8"), [
    (4, 4, 64, False), (4, 4, 128, False), (8, 4, 128, False), (4, 4, 128, True),
    (6, 2, 64, False)])
# the longest prompt and the keys on both sides of the lines of the waves: 16, 32, 64 and 128
# rows of 8, 4 and 2 waves, 128 and 512 keys
@pytest.mark.parametrize(("seqs", "longest", "past"), [
    (40, 9, 0), (40, 32, 96), (40, 33, 95), (40, 32, 97), (12, 64, 0), (12, 65, 63), (12, 128, 0),
    (12, 129, 0), (6, 64, 448), (6, 64, 449)])
def test_waves(heads, kv_heads, dim, fp8, seqs, longest, past):
    """Many short prompts: workgroups of two, four and eight waves."""
    _need()
    from vllm_tgis_adapter_amd import ops
    from vllm_tgis_adapter_amd.ops import reference as R

    gen = torch.Generator("cuda").manual_seed(longest)
    new = [1 + (7 * i) % longest for i in range(seqs - 1)] + [longest]
    lens = [n + past * (i % 2) for i, n in enumerate(new)]
    lens[-1] = longest + past
    (kc, vc), tables = _paged(lens, kv_heads, dim, gen, fp8=fp8,
                              unowned=0x7f if fp8 else float("nan"))
    q = torch.randn((sum(new), heads, dim), generator=gen, device="cuda").bfloat16()
    start = [sum(new[:i]) for i in range(seqs + 1)]
    kb, vb = (c.view(torch.uint8) if fp8 else c for c in (kc, vc))
    got = ops.paged_attention_prefill(q, kb, vb, tables.cuda(), _ints(start), _ints(lens), 0.1,
                                      longest, max(lens))

    def plain(v):
        return R.paged_attention(q.float().cpu(), kc.float().cpu().nan_to_num(), v, tables,
                                 torch.tensor(start), torch.tensor(lens), 0.1)

    v = vc.float().cpu().nan_to_num()
    _close(got, plain(v), plain(v.abs()))


# eight waves, whose tiles go round in three places of LDS: first to last place, once and twice round,
# a last tile of one key and a full one; blocks that a wave's load fits, that it does not, and of
# a size that is no power of two
@pytest.mark.parametrize("block", [32, 8, 4, 24])
@pytest.mark.parametrize(("dim", "fp8"), [(128, False), (64, False), (128, True)])
@pytest.mark.parametrize("keys", [65, 128, 129, 192, 193, 256, 321, 384, 449])
def test_places_of_tiles(block, dim, fp8, keys):
    _need()
    from vllm_tgis_adapter_amd import ops
    from vllm_tgis_adapter_amd.ops import reference as R

    gen = torch.Generator("cuda").manual_seed(keys)
    lens, new, heads = [keys] * 5, [64, 33, 1, 64, 50], 64
    (kc, vc), tables = _paged(lens, 8, dim, gen, block=block, fp8=fp8,
                              unowned=0x7f if fp8 else float("nan"))
    q = torch.randn((sum(new), heads, dim), generator=gen, device="cuda").bfloat16()
    start = [sum(new[:i]) for i in range(6)]
    kb, vb = (c.view(torch.uint8) if fp8 else c for c in (kc, vc))
    got = ops.paged_attention_prefill(q, kb, vb, tables.cuda(), _ints(start), _ints(lens), 0.1,
                                      64, keys)

    def plain(v):
        return R.paged_attention(q.float().cpu(), kc.float().cpu().nan_to_num(), v, tables,
                                 torch.tensor(start), torch.tensor(lens), 0.1)

    v = vc.float().cpu().nan_to_num()
    _close(got, plain(v), plain(v.abs()))


# parts of three tiles and more, of a sequence that has fewer too, four waves where eight were
@pytest.mark.parametrize("shape", [
    [(2, 600)] * 8, [(64, 500), (3, 190), (1, 0)], [(1000, 0)], [(256, 1000), (5, 190)],
    [(256, 0)] * 8], ids=str)
@pytest.mark.parametrize(("heads", "kv_heads"), [(32, 8), (64, 8)])
@pytest.mark.parametrize(("dim", "dtype"), [
    (64, torch.bfloat16), (128, torch.bfloat16), (128, torch.uint8)])
def test_prefill_of_served_heads(shape, heads, kv_heads, dim, dtype):
    test_prefill(shape, heads, kv_heads, dim, dtype, 16)
