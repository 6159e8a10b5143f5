"""Decode attention kernel (attention_decode_stream.hip) against the reference op:
tile, page and split edges, both caches."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

# around the 32-key tile, the four-tile share of a workgroup, and a cut sequence;
# 0: a padding row of a captured batch
EDGES = [1, 15, 16, 17, 31, 32, 33, 0, 63, 65, 127, 128, 129, 255, 257, 700]


def _caches(lens, block, kvh, hd, fp8, seed, width):
    g = torch.Generator().manual_seed(seed)
    need = [-(-n // block) for n in lens]
    ids = torch.randperm(sum(need) + 3, generator=g).tolist()
    tables = torch.zeros(len(lens), width, dtype=torch.int32)
    for i, n in enumerate(need):
        tables[i, :n] = torch.tensor([ids.pop() for _ in range(n)], dtype=torch.int32)
    kc, vc = (torch.randn(sum(need) + 3, block, kvh, hd, generator=g).bfloat16() for _ in "kv")
    if fp8:
        kc, vc = (c.to(torch.float8_e4m3fn).view(torch.uint8) for c in (kc, vc))
    return kc, vc, tables


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize(("kvh", "group", "hd", "block", "lens", "width"), [
    (8, 4, 128, 16, EDGES, 512),        # cut by the longest context the table takes
    (8, 4, 128, 16, EDGES, 44),         # fewer cuts
    (2, 8, 64, 16, EDGES, 512),
    (1, 1, 128, 8, [5000], 640),        # one head: as many cuts as there can be
    (1, 7, 64, 24, [3, 1000, 2999], 128),   # pages of no power of two
    (32, 1, 64, 1, [40, 77], 80),
    (8, 4, 128, 16, [97] * 200, 8),     # a batch that fills the chip: no cuts
])
def test_matches_the_reference(fp8, kvh, group, hd, block, lens, width):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from vllm_tgis_adapter_amd import ops
    from vllm_tgis_adapter_amd.ops import reference as R

    kc, vc, tables = _caches(lens, block, kvh, hd, fp8, 3, width)
    q = torch.randn(len(lens), kvh * group, hd,
                    generator=torch.Generator().manual_seed(4)).bfloat16()
    seq_lens = torch.tensor(lens, dtype=torch.int32)
    out = ops.paged_attention_decode(q.cuda(), kc.cuda(), vc.cuda(), tables.cuda(),
                                     seq_lens.cuda(), hd ** -0.5, max(lens)).float().cpu()
    if fp8:
        kc, vc = (c.view(torch.float8_e4m3fn) for c in (kc, vc))
    live = [i for i, n in enumerate(lens) if n]
    want = R.paged_attention(
        q[live].float(), kc.float(), vc.float(), tables[live],
        torch.arange(len(live) + 1, dtype=torch.int32), seq_lens[live], hd ** -0.5)
    # probabilities and the result are rounded to bf16: half a unit in the last of 8
    # bits each, of a weighted mean of values
    bound = 2 ** -8 * vc.float().abs().max()
    assert (out[live] - want).abs().max() <= bound
    assert torch.equal(out[[i for i, n in enumerate(lens) if not n]],
                       torch.zeros(len(lens) - len(live), kvh * group, hd))


def test_every_byte_of_a_cache():
    """One key: the result is its value, exactly, for all codes of e4m3."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from vllm_tgis_adapter_amd import ops

    codes = torch.arange(256, dtype=torch.uint8, device="cuda").view(1, 1, 2, 128)
    out = ops.paged_attention_decode(
        torch.ones((1, 2, 128), device="cuda").bfloat16(), torch.zeros_like(codes), codes,
        torch.zeros((1, 1), dtype=torch.int32, device="cuda"),
        torch.ones(1, dtype=torch.int32, device="cuda"), 0.1, 1)
    want = codes.view(torch.float8_e4m3fn).bfloat16().view(-1)
    torch.testing.assert_close(out.view(-1), want, rtol=0, atol=0, equal_nan=True)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize(("block", "lens", "width"), [
    (16, EDGES, 512), (16, [130, 640, 641, 1900], 160), (24, [3, 25, 1000, 3840], 160),
    (1, [1, 33, 129, 300], 320)])
def test_block_ids_past_the_end_say_nothing(fp8, block, lens, width):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from vllm_tgis_adapter_amd import ops

    kc, vc, tables = (t.cuda() for t in _caches(lens, block, 2, 128, fp8, 5, width))
    q = torch.randn(len(lens), 8, 128, generator=torch.Generator().manual_seed(6)).bfloat16().cuda()
    seq_lens = torch.tensor(lens, dtype=torch.int32, device="cuda")
    want = ops.paged_attention_decode(q, kc, vc, tables, seq_lens, 0.1, max(lens))
    used = (seq_lens + block - 1) // block
    past = torch.arange(width, device="cuda")[None] >= used[:, None]
    got = ops.paged_attention_decode(
        q, kc, vc, tables.masked_fill(past, 2 ** 31 - 1), seq_lens, 0.1, max(lens))
    assert torch.equal(got, want)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize(("kvh", "group", "hd", "nseq", "width"), [
    (8, 4, 128, 80, 40),       # 640 heads: up to two tiles a wave's each (bf16), sequences are cut
    (8, 1, 64, 81, 16),        # never
    (8, 8, 128, 192, 512),     # 1536: up to four tiles, uncut
    (4, 3, 64, 400, 9),
    (6, 2, 128, 300, 9),       # key heads are no whole workgroups: never
    # two tiles, four, of other heads and types
    (8, 4, 128, 112, 40), (8, 4, 64, 160, 40), (4, 1, 128, 640, 12), (4, 1, 64, 336, 40),
    (8, 4, 64, 256, 40), (8, 2, 128, 384, 12),
])
def test_heads_of_short_sequences_are_a_waves_each(fp8, kvh, group, hd, nseq, width):
    """Lengths on both sides of two and four tiles of 32 keys beside each other."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from vllm_tgis_adapter_amd import ops
    from vllm_tgis_adapter_amd.ops import reference as R

    edges = [1, 31, 33, 0, 64, 65, 128, 129]
    lens = [edges[i % 8] for i in range(nseq)]
    kc, vc, tables = _caches(lens, 16, kvh, hd, fp8, 5, width)
    q = torch.randn(nseq, kvh * group, hd, generator=torch.Generator().manual_seed(6)).bfloat16()
    seq_lens = torch.tensor(lens, dtype=torch.int32)
    out = ops.paged_attention_decode(q.cuda(), kc.cuda(), vc.cuda(), tables.cuda(),
                                     seq_lens.cuda(), hd ** -0.5, max(lens)).float().cpu()
    if fp8:
        kc, vc = (c.view(torch.float8_e4m3fn) for c in (kc, vc))
    live = [i for i, n in enumerate(lens) if n]
    want = R.paged_attention(
        q[live].float(), kc.float(), vc.float(), tables[live],
        torch.arange(len(live) + 1, dtype=torch.int32), seq_lens[live], hd ** -0.5)
    # as above
    assert (out[live] - want).abs().max() <= 2 ** -8 * vc.float().abs().max()
    assert not out[[i for i, n in enumerate(lens) if not n]].any()


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize(("dim", "off"), [(64, 1), (128, 2), (128, 3), (128, 4)])
def test_results_off_an_8_byte_boundary_are_stored_one_by_one(fp8, dim, off):
    """Short sequences, so many that elsewhere a wave has a key head; `off` results into the
    buffer a workgroup does, as in batches of a quarter of the size, whose bits these are."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from vllm_tgis_adapter_amd import ops

    lens = [(17, 33, 50, 64)[i % 4] for i in range(160)]
    kc, vc, tables = (t.cuda() for t in _caches(lens, 16, 8, dim, fp8, 7, 4))
    q = torch.randn(160, 32, dim, generator=torch.Generator().manual_seed(8)).bfloat16().cuda()
    seq_lens = torch.tensor(lens, dtype=torch.int32, device="cuda")

    def decode(out, rows):
        ops._C.paged_attention_decode(out, q[rows], kc, vc, tables[rows], seq_lens[rows],
                                      dim ** -0.5)
        return out

    assert ops._C.decode_alone_tiles(160, 8, 4, dim, fp8) == 2
    assert ops._C.decode_alone_tiles(40, 8, 4, dim, fp8) == -1
    few = torch.cat([decode(torch.empty_like(q[:40]), slice(i, i + 40)) for i in range(0, 160, 40)])
    whole = torch.full((q.numel() + 8,), 7.0, dtype=q.dtype, device="cuda")
    got = decode(whole[off:off + q.numel()].view_as(q), slice(0, 160))
    if off % 4:
        assert torch.equal(got, few)
    else:   # on such a boundary; sums in another order, rounded to 8 bits
        assert (got - few).abs().max() <= 2 ** -8 * few.abs().max()
    assert (whole[:off] == 7).all() and (whole[off + q.numel():] == 7).all()
