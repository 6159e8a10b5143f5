"""Queries, keys and values that are column slices of one projection: rotation,
cache write and a whole step of several rows, against the reference ops."""

from __future__ import annotations

import pytest
import torch

DEVICES = ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)]


def _need(device):
    if device == "cuda" and not torch.cuda.is_available():
        pytest.skip("no GPU")


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
# (query heads, key heads, head size): the last one's rows are not 16-byte aligned
@pytest.mark.parametrize(("nq", "nk", "hd"), [(32, 8, 128), (4, 2, 64), (3, 1, 6)])
@pytest.mark.parametrize("rows", [1, 2, 37])
def test_rotation_and_cache_write_of_slices(device, dtype, nq, nk, hd, rows):
    from vllm_tgis_adapter_amd import ops
    from vllm_tgis_adapter_amd.ops import reference as R

    _need(device)
    if device == "cuda" and hd == 6:
        pytest.skip("cache rows of a multiple of 16 bytes only")
    g = torch.Generator().manual_seed(0)
    qkv = torch.randn(rows, (nq + 2 * nk) * hd, generator=g).to(dtype)
    pos = torch.randint(0, 99, (rows,), generator=g)
    cs = R.make_cos_sin_cache(hd, 100, 10000.0, torch.float32)
    split = [nq * hd, nk * hd, nk * hd]
    want_q, want_k = R.rotary_embedding(pos, *(t.contiguous() for t in qkv.split(split, -1)[:2]),
                                        hd, cs)
    slots = torch.randperm(48, generator=g)[:rows]

    q, k, v = qkv.to(device).split(split, dim=-1)
    want_v = v.cpu().clone()
    q, k = ops.rotary_embedding(pos.to(device), q, k, hd, cs.to(device))
    assert device == "cpu" or q.is_contiguous()
    # one rounding to the type either way
    tol = 1e-5 if dtype == torch.float32 else 2 ** -7
    torch.testing.assert_close(q.cpu(), want_q, atol=tol, rtol=tol)
    torch.testing.assert_close(k.cpu(), want_k, atol=tol, rtol=tol)
    kc, vc = (torch.zeros(3, 16, nk, hd, dtype=dtype, device=device) for _ in "kv")
    ops.reshape_and_cache(k.view(rows, nk, hd), v.view(rows, nk, hd), kc, vc, slots.to(device))
    assert torch.equal(kc.view(48, -1)[slots.to(device)].cpu(), k.cpu())
    assert torch.equal(vc.view(48, -1)[slots.to(device)].cpu(), want_v)


@pytest.mark.gpu
@pytest.mark.parametrize(("heads", "kv_heads", "hd"), [(8, 2, 128), (8, 8, 64)])
@pytest.mark.parametrize("architecture", ["llama", "mixtral"])
def test_step_of_several_rows_matches_the_cpu(architecture, heads, kv_heads, hd):
    """Prompts and decoding sequences in one batch, on both devices."""
    _need("cuda")
    from vllm_tgis_adapter_amd.engine.config import CacheConfig, EngineConfig, ModelConfig
    from vllm_tgis_adapter_amd.engine.worker import Worker

    mc = ModelConfig(model="slices", architecture=architecture, vocab_size=512, hidden_size=256,
                     intermediate_size=256, num_layers=2, num_heads=heads,
                     num_kv_heads=kv_heads, head_dim=hd, max_model_len=128, dtype=torch.float32,
                     num_experts=4 if architecture == "mixtral" else 0, num_experts_per_tok=2)

    def worker(device):
        w = Worker(EngineConfig(model_config=mc, cache_config=CacheConfig(num_gpu_blocks=16),
                                device=device, enforce_eager=True))
        w.init_kv_cache()
        return w

    here, there = worker("cpu"), worker("cuda")
    there.model.load_state_dict({k: v.cuda() for k, v in here.model.state_dict().items()})
    g = torch.Generator().manual_seed(1)
    for a, b in zip(here.kv_caches, there.kv_caches):
        for x, y in zip(a, b):
            y.copy_(x.normal_(generator=g))
    ids = torch.randint(0, 512, (5 + 20 + 2,), generator=g).tolist()
    batch = dict(
        token_ids=ids, positions=[*range(5), *range(3, 23), 30, 17],
        slot_mapping=[*range(5), *range(16 + 3, 16 + 16), *range(32, 32 + 7), 64 + 14, 96 + 1],
        qsl=[0, 5, 25], prefill_seq_lens=[5, 23], prefill_tables=[[0], [1, 2]],
        decode_seq_lens=[31, 18], decode_tables=[[3, 4], [5, 6]],
        logit_rows=list(range(27)), num_sample_rows=27, lora_ids=None, state_slots=None)
    want, got = here.execute_batch(batch), there.execute_batch(batch).cpu()
    # float32 throughout, sums in another order
    assert (got - want).norm() <= 1e-4 * want.norm()
    for a, b in zip(here.kv_caches, there.kv_caches):
        for x, y in zip(a, b):
            torch.testing.assert_close(y.cpu(), x, atol=1e-4, rtol=1e-4)
