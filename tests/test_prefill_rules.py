"""How prompt attention is cut: functions of its sizes, which need no GPU."""

from __future__ import annotations

import pytest

ops = pytest.importorskip("vllm_tgis_adapter_amd.ops")
if not ops.has_native():
    pytest.skip("the extension is not built", allow_module_level=True)


def _plan(fp8, heads, dim, prompts, tokens, past, block=16):
    plan = ops._C.prefill_tile_plan(fp8, block, prompts, *heads, dim, tokens, tokens + past)
    return plan >> 8, plan & 255


# parts that fill the chip: what few tokens leave of each stays in the caches
@pytest.mark.parametrize(("fp8", "heads", "dim", "prompts", "tokens", "past", "parts"), [
    (True, (32, 8), 128, 2, 64, 4000, 10), (True, (32, 8), 128, 4, 64, 3000, 7),
    (False, (64, 8), 128, 1, 64, 4000, 10), (False, (64, 8), 128, 1, 30, 6000, 15),
    (False, (32, 8), 64, 4, 64, 3000, 7), (False, (64, 8), 64, 2, 32, 2000, 5)])
def test_keys_are_cut_as_far_as_fills_the_chip(fp8, heads, dim, prompts, tokens, past, parts):
    assert _plan(fp8, heads, dim, prompts, tokens, past)[1] >= parts


@pytest.mark.parametrize(("heads", "dim", "prompts", "tokens", "past"), [
    ((32, 8), 128, 1, 1000, 0), ((32, 8), 64, 1, 1000, 1000), ((64, 8), 128, 1, 512, 1000)])
def test_keys_of_many_tokens_stay_whole(heads, dim, prompts, tokens, past):
    assert _plan(False, heads, dim, prompts, tokens, past) == (4, 1)


# forms within 2 % of the fastest at blocks of 24: four waves whole, or eight and the parts of the keys
@pytest.mark.parametrize(("heads", "dim", "prompts", "tokens", "past", "plans"), [
    ((32, 8), 128, 1, 1000, 0, {(4, 1), (8, 1)}), ((32, 8), 128, 8, 256, 0, {(4, 1)}),
    ((32, 8), 128, 2, 1000, 0, {(8, 1)}), ((32, 8), 128, 1, 1000, 500, {(8, 2)}),
    ((32, 8), 128, 2, 500, 1000, {(8, 2)}), ((64, 8), 128, 1, 512, 1000, {(8, 2)}),
    ((32, 8), 64, 1, 1000, 0, {(4, 1)}), ((32, 8), 64, 1, 700, 700, {(4, 1)}),
    ((32, 8), 64, 1, 512, 1000, {(8, 3), (8, 4)}), ((32, 8), 64, 2, 200, 1000, {(8, 3), (8, 4)}),
    ((32, 8), 64, 3, 1000, 0, {(8, 1)}), ((64, 8), 64, 1, 1500, 1500, {(8, 1)})])
def test_blocks_that_are_no_power_of_two(heads, dim, prompts, tokens, past, plans):
    """Lanes that find their own rows take longer for a tile, four waves more so."""
    assert _plan(False, heads, dim, prompts, tokens, past, 24) in plans
