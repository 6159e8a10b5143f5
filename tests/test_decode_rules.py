"""Whether decode attention gives a wave a key head of short sequences: a function of shapes, which needs
no GPU."""

from __future__ import annotations

import pytest

ops = pytest.importorskip("vllm_tgis_adapter_amd.ops")
if not ops.has_native():
    pytest.skip("the extension is not built", allow_module_level=True)


# sequences from which on up to two tiles are, and four
@pytest.mark.parametrize(("kvh", "group", "dim", "fp8", "two", "four"), [
    (8, 4, 128, False, 80, 192), (8, 8, 128, False, 80, 192), (8, 4, 128, True, 112, 192),
    (8, 4, 64, False, 160, 256), (8, 4, 64, True, 160, 256), (32, 1, 128, False, 80, 96),
    (12, 1, 64, False, 112, 256), (8, 2, 128, False, 320, 384)])
def test_heads_that_are_a_waves(kvh, group, dim, fp8, two, four):
    def tiles(nseq):
        return ops._C.decode_alone_tiles(nseq, kvh, group, dim, fp8)

    assert [tiles(1), tiles(two - 1), tiles(two)] == [-1, -1, 2]
    assert [tiles(four - 1), tiles(four), tiles(4096)] == [2, 4, 4]


def test_key_heads_that_are_no_whole_workgroups():
    assert {ops._C.decode_alone_tiles(4096, kvh, 4, 128, False) for kvh in (1, 2, 3, 6, 10)} == {-1}
