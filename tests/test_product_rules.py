"""Which kernel, tile and cut of K a product gets: functions of its sizes, which need no GPU."""

from __future__ import annotations

import pytest

ops = pytest.importorskip("vllm_tgis_adapter_amd.ops")
if not ops.has_native():
    pytest.skip("the extension is not built", allow_module_level=True)

# 16-row tiles of x and 64-column blocks of W of every panel of int8 products
PANELS = [(5, 1), (5, 2), (6, 2), (8, 1), (8, 2), (8, 2), (10, 2), (10, 4)]


@pytest.mark.parametrize("k", [13 << 20, 14 << 20, (1 << 24) - 128])
@pytest.mark.parametrize("n", [512, 2048, 4096, 16384])
def test_int8_panels_lie_inside_32_bits(n, k):
    """Rows of a panel are found by 32-bit offsets up to the longest K that is taken."""
    for m in (65, 129, 160, 257, 300, 513, 1025, 1200):
        plan = ops._C.gemm_panel_plan(m, n, k)
        assert plan > 1
        rows, cols = PANELS[(plan >> 8) - 1]
        assert 16 * rows * k * 2 < 1 << 32 and 64 * cols * k < 1 << 32
