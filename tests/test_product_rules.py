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


# the same of 4 bits
PANELS4 = [(5, 1), (5, 2), (6, 2), (8, 1), (8, 2), (5, 4), (4, 2)]


@pytest.mark.parametrize("k", [128, 2048, 14336, 13 << 20, (1 << 24) - 128])
@pytest.mark.parametrize("n", [128, 512, 768, 4096, 28672])
def test_4_bit_panels_fit(n, k):
    """Whole columns, no part of K without a group, rows of a panel inside 32 bits; a gated
    product's panels have all of K."""
    for m in (65, 129, 160, 257, 300, 513, 899, 1200):
        for plan, gated in ((ops._C.gemm_panel_plan(m, n, k, 4), False),
                            (ops._C.gemm_panel_gated_plan(m, n // 2, k, 4), True)):
            if plan <= 1:
                assert plan == (0 if gated else 1) and (gated or k <= 2048)
                continue
            (rows, cols), parts = PANELS4[(plan >> 8) - 1], plan & 255
            assert n % (64 * cols) == 0 and not (gated and parts > 1)
            assert 16 * rows * k * 2 < 1 << 32 and 64 * cols * k // 2 < 1 << 32
            groups = -(-(k // 128) // parts)
            assert (parts - 1) * groups < k // 128 <= parts * groups


@pytest.mark.parametrize("qbits", [8, 4])
def test_longest_rows_are_widened(qbits):
    """Past the longest K that the kernels take (gemm_q) only the pass over a widened matrix is left."""
    for n in (128, 512, 16384):
        assert ops._quant_rows(qbits, n, (1 << 24) - 128) >= 900
        assert ops._quant_rows(qbits, n, 1 << 24) <= 64


# of up to 64 rows
FEW_PANELS = [(2, 1), (2, 2), (3, 1), (3, 2), (4, 1), (4, 2)]


@pytest.mark.parametrize("qbits", [8, 4])
@pytest.mark.parametrize("k", [128, 2048, 14336, 28672, (1 << 24) - 128])
@pytest.mark.parametrize("n", [128, 512, 768, 4096, 28672, 57344])
def test_panels_of_few_rows_fit(qbits, n, k):
    """The same for these, which have all rows in one panel."""
    for m in (2, 4, 9, 16, 17, 32, 33, 48, 49, 64):
        for plan, gated in ((ops._C.gemm_panel_few_plan(m, n, k, qbits), False),
                            (ops._C.gemm_panel_gated_plan(m, n // 2, k, qbits), True)):
            if plan == 0:
                continue
            (rows, cols), parts = FEW_PANELS[(plan >> 8) - 17], plan & 255
            assert 16 * rows >= m and n % (64 * cols) == 0 and not (gated and parts > 1)
            assert 16 * rows * k * 2 < 1 << 32 and 64 * cols * k < 1 << 32
            depth = -(-(k // (128 if qbits == 4 else 64)) // parts)
            assert (parts - 1) * depth < k // (128 if qbits == 4 else 64) <= parts * depth
    assert ops._C.gemm_panel_few_plan(1, n, k, qbits) == 0
    assert ops._C.gemm_panel_gated_plan(1, n // 2, k, qbits) == 0


@pytest.mark.parametrize(("m", "n", "k", "plans"), [
    # rounds of an XCD, of which counting the chip's took the slower: panel, parts of K
    (800, 1280, 8192, {(1, 4), (6, 4), (5, 3), (1, 2)}), (560, 1536, 4096, {(0, 3), (2, 3)}),
    (1100, 768, 4096, {(2, 3), (3, 2)})])
def test_int8_panels_are_counted_by_xcd(m, n, k, plans):
    plan = ops._C.gemm_panel_plan(m, n, k)
    assert ((plan >> 8) - 1, plan & 255) in plans


@pytest.mark.parametrize(("m", "n", "k", "tiles"), [
    (430, 768, 768, True), (1000, 768, 768, True), (1000, 128, 512, True), (1000, 3072, 768, True),
    (400, 2048, 1024, True), (640, 2048, 1024, False), (800, 3072, 768, False),
    (512, 128, 2048, False), (512, 4096, 2048, False)])
def test_int8_small_matrices(m, n, k, tiles):
    """Tiles of the whole K while they are one round."""
    assert (ops._C.gemm_panel_plan(m, n, k) == 1) == tiles


# sizes at which the model's first form was off by 4 to 25 %, and the tiles (form << 4 | parts of K)
# that measured within 4 % of the best
PLANS = [
    (96, 8192, 28672, False, {24, 36}), (128, 8192, 28672, False, {24, 36}),
    (301, 1280, 8192, False, {39, 40}), (640, 1280, 8192, False, {36}),
    (256, 8192, 8192, False, {6, 20, 34}), (340, 7168, 8192, False, {35}),
    (96, 8192, 14336, False, {36}), (384, 5120, 8192, False, {20}), (128, 2048, 4096, False, {68}),
    (160, 1536, 4096, False, {67}), (1024, 4096, 14336, False, {4}),
    (512, 4096, 14336, False, {6, 7, 20}), (56, 14336, 8192, False, {65}),
    (40, 3072, 2048, False, {67, 68}), (40, 8192, 1024, False, {65}),
    (24, 11008, 4096, False, {65}), (24, 10240, 4096, False, {51, 65, 67}),
    (224, 28672, 8192, True, {1}), (128, 3584, 4096, True, {65}),
    # columns of 64 where they fill the chip as they are, of 128 where they would be cut and two a CU
    (24, 4096, 14336, False, {68}), (24, 8192, 28672, False, {52}), (9, 5120, 28672, False, {54}),
    (17, 10240, 8192, False, {51}), (24, 14336, 14336, False, {50}), (40, 6144, 4096, False, {52}),
    (64, 8192, 8192, False, {51}), (17, 6144, 2048, False, {66}), (24, 6144, 8192, False, {66}),
    # gated, one and a half rounds of columns of 64, and more
    (17, 24576, 4096, True, {65}), (17, 24704, 4096, True, {49}), (40, 28672, 2048, True, {49})]


@pytest.mark.parametrize(("m", "n", "k", "gated", "plans"), PLANS)
def test_plans_that_measured_well(m, n, k, gated, plans):
    assert ops._C.gemm_ring_plan(m, n, k, gated) in plans


@pytest.mark.parametrize(("form", "rows", "least"), [
    (0, 256, 40), (1, 128, 40), (2, 128, 40), (3, 64, 20), (4, 64, 20)])
def test_weights_that_go_past_the_caches(form, rows, least):
    """Millions of weights from which on they do, while all rows are one tile."""
    for gated in (False, True):
        def once(m, cols):   # 10240 weights a column
            return ops._C.gemm_ring_reads_once(m, cols, 10240 // (1 + gated), form << 4 | 1, gated)

        cols = -(-least * 10**6 // 10240)
        assert once(1, cols) and once(rows, cols)
        assert not once(rows, cols - 1) and not once(rows + 1, cols)


@pytest.mark.parametrize(("m", "n", "k"), [
    (640, 8192, 28672),                                    # the library is faster
    (48, 4096, 1024), (64, 4096, 1792), (40, 2048, 1024),  # the streaming kernel is: short K
    (12, 8192, 4096), (16, 8192, 4096)])                   # a K that would be cut
def test_products_the_tiles_leave(m, n, k):
    assert not ops._C.gemm_ring_wins(m, n, k, False) and not ops._C.gemm_block_takes(m, n, k)


@pytest.mark.parametrize("gated", [False, True])
def test_plans_are_plans(gated):
    """Columns in whole tiles, no empty part, whatever the sizes."""
    bn = [256, 256, 128, 128, 64]
    for m in (1, 9, 64, 65, 129, 300, 1024, 5000):
        for n in (128, 384, 640, 1280, 4096, 28672):
            for k in (64, 128, 448, 832, 2112, 4096, 12352, 28672):
                plan = ops._C.gemm_ring_plan(m, n, k, gated)
                form, parts = plan >> 4, plan & 15
                assert (1 + gated) * n % bn[form] == 0 and 1 <= parts <= (1 if gated else 8)
                depth = -(-(k // 64) // parts)
                assert -(-(k // 64) // depth) == parts


# 0: 256 x 256, 1: 128 x 256, 2: 128 x 128; rows an expert, experts, columns of W, K
@pytest.mark.parametrize(("mean", "experts", "columns", "k", "gated", "tile"), [
    (737, 8, 28672, 4096, True, 0), (737, 8, 4096, 14336, False, 0), (125, 8, 28672, 4096, True, 0),
    (100, 8, 28672, 4096, True, 1), (249, 8, 28672, 4096, True, 0), (125, 8, 3584, 4096, True, 1),
    (230, 8, 7168, 4096, True, 0), (249, 8, 7168, 4096, True, 1), (260, 8, 7168, 4096, True, 0),
    (160, 4, 1024, 1024, True, 2), (160, 8, 2048 + 128, 4096, True, 2),
    (222, 8, 4096, 14336, False, 1), (230, 8, 4096, 14336, False, 0), (300, 8, 4096, 14336, False, 0),
    (222, 8, 4096, 3584, False, 1), (222, 16, 4096, 3584, False, 0), (222, 4, 1024, 512, False, 2),
    (400, 4, 1024, 512, False, 2), (222, 16, 2048, 2048, False, 1), (245, 16, 2048, 2048, False, 2),
    (118, 32, 2048, 1024, False, 2), (280, 32, 2048, 1024, False, 2), (420, 32, 2048, 1024, False, 0)])
def test_expert_tiles_fill_the_chip(mean, experts, columns, k, gated, tile):
    """Large tiles only where there are enough of them."""
    assert ops._C.moe_tile(mean, experts, columns, k, gated) == tile


def test_one_question_for_both_rules():
    """What linear asks says what the two rules say, the cut first, and nothing up to 64 rows."""
    for m in (1, 17, 64, 65, 129, 300, 640, 1024, 5000):
        for n in (128, 1280, 2048, 4096, 8192, 28672):
            for k in (64, 2048, 4096, 8192, 28672):
                block, ring = ops._C.gemm_block_takes(m, n, k), ops._C.gemm_ring_wins(m, n, k, False)
                want = 0 if m <= 64 else 1 if block else 2 if ring else 0
                assert ops._C.gemm_tiles_route(m, n, k) == want


def test_few_rows_are_not_asked_for():
    """Products of up to eight rows are none of the tiles', but with adapters."""
    for m in range(1, 9):
        for n in (128, 2048, 14336, 28672):
            for k in (64, 2048, 8192, 28672):
                assert not ops._tiles_take(m, n, k)


# both sides of every line, where one way is at least 4 % faster; n: of [gate; up] where it is gated
@pytest.mark.parametrize(("bits", "gated", "m", "n", "k", "panel"), [
    (8, False, 17, 1280, 8192, True), (8, False, 17, 6144, 14336, False), (8, False, 20, 57344, 7168, False),
    (8, False, 28, 57344, 7168, False), (8, False, 24, 5120, 8192, True), (8, False, 28, 768, 28672, False),
    (8, False, 17, 1280, 14336, False), (8, False, 28, 6144, 14336, True),
    (8, False, 2, 14336, 28672, False), (8, False, 2, 6144, 28672, True), (8, False, 12, 57344, 2560, False),
    (8, False, 14, 28672, 2560, True), (4, False, 2, 28672, 8192, False), (4, False, 10, 28672, 8192, True),
    (4, False, 2, 8192, 8192, True), (4, False, 8, 16384, 28672, True),
    (8, True, 2, 57344, 5120, False), (8, True, 4, 14336, 4096, True), (8, True, 6, 28672, 7168, False),
    (8, True, 3, 10240, 3584, False), (8, True, 17, 57344, 5120, False), (8, True, 32, 57344, 3584, True),
    (8, True, 17, 14336, 7168, True), (4, True, 10, 10240, 3584, False), (4, True, 4, 14336, 4096, False),
    (4, True, 12, 14336, 4096, True), (4, True, 4, 28672, 2560, True)])
def test_few_rows_take_panels_where_they_are_faster(bits, gated, m, n, k, panel):
    plan = (ops._C.gemm_panel_gated_plan(m, n // 2, k, bits) if gated
            else ops._C.gemm_panel_few_plan(m, n, k, bits))
    assert (plan > 0) == panel


# adapters of rank 8 on one row leave little to add up
@pytest.mark.parametrize(("m", "n", "k", "ranks"), [
    (1, 28672, 4096, {16, 32, 64}), (1, 16384, 2048, {16, 32, 64}), (2, 28672, 4096, {8, 16, 32, 64}),
    (1, 7168, 4096, {8, 16, 32, 64}), (1, 10240, 8192, {8, 16, 32, 64}), (1, 4096, 4096, set())])
def test_products_with_adapters_by_rank(m, n, k, ranks):
    assert {r for r in ops.LORA_RANKS if ops._lora_tiles_take(m, n, k, r)} == ranks


# waves, and those that K is dealt to: forms within 4 % of the fastest at sizes around every line of the rule
@pytest.mark.parametrize(("bits", "mode", "n", "k", "forms"), [
    (4, 0, 128, 8192, {0x88}), (4, 0, 1024, 28672, {0x88}), (4, 0, 2048, 8192, {0x84, 0x88}),
    (4, 0, 2560, 14336, {0x44, 0x88, 0x82}), (4, 0, 3072, 10240, {0x44, 0x88}),
    (4, 0, 3584, 7168, {0x84}), (4, 0, 3584, 14336, {0x82, 0x42, 0x84}), (4, 0, 3968, 14336, {0x82, 0x42, 0x84}),
    (4, 0, 4096, 8192, {0x84}), (4, 0, 4096, 14336, {0x82, 0x42}), (4, 0, 4096, 28672, {0x82}),
    (4, 0, 4224, 7168, {0x44, 0x88}), (4, 0, 4608, 7168, {0x44, 0x88}), (4, 0, 4608, 14336, {0x44}),
    (4, 0, 5120, 8192, {0x44, 0x88}), (4, 0, 5120, 14336, {0x44}), (4, 0, 5120, 28672, {0x88}),
    (4, 0, 6144, 8192, {0x42, 0x84, 0x88, 0x44}), (4, 0, 6144, 28672, {0x84}), (4, 0, 7680, 14336, {0x82}),
    (4, 0, 8192, 8192, {0x42, 0x82}), (4, 0, 8192, 28672, {0x82}), (4, 0, 9216, 8192, {0x42, 0x88}),
    (4, 0, 10240, 8192, {0x42}), (4, 0, 10240, 14336, {0x42, 0x44}), (4, 0, 14336, 8192, {0x42}),
    (4, 0, 28672, 8192, {0x42}), (4, 0, 57344, 14336, {0x41}), (4, 0, 57344, 28672, {0x82}),
    (8, 0, 256, 14336, {0x44}), (8, 0, 1280, 14336, {0x84}), (8, 0, 2560, 14336, {0x44, 0x82}),
    (8, 0, 4096, 8192, {0x84}), (8, 0, 4608, 8192, {0x44}), (8, 0, 2560, 28672, {0x84}),
    (8, 0, 3328, 20480, {0x84}), (8, 0, 8192, 28672, {0x84}),
    (8, 1, 512, 1024, {0x41, 0x42}), (8, 1, 768, 2048, {0x42}), (8, 1, 8192, 2048, {0x41}),
    (8, 1, 5120, 1280, {0x42}), (8, 1, 512, 4096, {0x44}), (8, 1, 14336, 4096, {0x42}),
    (16, 1, 768, 2048, {0x44, 0x84}), (16, 1, 3072, 1024, {0x42}), (16, 1, 2048, 1280, {0x44, 0x84}),
    (16, 1, 8192, 2048, {0x42}), (16, 0, 2176, 10240, {0x44}), (16, 0, 2048, 8192, {0x88}),
    (16, 0, 2560, 28672, {0x88}), (16, 0, 5120, 14336, {0x88}), (16, 0, 16384, 8192, {0x44, 0x84})])
def test_one_row_forms_that_measured_well(bits, mode, n, k, forms):
    assert ops._C.gemm_row_form(bits, mode, n, k) in forms


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize(("bits", "made"), [
    (16, [{0x44, 0x84, 0x88}, {0x44, 0x84, 0x42}, {0x44, 0x84, 0x88}]),
    (8, [{0x44, 0x42, 0x84}, {0x44, 0x42, 0x84, 0x41}, {0x44, 0x42, 0x84}]),
    (4, [{0x44, 0x42, 0x41, 0x82, 0x84, 0x88}, {0x44, 0x42, 0x41}, {0x44, 0x42, 0x41}])])
def test_one_row_forms_are_built(bits, mode, made):
    for n in (128, 384, 1152, 2048, 2176, 3072, 4096, 4224, 6144, 8192, 9216, 14336, 16512, 57344):
        for k in (128, 1024, 1280, 2048, 2176, 6144, 6272, 7168, 8192, 8320, 14336, 20480, 28672):
            assert ops._C.gemm_row_form(bits, mode, n, k) in made[mode]
