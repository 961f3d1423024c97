"""kvx_prefill_plan_for is a function of the tiles: at head dimension 256 kvx_prefill_plan_batch's count, at 64 and
128 the fewest splits that make 4096 workgroups of tiles.  Weights are rounded relative to the running maximum of
the split they fall in, so a count that moves moves the rows of every engine that plans with it."""
import ctypes as C

import pytest

from richengine_amd import kvx

LAYOUTS = {"d256": (4, 6, 256), "d128": (2, 8, 128), "d64": (8, 4, 64)}
FORMATS = {"int4": kvx.INT4, "int8": kvx.INT8, "fp8": kvx.FP8, "bf16": kvx.BF16}


def layout_of(layout, fmt):
    heads, _, dim = LAYOUTS[layout]
    return kvx.Layout(1, heads, dim, FORMATS[fmt], 0.0)


def plan(layout, fmt, committed, rows, sequences=1):
    heads, group, _ = LAYOUTS[layout]
    of = layout_of(layout, fmt)
    return kvx.lib().kvx_prefill_plan_for(C.byref(of), committed, rows, heads * group, sequences)


@pytest.mark.parametrize("fmt", sorted(FORMATS))
def test_head_dimension_256_is_the_batch_plan(fmt):
    for committed in (0, 384, 1000, 4096, 16384, 100_000):
        for rows in (1, 33, 40, 63, 64, 255, 777, 2048):
            for sequences in (1, 2, 4, 16, 32):
                want = kvx.prefill_plan(committed, rows, 4, 24, FORMATS[fmt], sequences)
                assert plan("d256", fmt, committed, rows, sequences) == want


@pytest.mark.parametrize("fmt", ("bf16", "int8"))
def test_batches_of_short_chunks_run_in_one_split(fmt):
    # (63 bf16 rows of 32 sequences after 8256 tokens in three splits, tile by tile: 2490 us a layer for 575)
    for rows in (33, 40, 63):
        for sequences in (16, 32):
            assert plan("d256", fmt, 8256, rows, sequences) == 1


@pytest.mark.parametrize("layout", ("d128", "d64"))
@pytest.mark.parametrize("fmt", sorted(FORMATS))
def test_head_dimensions_64_and_128_make_4096_workgroups_of_tiles(layout, fmt):
    heads, group, _ = LAYOUTS[layout]
    of = layout_of(layout, fmt)
    for committed in (0, 288, 1000, 6144, 16384):
        for rows in (33, 64, 256, 910, 2048):
            most = min(32, max(1, (committed + rows // 2 + 31) // 32 // 4))
            for splits in range(1, most + 1):
                together = kvx.lib().kvx_debug_prefill_tiles_together(C.byref(of), heads * group, committed, rows, splits)
                if -(-((rows + 7) // 8) // together) * heads * splits >= 4096:
                    break
            for sequences in (1, 2, 32):
                assert plan(layout, fmt, committed, rows, sequences) == splits


def test_sizes_beyond_the_limits_and_any_number_of_sequences():
    for committed, rows in ((0xFFFFFFFF, 64), (0, 0xFFFFFFFF), (0, 0), (1 << 20, 4096)):
        for layout in LAYOUTS:
            assert 0 <= plan(layout, "bf16", committed, rows) <= 32
    for sequences in (1000, 1 << 20, 0xFFFFFFFF):
        for layout in LAYOUTS:
            assert 1 <= plan(layout, "bf16", 16384, 2048, sequences) <= 32
