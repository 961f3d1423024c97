"""kvx_prefill_plan_for where chunks run as workgroups of 256 fused rows: the split count is one that runs
so, no split is shorter than 4 pages, and the sequences of a batch count as one launch."""
import ctypes as C

import pytest

from richengine_amd import kvx

LAYOUTS = {"d256": (4, 6, 256), "d128": (2, 8, 128), "d64": (8, 4, 64)}
FORMATS = {"int4": kvx.INT4, "int8": kvx.INT8, "fp8": kvx.FP8, "bf16": kvx.BF16}


def plan(layout, fmt, committed, rows, sequences=1):
    heads, group, dim = LAYOUTS[layout]
    of = kvx.Layout(1, heads, dim, FORMATS[fmt], 0.0)
    return kvx.lib().kvx_prefill_plan_for(C.byref(of), committed, rows, heads * group, sequences)


def by_chunk(layout, fmt, committed, rows, splits):
    heads, group, dim = LAYOUTS[layout]
    of = kvx.Layout(1, heads, dim, FORMATS[fmt], 0.0)
    return kvx.lib().kvx_debug_prefill_by_chunk(C.byref(of), heads * group, committed, rows, splits)


@pytest.mark.parametrize("layout", sorted(LAYOUTS))
@pytest.mark.parametrize("fmt", ("int8", "fp8", "bf16"))
def test_the_planned_count_runs_as_workgroups_that_share_their_pages(layout, fmt):
    for committed in (0, 32, 512, 1000, 4096, 16384, 100_000):
        for rows in (64, 65, 255, 777, 2048):
            for sequences in (1, 2, 3, 32):
                splits = plan(layout, fmt, committed, rows, sequences)
                assert 1 <= splits <= 32
                mean = committed - committed % 32 if sequences > 1 else committed
                possible = [s for s in range(1, 33) if by_chunk(layout, fmt, mean, rows, s)
                            and (s == 1 or s * 4 <= (committed + rows // 2 + 31) // 32)]
                if possible:
                    assert by_chunk(layout, fmt, mean, rows, splits)


def test_counts_of_full_rounds():
    assert plan("d256", "bf16", 16384, 2048) == 4        # 192 workgroups a split: three full rounds of 256
    assert plan("d256", "bf16", 16384, 2048, 4) == 1     # 768
    assert plan("d256", "int8", 4032, 366, 2) == 3       # 72 a split
    assert plan("d128", "fp8", 6144, 256, 2) == 16       # 32 a split: two rounds (8 splits would run tile by tile)
    assert plan("d64", "bf16", 8192, 256) == 16          # 32 a split, 512 at a time
    assert plan("d64", "int4", 288, 910, 4) == 2


@pytest.mark.parametrize("fmt", sorted(FORMATS))
def test_few_rows_at_head_dimension_256_keep_the_tiles_count_or_three(fmt):
    for committed in (0, 100, 384, 4096, 65536):
        for rows in (1, 33, 63):
            old = kvx.prefill_plan(committed, rows, 4, 24, FORMATS[fmt])
            pages = (committed + rows // 2 + 31) // 32
            assert plan("d256", fmt, committed, rows) == max(old, min(3, max(1, pages // 4)))


def test_int4_alone_is_planned_by_tiles():
    for committed, rows in ((0, 64), (384, 300), (16384, 2048)):
        assert plan("d256", "int4", committed, rows) == kvx.prefill_plan(committed, rows, 4, 24, kvx.INT4)
        for layout in ("d128", "d64"):  # the fewest splits that make 4096 workgroups of tiles, none below 4 pages
            assert plan(layout, "int4", committed, rows) <= max(1, (committed + rows // 2 + 31) // 32 // 4)


def test_sizes_beyond_the_limits_keep_the_tiles_count():
    for committed, rows in ((0xFFFFFFFF, 64), (0, 0xFFFFFFFF), (0, 0), (1 << 20, 4096)):
        for layout in LAYOUTS:
            assert 0 <= plan(layout, "bf16", committed, rows) <= 32


def test_any_number_of_sequences_is_planned():
    for sequences in (1000, 1 << 20, 0xFFFFFFFF):
        for layout in LAYOUTS:
            assert 1 <= plan(layout, "bf16", 16384, 2048, sequences) <= 32
