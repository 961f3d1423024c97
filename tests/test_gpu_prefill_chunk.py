"""Chunks that run as workgroups of 256 fused rows sharing their pages (kvx_prefill.hip): the sizes
where a workgroup, a wave or a tile is partly filled, every format and head dimension, one split
(rows written directly) and several (merged), histories on and off a page boundary, held to the
oracle at the bar of every other prefill test (2e-3 a row, bf16 rounding of the row alone being
1.6e-3 to 2e-3)."""
import pytest

import test_gpu_attention as A
from test_gpu_prefill_small_groups import layout  # noqa: F401

pytestmark = pytest.mark.gpu

# (KV heads, group, head dimension): (committed, rows, splits).  256 fused rows to a workgroup, 32 to
# a wave; more work items than the rule's line, or one split at head dimension 256.
CASES = {
    (4, 6, 256): [(0, 1, 1), (31, 9, 1), (70, 43, 1), (512, 264, 8), (500, 301, 7)],
    (2, 16, 256): [(40, 16, 1), (64, 17, 1), (300, 130, 10)],
    (1, 1, 256): [(95, 257, 1)],
    (2, 8, 128): [(1024, 129, 32), (1003, 320, 8)],
    (3, 5, 128): [(1100, 90, 32)],
    (8, 4, 64): [(1024, 65, 32), (777, 131, 9)],
    (2, 13, 64): [(1090, 61, 32)],
}


@pytest.mark.parametrize("fmt", A.FORMATS)
@pytest.mark.parametrize("layout", sorted(CASES), indirect=True)
def test_shared_pages_match_the_oracle(layout, fmt):  # noqa: F811
    for committed, rows, splits in CASES[layout]:
        print(f"chunk layout={layout} fmt={fmt} committed={committed} rows={rows} splits={splits}", flush=True)
        A.prefill_case(fmt, committed, rows, forced_splits=splits)
