"""Chunks that run as workgroups of 256 fused rows sharing their pages (kvx_prefill.hip): the sizes
where a workgroup, a wave or a tile is partly filled, every format and head dimension, one split
(rows written directly) and several (merged), histories on and off a page boundary, held to the
oracle at the bar of every other prefill test (2e-3 a row, bf16 rounding of the row alone being
1.6e-3 to 2e-3)."""
import ctypes as C

import numpy as np
import pytest
import torch

from oracle import kvoracle as ko
from richengine_amd import kvx
import gpulib as Gp
import kvtestlib as T
import test_gpu_attention as A
import test_gpu_prefill_batch as B
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


def by_chunk(layout, fmt, committed, rows, splits):
    """Whether the call runs as workgroups of 256 fused rows at all."""
    H, G, D = layout
    return bool(kvx.lib().kvx_debug_prefill_by_chunk(C.byref(kvx.Layout(1, H, D, fmt, 0.0)), H * G, committed, rows, splits))


def tile_by_tile(layout, fmt, splits):
    """Of the cases of this file: int4 and, under a group of one head, e4m3 pages in one split at 256."""
    return layout[2] == 256 and splits == 1 and (fmt == ko.INT4 or (fmt == ko.FP8 and layout[1] == 1))


def test_the_cases_run_as_workgroups():
    cases = [(layout, *case) for layout in CASES for case in CASES[layout]] + SHARED
    for fmt in A.FORMATS:
        for layout, committed, rows, splits in cases:
            assert by_chunk(layout, fmt, committed, rows, splits) != tile_by_tile(layout, fmt, splits)


class Chunk:
    """A sequence of `committed` tokens and a chunk of `rows` behind them, drawn unit normal;
    `change(keys, values, queries)` ([H, tokens, D] twice and [H, rows, G, D], floats) may rewrite them
    before they are stored.  `stale` more tokens lie in the last page behind the chunk."""

    def __init__(self, layout, fmt, committed, rows, splits, change=None, stale=0, score_scale=0.0):
        self.layout, self.fmt, self.committed, self.rows, self.splits = layout, fmt, committed, rows, splits
        H, G, D = layout
        tokens = committed + rows
        assert stale <= -tokens % 32
        rng = np.random.default_rng(tokens)
        k, v = (rng.standard_normal((H, tokens + stale, D)).astype(np.float32) for _ in range(2))
        q = rng.standard_normal((H, rows, G, D)).astype(np.float32)
        if change:
            change(k, v, q)
        self.tw = Gp.Twin(fmt, H, D, 2, (tokens + 31) // 32)
        self.pages = self.tw.pages((tokens + 31) // 32, seed=tokens)
        self.th, self.td = self.tw.tables(self.pages)
        stride = (tokens + stale + 31) // 32 * 32
        ck, cv = T.chunk_buffers(k, v, stride)
        kvx.append(self.tw.dev, 1, Gp.dev(ck), Gp.dev(cv), [self.td],
                   [kvx.ChunkParams(0, tokens + stale, stride, len(self.pages))], H * stride * D)
        torch.cuda.synchronize()
        self.tw.download()
        self.stride = (rows + 31) // 32 * 32
        self.q = np.zeros((H, self.stride, G, D), dtype=np.uint16)
        self.q[:, :rows] = ko.f32_to_bf16(q).reshape(q.shape)
        self.score_scale = score_scale

    def output(self):
        H, G, D = self.layout
        out = torch.full((H, self.stride, G, D), 0x5A5A, dtype=torch.int16, device="cuda")
        ws = torch.empty(kvx.prefill_workspace_bytes(self.tw.dev, self.rows, H * G, self.splits), dtype=torch.uint8,
                         device="cuda")
        kvx.attend_prefill(self.tw.dev, 1, H * G, Gp.dev(self.q), out, self.td,
                           kvx.PrefillParams(self.committed, self.rows, self.stride, len(self.pages), kvx.KvLayer(),
                                             self.splits, self.score_scale), ws)
        torch.cuda.synchronize()
        return Gp.host_u16(out)[:, :self.rows]

    def check(self, label):
        """The rows against the oracle's, at the bar of every other prefill test."""
        H, G, D = self.layout
        params = ko.PrefillParams(self.committed, self.rows, self.stride, len(self.pages), self.tw.host.layer(1),
                                  self.splits, self.score_scale)
        ok, want, want32 = ko.attend_prefill(self.fmt, H, G, D, self.q, self.th, params)
        assert ok == 1
        explain = Gp.prefill_explainer(self.fmt, H, G, D, self.q, self.th, self.tw.host.layer(1), self.committed,
                                       self.rows, self.splits)
        if self.score_scale:
            described = explain
            explain = lambda index: dict(described(index), score_scale=self.score_scale)  # noqa: E731
        Gp.check_attention(self.output(), want[:, :self.rows], want32[:, :self.rows],
                           np.ones((H, self.rows), dtype=bool), A.tol(self.fmt), label, explain=explain)

    def close(self):
        self.tw.close()


# a chunk of each head dimension that shares its pages, in one split and in several
SHARED = [((4, 6, 256), 70, 43, 1), ((4, 6, 256), 500, 301, 7), ((2, 8, 128), 1003, 320, 8),
          ((8, 4, 64), 777, 131, 9), ((8, 4, 64), 40, 1027, 1), ((4, 5, 128), 0, 2011, 1)]


@pytest.mark.parametrize("layout,committed,rows,splits", SHARED[1:4])
@pytest.mark.parametrize("fmt", A.FORMATS)
def test_small_values_keep_their_bits(layout, committed, rows, splits, fmt):
    """A weight carries its token's value scale: with values of 1e-3 the products lie below 2^-14,
    where fp16 runs out of places."""
    def change(k, v, q):
        v *= 1e-3

    print(f"small values layout={layout} fmt={fmt}", flush=True)
    case = Chunk(layout, fmt, committed, rows, splits, change)
    case.check(f"small values layout={layout} fmt={fmt}")
    case.close()


@pytest.mark.parametrize("layout,committed,rows,splits", SHARED[1:4])
@pytest.mark.parametrize("fmt", [ko.INT4, ko.INT8, ko.BF16])   # (the fp8 tile's queries are fp16)
def test_large_queries_stay_finite(layout, committed, rows, splits, fmt):
    """Queries beyond fp16's 65504, on keys as much smaller."""
    def change(k, v, q):
        q *= 1e5
        k *= 1e-5

    print(f"large queries layout={layout} fmt={fmt}", flush=True)
    case = Chunk(layout, fmt, committed, rows, splits, change)
    case.check(f"large queries layout={layout} fmt={fmt}")
    case.close()


def spoiled_and_clean(layout, fmt, committed, rows, splits, row):
    """The rows of a chunk whose row `row` (rows: the first token behind the chunk, in the same page) has an
    infinite element 5 in its key and its value, and the rows of the same chunk without it."""
    stale = min(1, -(committed + rows) % 32)

    def spoil(k, v, q):
        k[:, committed + row, 5] = v[:, committed + row, 5] = np.inf

    outputs = []
    for change in (spoil, None):
        case = Chunk(layout, fmt, committed, rows, splits, change, stale=stale)
        outputs.append(case.output())
        case.close()
    return outputs


@pytest.mark.parametrize("layout,committed,rows,splits", SHARED)
@pytest.mark.parametrize("fmt", A.FORMATS)
def test_a_token_that_a_row_does_not_see_does_not_reach_it(layout, committed, rows, splits, fmt):
    """A token with an infinite element is stored with an infinite scale; neither a row before it in the chunk
    nor, once its page is another sequence's, a row that ends before it may change by it.  (An element that
    is itself no number, on bf16 and e4m3 pages, does reach its own dimension of the rows of its page.)"""
    others = np.arange(layout[2]) != 5
    if fmt in (ko.INT4, ko.INT8):
        others[:] = True
    for row in (2 * rows // 3, rows):
        if row == rows and (committed + rows) % 32 == 0:
            continue
        print(f"unseen token layout={layout} fmt={fmt} row={row} of {rows}", flush=True)
        spoiled, clean = spoiled_and_clean(layout, fmt, committed, rows, splits, row)
        assert np.array_equal(spoiled[:, :row][..., others], clean[:, :row][..., others])


@pytest.mark.parametrize("layout,committed,rows,splits", SHARED + [((3, 5, 128), 1100, 90, 32), ((2, 13, 64), 1090, 61, 32)])
@pytest.mark.parametrize("fmt", A.FORMATS)
def test_an_element_that_is_no_number_stays_in_its_pages(layout, committed, rows, splits, fmt):
    """The first token of a page that begins in the chunk has an infinite element: rows whose tiles end before
    that page have the bits that they have without it."""
    first = -committed % 32
    for row in {first, first + 32 * ((rows - 1 - first) // 32)}:
        print(f"no number layout={layout} fmt={fmt} row={row} of {rows}", flush=True)
        spoiled, clean = spoiled_and_clean(layout, fmt, committed, rows, splits, row)
        before = row // 8 * 8
        assert before == 0 or np.isfinite(ko.bf16_to_f32(clean[:, :before].copy())).all()
        assert np.array_equal(spoiled[:, :before], clean[:, :before])


@pytest.mark.parametrize("fmt,layout,committed,rows,splits",
                         [(f, *c) for f in A.FORMATS for c in SHARED if not tile_by_tile(c[0], f, c[3])])
def test_a_score_that_is_no_number_leaves_no_row(layout, committed, rows, splits, fmt):
    """A key with an infinite element against queries that are 0 there: the score is no number, nor is the sum of
    the weights, and such a row is written as zeros, in one split and in several, at every head dimension."""
    row = 2 * rows // 3

    def change(k, v, q):
        k[:, committed + row, 5] = np.inf
        q[..., 5] = 0.0

    print(f"no score layout={layout} fmt={fmt} row={row} of {rows}", flush=True)
    case = Chunk(layout, fmt, committed, rows, splits, change)
    got = case.output()
    assert not got[:, row:].any()
    assert got[:, :row].any(axis=-1).all() and np.isfinite(ko.bf16_to_f32(got[:, :row].copy())).all()
    case.close()


@pytest.mark.parametrize("layout,committed,rows,splits", SHARED[1:])
def test_int4_keys_near_the_largest_number(layout, committed, rows, splits):
    """A key element of 2e38 against queries that are 0 there: every other code of the key is 0, and so is its score,
    whatever the code unit and the score scale are multiplied into."""
    def change(k, v, q):
        k[:, committed // 2, 5] = 2e38
        q[..., 5] = 0.0

    print(f"large key layout={layout} splits={splits}", flush=True)
    case = Chunk(layout, ko.INT4, committed, rows, splits, change)
    case.check(f"large key layout={layout}")
    case.close()


@pytest.mark.parametrize("layout,committed,rows,splits", SHARED[4:])
@pytest.mark.parametrize("fmt", A.FORMATS)
def test_one_split_at_64_and_128_is_written_directly(layout, committed, rows, splits, fmt):
    print(f"one split layout={layout} fmt={fmt}", flush=True)
    case = Chunk(layout, fmt, committed, rows, splits)
    case.check(f"one split layout={layout} fmt={fmt}")
    case.close()


@pytest.mark.parametrize("layout,committed,rows,splits", SHARED[:4])
@pytest.mark.parametrize("fmt", A.FORMATS)
def test_a_score_scale_of_the_callers(layout, committed, rows, splits, fmt):
    """No power of two and not the default; at 64 and 256 it goes into the staged key scales."""
    print(f"score scale layout={layout} fmt={fmt}", flush=True)
    case = Chunk(layout, fmt, committed, rows, splits, score_scale=0.11)
    case.check(f"score scale layout={layout} fmt={fmt}")
    case.close()


# the sequences' histories, rows and splits; the last two of sequences that go either way
BATCHES = [((2, 8, 128), (1003, 640, 1024), 320, 8), ((8, 4, 64), (777, 512, 1000), 131, 9),
           ((3, 5, 128), (1100, 1500, 1088), 90, 32), ((4, 6, 256), (500, 512, 1000), 301, 7),
           ((8, 4, 64), tuple(512 + 32 * (i % 5) + i for i in range(35)), 66, 16),
           ((8, 4, 64), (0, 777, 64, 32, 1024, 0), 131, 9), ((4, 6, 256), (512, 500, 1000, 480, 1024, 1030), 64, 3)]


@pytest.mark.parametrize("layout,committed,rows,splits", BATCHES)
@pytest.mark.parametrize("fmt", A.FORMATS)
def test_a_batch_has_the_bits_of_its_sequences_alone(monkeypatch, layout, committed, rows, splits, fmt):
    """Equal chunks share the workgroups' launches, 32 sequences at a time, whatever their histories; those that
    run tile by tile do not disturb them."""
    for name, value in zip(("H", "G", "D", "QH"), (*layout, layout[0] * layout[1])):
        monkeypatch.setattr(B, name, value)
    ways = {by_chunk(layout, fmt, c, rows, splits) for c in committed}
    if (layout, committed, rows, splits) not in BATCHES[-2:]:
        assert ways == {True}
    else:
        assert ways == ({False} if layout[2] == 256 and fmt == ko.INT4 else {True, False})
    print(f"batch layout={layout} fmt={fmt} sequences={len(committed)} rows={rows} splits={splits}", flush=True)
    n = len(committed)
    together, alone, tw = B.run_batch(fmt, list(committed), [rows] * n, [splits] * n)
    assert np.array_equal(together, alone)
    assert (alone != 0x5A5A).any(axis=1).all()
    tw.close()
