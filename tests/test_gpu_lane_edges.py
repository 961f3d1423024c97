"""One-row decode at head dimensions 64 and 128 (kvx_decode_small.hip) and verify lanes of more than 32 fused rows
(kvx_verify.hip, kvx_decode_int4.hip) at the ends of the numbers: tokens with infinite elements that a row does not
see, scores that are no number, values and queries beyond fp16's range, a score scale of the caller's."""
import numpy as np
import pytest
import torch

from oracle import kvoracle as ko
from richengine_amd import kvx
import gpulib as Gp
import kvtestlib as T
import test_gpu_attention as A

pytestmark = pytest.mark.gpu

# (KV heads, group, head dimension), rows, lanes, splits; 3328 waves: two int4 heads to a wave
DECODE = [((8, 4, 64), 1, 2, 3), ((2, 8, 128), 1, 2, 5), ((3, 16, 64), 1, 1, 1), ((8, 4, 64), 1, 32, 13)]
VERIFY = [((4, 6, 256), 8, 2, 3), ((4, 6, 256), 16, 2, 5), ((2, 16, 256), 8, 1, 1)]
COMMITTED = 420  # 421, 428 and 436 tokens: a last page partly filled


class Lanes:
    """`lanes` lanes over one sequence of COMMITTED tokens and `rows` behind them, drawn unit normal;
    `change(keys, values, queries)` ([H, tokens, D] twice and [lanes, H, rows, G, D], floats) may rewrite them before
    they are stored.  One more token lies in the last page behind the rows."""

    def __init__(self, layout, fmt, rows, lanes, splits, change=None, masks=None, score_scale=0.0):
        self.layout, self.fmt, self.rows, self.lanes, self.splits = layout, fmt, rows, lanes, splits
        self.score_scale = score_scale
        H, G, D = layout
        tokens = COMMITTED + rows
        rng = np.random.default_rng(tokens + D)
        k, v = (rng.standard_normal((H, tokens + 1, D)).astype(np.float32) for _ in range(2))
        q = rng.standard_normal((lanes, H, rows, G, D)).astype(np.float32)
        if change:
            change(k, v, q)
        self.entries = (tokens + 31) // 32
        self.tw = Gp.Twin(fmt, H, D, 2, self.entries)
        self.th, self.td = self.tw.tables(self.tw.pages(self.entries, seed=tokens))
        stride = 32 * self.entries
        ck, cv = T.chunk_buffers(k, v, stride)
        kvx.append(self.tw.dev, 1, Gp.dev(ck), Gp.dev(cv), [self.td], [kvx.ChunkParams(0, tokens + 1, stride, self.entries)],
                   H * stride * D)
        torch.cuda.synchronize()
        self.tw.download()
        self.stride = 1 if rows == 1 else 32
        self.q = np.zeros((lanes, H, self.stride, G, D), dtype=np.uint16)
        self.q[:, :, :rows] = ko.f32_to_bf16(q).reshape(q.shape)
        self.masks = None if masks is None else np.repeat(masks[None], lanes, 0)

    def output(self):
        H, G, D = self.layout
        params = [kvx.VerifyParams(COMMITTED, self.entries, kvx.KvLayer(), self.splits, self.splits, self.rows, self.rows,
                                   self.score_scale)] * self.lanes
        out = torch.full(self.q.shape, 0x5A5A, dtype=torch.int16, device="cuda")
        ws = torch.empty(kvx.attend_workspace_bytes(self.tw.dev, params, H * G), dtype=torch.uint8, device="cuda")
        args = (self.tw.dev, 1, H * G, Gp.dev(self.q), out, [self.td] * self.lanes, params)
        if self.rows == 1:
            kvx.attend_decode(*args, self.stride, ws)
        else:
            kvx.attend_verify(*args, None if self.masks is None else Gp.dev(self.masks), self.stride, ws)
        torch.cuda.synchronize()
        return Gp.host_u16(out)[:, :, :self.rows]

    def check(self, label):
        H, G, D = self.layout
        params = [ko.VerifyParams(COMMITTED, self.entries, self.tw.host.layer(1), self.splits, 128, self.rows, self.rows,
                                  self.score_scale)] * self.lanes
        q = np.zeros((self.lanes, H, 32, G, D), dtype=np.uint16)
        q[:, :, :self.rows] = self.q[:, :, :self.rows]
        n, want, want32 = ko.attend_verify(self.fmt, H, G, D, q, [self.th] * self.lanes, params)
        assert n == self.lanes
        described = Gp.lanes_explainer(self.fmt, H, G, D, q, [self.th] * self.lanes, self.tw.host.layer(1),
                                       [COMMITTED] * self.lanes, self.rows, [self.splits] * self.lanes, self.rows)
        Gp.check_attention(self.output(), want[:, :, :self.rows], want32[:, :, :self.rows],
                           np.ones((self.lanes, H, self.rows), dtype=bool), A.tol(self.fmt), label,
                           explain=lambda index: dict(described(index), score_scale=self.score_scale))

    def close(self):
        self.tw.close()


def spoiled_and_clean(layout, fmt, rows, lanes, splits, spoil, **more):
    outputs = []
    for change in (spoil, None):
        case = Lanes(layout, fmt, rows, lanes, splits, change, **more)
        outputs.append(case.output())
        case.close()
    assert np.isfinite(ko.bf16_to_f32(outputs[1].copy())).all()
    return outputs


def dims_that_stay(layout, fmt):
    """An element that is itself no number, on bf16 and e4m3 pages, reaches its own dimension of the rows of its page."""
    others = np.ones(layout[2], dtype=bool)
    others[5] = fmt in (ko.INT4, ko.INT8)
    return others


@pytest.mark.parametrize("layout,rows,lanes,splits", DECODE + VERIFY)
@pytest.mark.parametrize("fmt", A.FORMATS)
def test_what_lies_behind_the_visible_tokens_reaches_no_row(layout, rows, lanes, splits, fmt):
    """The slot behind the last row holds a token with an infinite element, stored with an infinite scale."""
    def spoil(k, v, q):
        k[:, COMMITTED + rows, 5] = v[:, COMMITTED + rows, 5] = np.inf

    spoiled, clean = spoiled_and_clean(layout, fmt, rows, lanes, splits, spoil)
    others = dims_that_stay(layout, fmt)
    assert np.array_equal(spoiled[..., others], clean[..., others])


@pytest.mark.parametrize("layout,rows,lanes,splits", VERIFY)
@pytest.mark.parametrize("fmt", A.FORMATS)
@pytest.mark.parametrize("tree", [False, True])
def test_a_row_that_is_not_seen_reaches_no_other(layout, rows, lanes, splits, fmt, tree):
    """One of the lane's own rows has an infinite element: in a chain the rows before it, in a tree (it is a leaf
    beside the path) every other row."""
    if tree and fmt == ko.FP8:
        pytest.skip("tree verify has no fp8 kernels")
    row = 2 * rows // 3
    parents = [-1] + [i - 1 if i - 1 != row else row - 1 for i in range(1, rows)]
    masks = np.zeros(rows, dtype=np.uint32)
    masks[:] = A.tree_masks(parents)

    def spoil(k, v, q):
        k[:, COMMITTED + row, 5] = v[:, COMMITTED + row, 5] = np.inf

    spoiled, clean = spoiled_and_clean(layout, fmt, rows, lanes, splits, spoil, masks=masks if tree else None)
    others = dims_that_stay(layout, fmt)
    unseen = [r for r in range(rows) if (r != row if tree else r < row)]
    assert np.array_equal(spoiled[:, :, unseen][..., others], clean[:, :, unseen][..., others])


@pytest.mark.parametrize("layout,rows,lanes,splits,fmt", [(*case, fmt) for case in DECODE + VERIFY for fmt in A.FORMATS
                                                          if case not in VERIFY or fmt != ko.INT4])
def test_a_score_that_is_no_number_leaves_no_row_and_stays_in_its_head(layout, rows, lanes, splits, fmt):
    """A key of one head with an infinite element against queries that are 0 there: no row of that head is left, and
    the other heads' have their bits.  (int4 verify lanes are left out: their codes are multiplied with a bias, of
    which the products keep a rest, so that such a score can also be infinite, and the token has weight 0.)"""
    def spoil(k, v, q):
        q[..., 5] = 0.0
        k[0, COMMITTED // 2, 5] = np.inf

    def clean(k, v, q):
        q[..., 5] = 0.0

    outputs = []
    for change in (spoil, clean):
        case = Lanes(layout, fmt, rows, lanes, splits, change)
        outputs.append(case.output())
        case.close()
    assert not outputs[0][:, 0].any()
    assert np.array_equal(outputs[0][:, 1:], outputs[1][:, 1:]) and outputs[1].any(axis=-1).all()


@pytest.mark.parametrize("layout,rows,lanes,splits", DECODE + VERIFY)
@pytest.mark.parametrize("fmt", A.FORMATS)
def test_small_values_large_queries_and_a_score_scale_match_the_oracle(layout, rows, lanes, splits, fmt):
    def small(k, v, q):
        v *= 1e-3

    def large(k, v, q):
        q *= 1e5
        k *= 1e-5

    cases = [("small values", small, 0.0), ("score scale", None, 0.11)]
    if fmt != ko.FP8:  # (the fp8 tile's queries are fp16)
        cases.append(("large queries", large, 0.0))
    for label, change, score_scale in cases:
        label = f"{label} layout={layout} rows={rows} lanes={lanes} fmt={fmt}"
        print(label, flush=True)
        case = Lanes(layout, fmt, rows, lanes, splits, change, score_scale=score_scale)
        case.check(label)
        case.close()
