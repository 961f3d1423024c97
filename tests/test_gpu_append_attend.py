"""kv_append_attend_decode where the attention kernel stores the step's token itself: the page bytes are those
of kv_append and the rows those of kv_attend_decode, for more lanes than a launch holds, splits of one page
(the token's page is the first a wave loads) and long ones, first and last slots of a page, every group."""
import numpy as np
import pytest
import torch

from oracle import kvoracle as ko
from richengine_amd import kvx
import gpulib as Gp
import kvtestlib as T
import test_gpu_attention as A

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,group,dim", [(4, 6, 256), (3, 1, 256), (1, 16, 256),
                                             (8, 4, 64), (2, 8, 128), (3, 5, 64), (5, 3, 128), (1, 16, 128), (6, 1, 64),
                                             (16, 2, 64)])  # splits of a page: two int4 heads to a wave
@pytest.mark.parametrize("fmt", A.FORMATS)
@pytest.mark.parametrize("one_page_splits", [False, True])
def test_token_stored_by_the_attention_kernel(heads, group, dim, fmt, one_page_splits):
    committed = [0, 31, 32, 63, 700, 1023, 33, 95, 96, 352] + [int(x) for x in np.random.default_rng(5).integers(0, 500, 26)]
    lanes, total = len(committed), [c + 1 for c in committed]
    counts = [(t + 31) // 32 for t in total]
    tw = Gp.Twin(fmt, heads, dim, 2, sum(counts))
    ids, at, dts, hts = tw.pages(sum(counts), 9), 0, [], []
    rng = np.random.default_rng(6)
    for lane, n in enumerate(counts):
        th, td = tw.tables(ids[at:at + n])
        at += n
        hts.append(th)
        dts.append(td)
        if committed[lane]:
            stride = n * 32
            k = rng.standard_normal((heads, committed[lane], dim)).astype(np.float32)
            ck, cv = T.chunk_buffers(k, rng.standard_normal(k.shape).astype(np.float32), stride)
            kvx.append(tw.dev, 1, Gp.dev(ck), Gp.dev(cv), [td], [kvx.ChunkParams(0, committed[lane], stride, n)],
                       heads * stride * dim)
    k = rng.standard_normal((lanes, heads, 1, dim)).astype(np.float32)
    v = rng.standard_normal((lanes, heads, 1, dim)).astype(np.float32)
    k[2] = 0                                       # a zero row: scale 0, codes 0
    v[3] *= 1e-20
    ck = np.zeros((lanes, heads, 32, dim), dtype=np.uint16)
    cv = np.zeros((lanes, heads, dim, 32), dtype=np.uint16)
    for lane in range(lanes):
        ck[lane], cv[lane] = T.chunk_buffers(k[lane], v[lane], 32)
    # the token's rows at an address that is aligned to an element and no more
    shifted = [torch.empty(a.size + 1, dtype=torch.int16, device="cuda") for a in (ck, cv)]
    for t, a in zip(shifted, (ck, cv)):
        t[1:] = Gp.dev(a).flatten()
    ck_dev, cv_dev = (t[1:] for t in shifted)
    q = A.queries((lanes, heads, 1, group, dim), 63)
    splits = [n if one_page_splits else max(1, n // 9) for n in counts]
    dp = [kvx.VerifyParams(committed[i], counts[i], kvx.KvLayer(), splits[i], splits[i], 1, 1, 0.0) for i in range(lanes)]
    ws = torch.empty(kvx.attend_workspace_bytes(tw.dev, dp, heads * group), dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    before = [tw.dev.extent_read(e).copy() for e in range(tw.extents)]
    kvx.append(tw.dev, 1, ck_dev, cv_dev, dts, [kvx.ChunkParams(c, 1, 32, n) for c, n in zip(committed, counts)],
               heads * 32 * dim)
    two = torch.zeros((lanes, heads, 1, group, dim), dtype=torch.int16, device="cuda")
    kvx.attend_decode(tw.dev, 1, heads * group, Gp.dev(q), two, dts, dp, 1, ws)
    torch.cuda.synchronize()
    after = [tw.dev.extent_read(e).copy() for e in range(tw.extents)]
    for e in range(tw.extents):
        tw.dev.extent_write(e, before[e])
    one = torch.zeros_like(two)
    ws.fill_(0xA5)
    kvx.append_attend_decode(tw.dev, 1, ck_dev, cv_dev, heads * 32 * dim, 32, heads * group, Gp.dev(q), one, dts, dp, 1, ws)
    torch.cuda.synchronize()
    for e in range(tw.extents):
        assert np.array_equal(tw.dev.extent_read(e), after[e])
    assert torch.equal(one, two)
    tw.close()


@pytest.mark.parametrize("heads,group,dim", [(4, 6, 256), (8, 4, 64), (2, 8, 128)])
@pytest.mark.parametrize("fmt", A.FORMATS)
@pytest.mark.parametrize("written", ["output over keys", "output over values", "hidden", "workspace"])
def test_a_call_that_writes_over_its_chunk_rows(heads, group, dim, fmt, written):
    """What the step writes lies in the memory that its chunk rows came in: every row is stored first."""
    lanes, n, splits = 40, 3, 1 if written.startswith("output") else 2
    committed = [int(c) for c in np.random.default_rng(7).integers(64, 96, lanes)]
    tw = Gp.Twin(fmt, heads, dim, 2, lanes * n)
    ids, rng = tw.pages(lanes * n, 9), np.random.default_rng(8)
    dts = [tw.tables(ids[n * i:n * i + n])[1] for i in range(lanes)]
    rows = lambda *shape: rng.standard_normal(shape).astype(np.float32)
    for lane, c in enumerate(committed):
        ck, cv = T.chunk_buffers(rows(heads, c, dim), rows(heads, c, dim), 32 * n)
        kvx.append(tw.dev, 1, Gp.dev(ck), Gp.dev(cv), [dts[lane]], [kvx.ChunkParams(0, c, 32 * n, n)], heads * 32 * n * dim)
    chunks = [T.chunk_buffers(rows(heads, 1, dim), rows(heads, 1, dim), 32) for _ in range(lanes)]
    keys, values = (Gp.dev(np.stack([c[i] for c in chunks])).flatten() for i in (0, 1))
    q = Gp.dev(A.queries((lanes, heads, 1, group, dim), 63))
    dp = [kvx.VerifyParams(c, n, kvx.KvLayer(), splits, splits, 1, 1, 0.0) for c in committed]
    ws = torch.empty(kvx.attend_workspace_bytes(tw.dev, dp, heads * group), dtype=torch.uint8, device="cuda")
    want = torch.zeros_like(q)
    hidden_want = torch.zeros((lanes, 1, heads * group, dim), dtype=torch.int16, device="cuda")
    torch.cuda.synchronize()
    before = [tw.dev.extent_read(e).copy() for e in range(tw.extents)]
    kvx.append(tw.dev, 1, keys, values, dts, [kvx.ChunkParams(c, 1, 32, n) for c in committed], heads * 32 * dim)
    if written == "hidden":
        kvx.attend_verify_hidden(tw.dev, 1, heads * group, q, want, dts, dp, None, 1, ws, None, hidden_want)
    else:
        kvx.attend_decode(tw.dev, 1, heads * group, q, want, dts, dp, 1, ws)
    torch.cuda.synchronize()
    after = [tw.dev.extent_read(e).copy() for e in range(tw.extents)]
    for e in range(tw.extents):
        tw.dev.extent_write(e, before[e])
    args = (tw.dev, 1, keys, values, heads * 32 * dim, 32, heads * group, q)
    if written == "hidden":
        out, hidden = torch.zeros_like(q), keys[16:16 + hidden_want.numel()].view_as(hidden_want)
        kvx.append_attend_decode_hidden(*args, out, dts, dp, 1, ws, None, hidden)
    elif written == "workspace":
        out, ws = torch.zeros_like(q), torch.cat([values, values.new_zeros(ws.numel())])
        kvx.append_attend_decode(*args[:3], ws[:values.numel()], *args[4:], out, dts, dp, 1, ws.view(torch.uint8))
    else:
        over = keys if written == "output over keys" else values
        out = over[:q.numel()].view_as(q)
        kvx.append_attend_decode(*args, out, dts, dp, 1, ws)
    torch.cuda.synchronize()
    for e in range(tw.extents):
        assert np.array_equal(tw.dev.extent_read(e), after[e])
    assert torch.equal(out, want)
    if written == "hidden":
        assert torch.equal(hidden, hidden_want)
    tw.close()


@pytest.mark.parametrize("heads,group,dim", [(4, 6, 256), (8, 4, 64), (2, 8, 128)])
@pytest.mark.parametrize("fmt", A.FORMATS)
def test_tokens_that_are_no_numbers(heads, group, dim, fmt):
    """Rows of nothing but NaN, with one, with infinities of either sign, with both: the bytes of kv_append."""
    n, committed = 2, [40, 41, 42, 43, 44, 45, 46, 47]
    lanes, rng = len(committed), np.random.default_rng(9)
    tw = Gp.Twin(fmt, heads, dim, 2, lanes * n)
    ids = tw.pages(lanes * n, 9)
    dts = [tw.tables(ids[n * i:n * i + n])[1] for i in range(lanes)]
    for lane, c in enumerate(committed):
        ck, cv = T.chunk_buffers(*(rng.standard_normal((heads, c, dim)).astype(np.float32) for _ in range(2)), 32 * n)
        kvx.append(tw.dev, 1, Gp.dev(ck), Gp.dev(cv), [dts[lane]], [kvx.ChunkParams(0, c, 32 * n, n)], heads * 32 * n * dim)
    rows = rng.standard_normal((2, lanes, heads, 1, dim)).astype(np.float32)
    rows[:, 0] = np.nan
    rows[0, 1], rows[1, 2] = np.nan, np.nan
    rows[:, 3, ..., 5] = np.nan
    rows[:, 4, ..., 5] = np.inf
    rows[:, 5, ..., dim - 1] = -np.inf
    rows[:, 6, ..., 1:] = np.nan
    rows[:, 7, ..., ::2], rows[:, 7, ..., 1] = np.nan, np.inf
    chunks = [T.chunk_buffers(rows[0, i], rows[1, i], 32) for i in range(lanes)]
    keys, values = (Gp.dev(np.stack([c[i] for c in chunks])).flatten() for i in (0, 1))
    q = Gp.dev(A.queries((lanes, heads, 1, group, dim), 63))
    dp = [kvx.VerifyParams(c, n, kvx.KvLayer(), 2, 2, 1, 1, 0.0) for c in committed]
    ws = torch.empty(kvx.attend_workspace_bytes(tw.dev, dp, heads * group), dtype=torch.uint8, device="cuda")
    two, one = torch.zeros_like(q), torch.zeros_like(q)
    torch.cuda.synchronize()
    before = [tw.dev.extent_read(e).copy() for e in range(tw.extents)]
    kvx.append(tw.dev, 1, keys, values, dts, [kvx.ChunkParams(c, 1, 32, n) for c in committed], heads * 32 * dim)
    kvx.attend_decode(tw.dev, 1, heads * group, q, two, dts, dp, 1, ws)
    torch.cuda.synchronize()
    after = [tw.dev.extent_read(e).copy() for e in range(tw.extents)]
    for e in range(tw.extents):
        tw.dev.extent_write(e, before[e])
    kvx.append_attend_decode(tw.dev, 1, keys, values, heads * 32 * dim, 32, heads * group, q, one, dts, dp, 1, ws)
    torch.cuda.synchronize()
    for e in range(tw.extents):
        assert np.array_equal(tw.dev.extent_read(e), after[e])
    assert torch.equal(one, two)
    tw.close()
