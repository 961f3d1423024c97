"""int4 verify lanes of more than 16 fused rows run as waves of 16, 32 or 48 rows by the size of the
launch and the length of the splits: the rows of a lane are the same bits whichever it is."""
import ctypes as C

import numpy as np
import pytest
import torch

from oracle import kvoracle as ko
from richengine_amd import kvx
import gpulib as Gp
import test_gpu_attention as A
import test_gpu_prefill_batch as B

pytestmark = pytest.mark.gpu
D = 256


def rows_to_a_wave(heads, group, params):
    layout = kvx.Layout(2, heads, D, kvx.INT4, 0.0)
    lanes = (kvx.VerifyParams * len(params))(*params)
    return kvx.lib().kvx_debug_int4_verify_rows(C.byref(layout), heads * group, lanes, len(params), 0)


def verify(tw, tables, heads, group, q, params):
    out = torch.full(q.shape, 0x5A5A, dtype=torch.int16, device="cuda")
    ws = torch.empty(kvx.attend_workspace_bytes(tw.dev, params, heads * group), dtype=torch.uint8, device="cuda")
    kvx.attend_verify(tw.dev, 1, heads * group, Gp.dev(np.ascontiguousarray(q)), out, tables, params, None, q.shape[2], ws)
    torch.cuda.synchronize()
    return Gp.host_u16(out)


# 18 and 24 fused rows: a second block of 16 partly filled; 48: one wave of 48 over long splits; 35: that wave
# partly filled; 96 and 128: most there are
@pytest.mark.parametrize("heads,group,rows,long_form", [(3, 2, 9, 32), (4, 6, 4, 32), (1, 16, 8, 32), (4, 6, 8, 48),
                                                        (3, 5, 7, 48), (4, 6, 16, 32), (2, 16, 8, 32)])
@pytest.mark.parametrize("committed", [700, 1023])
def test_a_lane_in_every_form(heads, group, rows, long_form, committed):
    fused = rows * group
    blocks = -(-fused // 16) * heads
    splits = -(-3073 // (32 * blocks))  # 32 such lanes leave no place for waves of 16 rows
    long_committed = 1700               # 54 pages, in one split
    entries, long_entries = (committed + rows + 31) // 32, (long_committed + rows + 31) // 32
    tw = Gp.Twin(ko.INT4, heads, D, 2, entries + long_entries)
    ids = tw.pages(entries + long_entries, committed + group)
    _, _, td = A.fill(tw, committed + rows, seed=committed + rows + group, pages=ids[:entries])
    _, _, long_td = A.fill(tw, long_committed + rows, seed=rows, pages=ids[entries:])
    q = np.zeros((1, heads, rows, group, D), dtype=np.uint16)
    q[0] = A.queries((heads, rows, group, D), rows)
    one = kvx.VerifyParams(committed, entries, kvx.KvLayer(), splits, splits, rows, rows, 0.0)
    long = kvx.VerifyParams(long_committed, long_entries, kvx.KvLayer(), 1, 1, rows - 1, rows, 0.0)
    assert rows_to_a_wave(heads, group, [one]) == 16
    assert rows_to_a_wave(heads, group, [one] * 32) == 32
    assert rows_to_a_wave(heads, group, [one, long]) == long_form
    alone = verify(tw, [td], heads, group, q, [one])
    among = verify(tw, [td] * 32, heads, group, np.repeat(q, 32, 0), [one] * 32)
    for lane in range(32):
        assert np.array_equal(among[lane], alone[0]), lane
    beside = verify(tw, [td, long_td], heads, group, np.repeat(q, 2, 0), [one, long])
    assert np.array_equal(beside[0], alone[0]) and not beside[1][:, rows - 1].any()
    # the long lane in waves of 16 rows: 48 pages to a split and fewer, the same splits otherwise
    halves = kvx.VerifyParams(long_committed, long_entries, kvx.KvLayer(), 2, 2, rows, rows, 0.0)
    assert rows_to_a_wave(heads, group, [halves]) == 16
    assert rows_to_a_wave(heads, group, [halves, long]) == long_form
    alone = verify(tw, [long_td], heads, group, q, [halves])
    beside = verify(tw, [long_td, long_td], heads, group, np.repeat(q, 2, 0), [halves, long])
    assert np.array_equal(beside[0], alone[0])
    tw.close()


# pairs of tiles alone in waves of 16 rows, together in waves of 32: a wave to a workgroup up to 2048 of them and where
# the last wave of a pair is half full (five blocks of 16), else four, those that see the most first; odd tiles beside the
# pairs, histories that end anywhere, two splits
@pytest.mark.parametrize("heads,group,committed,rows,splits,waves", [
    (4, 6, (96, 0, 45, 1000), 264, 1, 768), (4, 6, (96, 0, 45, 100, 32, 7), 680, 1, 3024),
    (2, 6, (64, 320, 0, 96, 32, 0), 515, 2, 2304), (3, 5, (96, 33, 7), 488, 1, 810), (8, 2, tuple(range(0, 320, 32)), 521, 1, 2640),
    (1, 16, (31, 500, 0, 7, 64, 100, 200, 3, 90), 530, 1, 2376)])
def test_pairs_of_tiles_of_several_sequences(monkeypatch, heads, group, committed, rows, splits, waves):
    for name, value in zip(("H", "G", "D", "QH"), (heads, group, D, heads * group)):
        monkeypatch.setattr(B, name, value)
    n, pairs = len(committed), rows // 16 + (rows % 16 > 8)
    assert n * pairs * heads * splits * group > 1024 and n * pairs * heads * splits * -(-group // 2) == waves
    together, alone, tw = B.run_batch(ko.INT4, list(committed), [rows] * n, [splits] * n)
    assert np.array_equal(together, alone)
    assert (alone != 0x5A5A).any(axis=1).all()
    tw.close()
