"""int4 verify lanes of more than 16 fused rows run as waves of 16, 32 or 48 rows by the size of the
launch and the length of the splits: the rows of a lane are the same bits whichever it is."""
import numpy as np
import pytest
import torch

from oracle import kvoracle as ko
from richengine_amd import kvx
import gpulib as Gp
import test_gpu_attention as A

pytestmark = pytest.mark.gpu
D = 256


def verify(tw, tables, heads, group, q, params, masks=None):
    lanes, stride = q.shape[0], q.shape[2]
    out = torch.full(q.shape, 0x5A5A, dtype=torch.int16, device="cuda")
    ws = torch.empty(kvx.attend_workspace_bytes(tw.dev, params, heads * group), dtype=torch.uint8, device="cuda")
    kvx.attend_verify(tw.dev, 1, heads * group, Gp.dev(np.ascontiguousarray(q)), out, tables, params, masks, stride, ws)
    torch.cuda.synchronize()
    return Gp.host_u16(out)


# 18 and 24 fused rows: a second block of 16 partly filled; 48: waves of 48 over long splits; 96 and 128: most there are
@pytest.mark.parametrize("heads,group,rows", [(3, 2, 9), (4, 6, 4), (1, 16, 8), (4, 6, 8), (4, 6, 16), (2, 16, 8)])
@pytest.mark.parametrize("committed,splits", [(40, 1), (700, 5), (1700, 1)])
def test_a_lane_alone_and_among_many(heads, group, rows, committed, splits):
    tw = Gp.Twin(ko.INT4, heads, D, 2, (committed + rows + 31) // 32)
    pages, th, td = A.fill(tw, committed + rows, seed=committed + rows + group)
    q = np.zeros((1, heads, rows, group, D), dtype=np.uint16)
    q[0] = A.queries((heads, rows, group, D), rows)
    one = kvx.VerifyParams(committed, len(pages), kvx.KvLayer(), splits, splits, rows, rows, 0.0)
    alone = verify(tw, [td], heads, group, q, [one])          # few waves: 16 rows each, unless the split is long
    blocks = -(-rows * group // 16) * heads * splits
    many = min(32, 3072 // blocks + 1)
    # as many lanes as leave no place for a wave of 16 rows each (or the launch's 32), and a long split among them
    among = verify(tw, [td] * many, heads, group, np.repeat(q, many, 0), [one] * many)
    for lane in range(many):
        assert np.array_equal(among[lane], alone[0]), lane
    long = [one, kvx.VerifyParams(committed, len(pages), kvx.KvLayer(), splits, splits, rows - 1, rows, 0.0)]
    two = verify(tw, [td] * 2, heads, group, np.repeat(q, 2, 0), long)
    assert np.array_equal(two[0], alone[0]) and not two[1][:, rows - 1].any()
    tw.close()
