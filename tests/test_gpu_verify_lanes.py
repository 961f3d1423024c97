"""Verify lanes of 33 to 128 fused rows on int8 and e4m3 pages, and of 33 to 96 on bf16 pages, run as waves of 32
rows beside waves that stage the pages (kvx_verify.hip): the number of row waves, a last wave partly filled, live
rows below the capacity, one split (rows written directly) and several, splits of one page.  bf16 lanes of 98 and
128 rows run on group_wide_kernel (kvx_attend_wide.hip); tests/test_shared_prefix.py has the other form's."""
import numpy as np
import pytest
import torch

from oracle import kvoracle as ko
from richengine_amd import kvx
import gpulib as Gp
import test_gpu_attention as A

pytestmark = pytest.mark.gpu


# group x capacity: 33 = one row in the second wave, 64 = two full waves, 65 (13 x 5) = one row in the third,
# 96 = three full ones, 98 (14 x 7) = two rows in the fourth, 128 the most there are
@pytest.mark.parametrize("heads,group,capacity", [(2, 11, 3), (4, 4, 16), (1, 13, 5), (4, 6, 16), (1, 14, 7), (2, 16, 8)])
@pytest.mark.parametrize("fmt", [ko.INT8, ko.BF16, ko.FP8])
@pytest.mark.parametrize("tree", [False, True])
def test_verify_lanes_match_oracle(heads, group, capacity, fmt, tree):
    if tree and fmt == ko.FP8:
        pytest.skip("tree verify has no fp8 kernels")
    saved = (A.H, A.G, A.QH)
    A.H, A.G, A.QH = heads, group, heads * group
    try:
        H, G, D, QH = A.H, A.G, 256, A.QH
        rows = capacity - 1 if tree else capacity   # a tree leaves the last row of the tile empty
        committed, splits = [0, 31, 95, 1000, 700], [1, 2, 3, 7, 1]   # 95: splits of a page; 700: one split
        lanes = len(committed)
        tw, counts, hts, dts = A.shared_pool_lanes(fmt, committed, rows, seed=capacity * group)
        rng = np.random.default_rng(capacity)
        masks = np.zeros((lanes, capacity), dtype=np.uint32)
        for lane in range(lanes):
            parents = [-1] + [int(rng.integers(max(0, i - 3), i)) for i in range(1, rows)]
            masks[lane, :rows] = A.tree_masks(parents)
        q = np.zeros((lanes, H, 32, G, D), dtype=np.uint16)
        q[:, :, :capacity] = A.queries((lanes, H, capacity, G, D), 7)
        given = (masks,) if tree else ()
        hp = [ko.VerifyParams(committed[i], counts[i], tw.host.layer(1), splits[i], 128, rows, capacity, 0.0)
              for i in range(lanes)]
        n, want, want32 = ko.attend_verify(fmt, H, G, D, q, hts, hp, *given)
        assert n == lanes
        dp = [kvx.VerifyParams(committed[i], counts[i], kvx.KvLayer(), splits[i], splits[i], rows, capacity, 0.0)
              for i in range(lanes)]
        out = torch.full((lanes, H, 32, G, D), 0x5A5A, dtype=torch.int16, device="cuda")
        ws = torch.empty(kvx.attend_workspace_bytes(tw.dev, dp, QH), dtype=torch.uint8, device="cuda")
        kvx.attend_verify(tw.dev, 1, QH, Gp.dev(q), out, dts, dp, Gp.dev(masks) if tree else None, 32, ws)
        torch.cuda.synchronize()
        got = Gp.host_u16(out)
        live = np.zeros((lanes, H, 32), dtype=bool)
        live[:, :, :rows] = True
        Gp.check_attention(got, want, want32, live, A.tol(fmt), f"verify lanes fmt={fmt} M={capacity * group}",
                           explain=Gp.lanes_explainer(fmt, H, G, D, q, hts, tw.host.layer(1), committed, rows,
                                                      splits, capacity, *given))
        assert not got[:, :, rows:capacity].any() and (got[:, :, capacity:] == 0x5A5A).all()
        tw.close()
    finally:
        A.H, A.G, A.QH = saved
