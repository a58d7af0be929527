"""Narrow items of a batch: rows that tiles of 16 nonzeros per lane leave whole
are summed like the host loop, and are not cut into carries and a combine each.
"""
import numpy as np
import pytest

import dspmm as D
import oracle as O
from gpu_common import assert_bitwise, note

pytestmark = pytest.mark.gpu
RM = D.DENSE_ROW_MAJOR


def rows(lo, hi, nr=3000, nc=2500, seed=4):
    rng = np.random.default_rng(seed)
    lens = rng.integers(lo, hi + 1, nr)
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    ci = np.concatenate([np.sort(rng.choice(nc, int(n), replace=False)) for n in lens])
    return nr, nc, rp, ci.astype(np.int32), rng.standard_normal(ci.size).astype(np.float32)


@pytest.mark.parametrize("btype", [D.DSPMM_R_32F, D.DSPMM_R_16BF])
def test_rows_stay_whole(btype):
    """nv and the longest row that 16 nonzeros per lane hold (a lane holds four
    columns, eight in BF16)."""
    bf16 = btype == D.DSPMM_R_16BF
    rng = np.random.default_rng(7)
    items, want, keep = [], [], []
    for nv, most in ((1, 16), (2, 16), (3, 16 if bf16 else 32), (4, 16), (7, 32), (8, 16 if bf16 else 32)):
        nr, nc, rp, ci, va = rows(max(1, most - 7), most, seed=nv)
        B = rng.uniform(-1, 1, (nc, nv)).astype(np.float32)
        h = D.Matrix(nr, nc, rp, ci, va)
        d_B = D.DeviceArray.from_numpy(B)
        if bf16:
            d_B = D.to_bf16_device(d_B)
        d_C = D.DeviceArray.from_numpy(np.full((nr, nv), np.nan, np.float32))
        items.append((h, nv, d_B, d_C))
        want.append(O.spmm_host32(RM, nr, nc, nv, rp, ci, va, O.round_bf16(B) if bf16 else B))
        keep.append((h, d_B, d_C))
    b = D.Batch(items, btype=btype)
    note(str(b.describe()))
    assert b.describe()["splits"] == 0
    b.run()
    D.synchronize()
    for (h, nv, _, d_C), w in zip(items, want):
        assert_bitwise(d_C.numpy().reshape(-1), w.reshape(-1), f"nv={nv}")
    b.close()
    for h, _, _ in keep:
        h.close()
