"""SpMV on diagonal slices (matrices with few distinct column-minus-row
distances) at the sizes where the slicing can go wrong, against the oracle:
rows of at most 16 nonzeros equal the host loop bit for bit, longer ones pass
the FP32 gate; what padding would read never reaches a result.
"""
import numpy as np
import pytest

import dspmm as D
import oracle as O
from gpu_common import assert_bitwise, assert_fp32, note

pytestmark = pytest.mark.gpu
RM, CM = D.DENSE_ROW_MAJOR, D.DENSE_COL_MAJOR
SPMV = D.make_config(D.VARIANT_SPMV_TILED)


def banded(nr, nc, dists, keep=1.0, seed=3):
    """Row r holds columns r + d (within range) for the given distances, each
    kept with probability `keep`, in the order given."""
    rng = np.random.default_rng(seed)
    rp, ci = [0], []
    for r in range(nr):
        ci += [r + d for d in dists if 0 <= r + d < nc and rng.random() < keep]
        rp.append(len(ci))
    return (np.array(rp, np.int32), np.array(ci, np.int32),
            rng.standard_normal(len(ci)).astype(np.float32))


CASES = {
    "one_row": (1, 40, range(40), 1.0),
    "n63": (63, 63, (-1, 0, 1), 1.0),
    "n64_27": (64, 200, range(0, 81, 3), 1.0),
    "n65": (65, 65, (-7, -1, 0, 1, 7), 1.0),
    "n257_mixed": (257, 300, range(-12, 13), 0.6),
    "unsorted": (130, 130, (5, -3, 0, 2, -1), 1.0),
    "repeated": (130, 140, (4, 4, 0, -1), 1.0),
    "lens_16_17": (300, 400, range(17), 0.97),
    "wide": (500, 1200, range(256), 1.0),            # every diagonal the plan can hold
    "too_many": (500, 1200, range(257), 1.0),        # one more: the tiles
}


@pytest.mark.parametrize("name", CASES)
def test_diag_slices(name):
    nr, nc, dists, keep = CASES[name]
    rp, ci, va = banded(nr, nc, dists, keep)
    lens = np.diff(rp).astype(np.float64)
    short = lens <= 16
    m = D.Matrix(nr, nc, rp, ci, va)
    rng = np.random.default_rng(8)
    x = rng.uniform(-1, 1, (nc, 3)).astype(np.float32)
    for ldx, ldy, layout, bf16 in ((1, 1, RM, False), (3, 2, RM, False), (1, 1, CM, False),
                                   (1, 1, RM, True)):
        note(f"{name} ldx={ldx} ldy={ldy} layout={layout} bf16={bf16}")
        xs = np.ascontiguousarray(x[:, :ldx])
        d_x = D.DeviceArray.from_numpy(xs)
        if bf16:
            d_x = D.to_bf16_device(d_x)
        x0 = np.ascontiguousarray(xs[:, 0])
        xr = O.round_bf16(x0) if bf16 else x0
        h32 = O.spmm_host32(RM, nr, nc, 1, rp, ci, va, xr).reshape(-1)
        c64, ab = O.spmm_fp64(RM, nr, nc, 1, rp, ci, va, xr)
        d_y = D.DeviceArray.from_numpy(np.full((nr, ldy), np.nan, np.float32))
        m.spmm(d_x, d_y, 1, layout=layout, ldb=nc if layout == CM else ldx,
               ldc=nr if layout == CM else ldy, config=SPMV,
               btype=D.DSPMM_R_16BF if bf16 else D.DSPMM_R_32F)
        D.synchronize()
        y = d_y.numpy().reshape(nr, ldy)
        assert np.isnan(y[:, 1:]).all()
        assert_bitwise(y[:, 0][short], h32[short], f"{name} rows <= 16")
        assert_fp32(y[:, 0].copy(), c64.reshape(-1), ab.reshape(-1), lens, name, h32)
    m.close()


def test_padding_reads_reach_no_result():
    """Infinities where only padded entries look (x[0] and the rows' own
    columns) leave every finite result finite."""
    nr = nc = 200
    rp, ci, va = banded(nr, nc, (3, 11, 40), 0.8)
    m = D.Matrix(nr, nc, rp, ci, va)
    x = np.ones(nc, np.float32)
    x[np.setdiff1d(np.arange(nc), ci)] = np.inf
    assert np.isinf(x[0])
    d_y = D.DeviceArray.from_numpy(np.full(nr, np.nan, np.float32))
    m.spmm(D.DeviceArray.from_numpy(x), d_y, 1, config=SPMV)
    D.synchronize()
    h32 = O.spmm_host32(RM, nr, nc, 1, rp, ci, va, x).reshape(-1)
    assert np.isfinite(h32).all()
    assert_bitwise(d_y.numpy(), h32, "padding")
    m.close()
