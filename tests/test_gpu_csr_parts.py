"""CSR_PARTS: a row's products four at a time, these in two sums in turn.  The
edges of both kernels (by wavefronts, by blocks) against 64 bits, whole
numbers exactly, and what the variant refuses."""
import ctypes as C

import numpy as np
import pytest

import dspmm as D
import oracle as O
from gpu_common import assert_bf16, assert_fp32

pytestmark = pytest.mark.gpu
RM, CM = D.DENSE_ROW_MAJOR, D.DENSE_COL_MAJOR
EDGES = [0, 1, 3, 4, 5, 7, 8, 9, 15, 16, 17, 63, 64, 65, 255, 256, 257, 511, 512, 513, 1023, 1024, 1025, 2600]


def rows(lens, nc, whole=False, seed=5):
    rng = np.random.default_rng(seed)
    ptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    col = rng.integers(0, nc, ptr[-1]).astype(np.int32)
    val = (rng.integers(-8, 9, ptr[-1]) if whole else rng.standard_normal(ptr[-1])).astype(np.float32)
    return ptr, col, val


def run(ptr, col, val, nc, nv, layout, bf16, whole, **cfg):
    nr = ptr.size - 1
    rng = np.random.default_rng(nv)
    shape = (nc, nv) if layout == RM else (nv, nc)
    B = (rng.integers(-4, 5, shape) if whole else rng.uniform(-1, 1, shape)).astype(np.float32)
    d_B = D.DeviceArray.from_numpy(B)
    d_B = D.to_bf16_device(d_B) if bf16 else d_B
    d_C = D.DeviceArray.from_numpy(np.full((nr, nv) if layout == RM else (nv, nr), np.nan, np.float32))
    m = D.Matrix(nr, nc, ptr, col, val)
    m.spmm(d_B, d_C, nv, layout, btype=D.DSPMM_R_16BF if bf16 else D.DSPMM_R_32F,
           config=D.make_config(D.VARIANT_CSR_PARTS, **cfg))
    D.synchronize()
    m.close()
    got = d_C.numpy()
    if layout == CM:
        got, B = np.ascontiguousarray(got.T), np.ascontiguousarray(B.T)
    c64, ab = O.spmm_fp64(RM, nr, nc, nv, ptr, col, val, B)
    what = f"nr={nr} nv={nv} layout={layout} bf16={bf16} {cfg}"
    if whole:
        assert np.array_equal(got.reshape(-1), c64.reshape(-1)), what
    elif bf16:
        assert_bf16(got.reshape(-1), c64.reshape(-1), ab.reshape(-1), what)
    else:
        h32 = O.spmm_host32(RM, nr, nc, nv, ptr, col, val, B).reshape(-1)
        assert_fp32(got.reshape(-1), c64.reshape(-1), ab.reshape(-1),
                    np.repeat(np.diff(ptr).astype(np.float64), nv), what, h32)


@pytest.mark.parametrize("nv", [1, 2, 3, 4, 5, 7, 8, 12, 16, 17, 31, 32, 33, 100, 260])
@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("whole", [False, True])
def test_edges(nv, bf16, whole):
    rng = np.random.default_rng(nv)
    lens = np.concatenate([EDGES, rng.integers(0, 40, 900), rng.permutation(EDGES), rng.integers(0, 9, 77)])
    ptr, col, val = rows(lens, 700, whole)
    for layout in (RM, CM):
        for unroll in (0, 8):
            run(ptr, col, val, 700, nv, layout, bf16, whole, unroll=unroll, tile_nnz=nv % 2)


@pytest.mark.parametrize("lens", [[1], [0], [5000], [0] * 300, [200] * 65, [3] * 129, [9, 0] * 128])
@pytest.mark.parametrize("nv", [6, 24, 40])
def test_small(lens, nv):
    ptr, col, val = rows(lens, 90)
    for unroll in (0, 8):
        run(ptr, col, val, 90, nv, RM, False, False, unroll=unroll)


def test_refused():
    ptr, col, val = rows([4] * 50, 60)
    m = D.Matrix(50, 60, ptr, col, val)
    d_B, d_C = D.DeviceArray.zeros(60 * 8), D.DeviceArray.zeros(50 * 8)
    for cfg in (dict(unroll=4), dict(unroll=3), dict(tile_nnz=2, unroll=8)):
        with pytest.raises(D.DspmmError):
            m.spmm(d_B, d_C, 8, config=D.make_config(D.VARIANT_CSR_PARTS, **cfg))
    m.close()


@pytest.mark.parametrize("layout", [RM, CM])
@pytest.mark.parametrize("bf16", [False, True])
def test_without_allocation(layout, bf16):
    """Prepared, it runs in the no-alloc call too, with the same bits."""
    nr, nc, nv = 1500, 900, 24
    ptr, col, val = rows(np.random.default_rng(2).integers(0, 90, nr), nc)
    m = D.Matrix(nr, nc, ptr, col, val)
    bt = D.DSPMM_R_16BF if bf16 else D.DSPMM_R_32F
    d_B = D.DeviceArray.from_numpy(np.random.default_rng(3).uniform(-1, 1, nc * nv).astype(np.float32))
    d_B = D.to_bf16_device(d_B) if bf16 else d_B
    out = [D.DeviceArray.from_numpy(np.full(nr * nv, np.nan, np.float32)) for _ in range(2)]
    cfg = D.make_config(D.VARIANT_CSR_PARTS)
    m.spmm(d_B, out[0], nv, layout, btype=bt, config=cfg)
    m.prepare(d_B, out[1], nv, layout, btype=bt, config=cfg)
    ld = (nv, nv) if layout == RM else (nc, nr)
    st = D.lib().dspmm_spmm_ex_noalloc(m.handle, layout, nv, d_B.ptr, ld[0], bt, out[1].ptr, ld[1],
                                       C.byref(cfg), None)
    assert st == 0, D.status_string(st)
    D.synchronize()
    a, b = out[0].numpy(), out[1].numpy()
    assert np.isfinite(a).all() and np.array_equal(a.view(np.uint32), b.view(np.uint32))
    m.close()
