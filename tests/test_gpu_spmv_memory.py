"""SpMV where the device has no memory left for a second copy of the matrix:
the slices of diagonals are given up, the tiles run."""
import numpy as np
import pytest

import dspmm as D
import oracle as O
import workloads as W
from gpu_common import assert_fp32, note

pytestmark = pytest.mark.gpu
RM = D.DENSE_ROW_MAJOR
LEFT = 48 << 20                      # bytes left free; the slices of the stencil need 120 MB


def test_slices_without_memory():
    a = W.c3_matrix(90)
    m = D.Matrix(a.nr, a.nc, a.rowPtr, a.colIdx, a.values)
    x = np.random.default_rng(1).uniform(-1, 1, a.nc).astype(np.float32)
    d_x, d_y = D.DeviceArray.from_numpy(x), D.DeviceArray.from_numpy(np.full(a.nr, np.nan, np.float32))
    small = W.c3_matrix(8)           # the kernels are loaded before the memory goes
    s = D.Matrix(small.nr, small.nc, small.rowPtr, small.colIdx, small.values)
    s.spmm(d_x, d_y, 1)
    D.synchronize()
    s.close()
    d_y = D.DeviceArray.from_numpy(np.full(a.nr, np.nan, np.float32))
    before = m.describe()["hbm_bytes"]
    assert D.lib().dspmm_release_scratch() == 0      # else the slices take what other products keep
    D.synchronize()
    taken = []
    try:
        step = 64 << 30
        while step >= 16 << 20:
            free = D.device_info()["free_mem"]
            if free < LEFT + step:
                step //= 2
                continue
            try:
                taken.append(D.DeviceArray(step, np.uint8, (step,)))
            except RuntimeError:
                step //= 2
        note(f"free {D.device_info()['free_mem'] >> 20} MiB of {D.device_info()['total_mem'] >> 30} GiB")
        for _ in range(2):
            m.spmm(d_x, d_y, 1)
            D.synchronize()
    finally:
        for t in taken:
            t.free()
    assert m.describe()["hbm_bytes"] - before < 32 << 20
    h32 = O.spmm_host32(RM, a.nr, a.nc, 1, a.rowPtr, a.colIdx, a.values, x).reshape(-1)
    c64, ab = O.spmm_fp64(RM, a.nr, a.nc, 1, a.rowPtr, a.colIdx, a.values, x)
    assert_fp32(d_y.numpy(), c64.reshape(-1), ab.reshape(-1), np.diff(a.rowPtr).astype(np.float64),
                "tiles", h32)
    m.close()


def test_a_tile_size_asks_for_the_tiles():
    """SPMV_TILED with a tile size runs the tiles also on few diagonals; without
    one, and under AUTO, the slices; the autotuner times the slices once."""
    a = W.c3_matrix(24)
    x = np.random.default_rng(2).uniform(-1, 1, a.nc).astype(np.float32)
    d_x, d_y = D.DeviceArray.from_numpy(x), D.DeviceArray.zeros(a.nr)
    grown = {}
    for name, cfg in (("tiles", D.make_config(D.VARIANT_SPMV_TILED, tile_nnz=1024)),
                      ("default", D.make_config(D.VARIANT_SPMV_TILED)), ("auto", None)):
        m = D.Matrix(a.nr, a.nc, a.rowPtr, a.colIdx, a.values)
        before = m.describe()["hbm_bytes"]
        m.spmm(d_x, d_y, 1, config=cfg)
        D.synchronize()
        grown[name] = (m.describe()["hbm_bytes"] - before) / a.nnz
        if cfg is None:
            table = m.autotune_table(d_x, d_y, 1, reps=1)
            sizes = [c.tile_nnz for c, _ in table if c.variant == D.VARIANT_SPMV_TILED]
            assert sorted(sizes) == [0, 512, 1024, 2048, 4096]
        m.close()
    note(str(grown))
    assert grown["tiles"] < 1 and grown["default"] > 5 and grown["auto"] > 5


def test_autotuner_without_diagonals():
    rng = np.random.default_rng(3)
    ci = np.sort(rng.integers(0, 3000, (2000, 8)), 1).astype(np.int32)
    m = D.Matrix(2000, 3000, (np.arange(2001) * 8).astype(np.int32), ci.reshape(-1),
                 rng.standard_normal(16000).astype(np.float32))
    d_x, d_y = D.DeviceArray.from_numpy(rng.uniform(-1, 1, 3000).astype(np.float32)), D.DeviceArray.zeros(2000)
    table = m.autotune_table(d_x, d_y, 1, reps=1)
    assert sorted(c.tile_nnz for c, _ in table if c.variant == D.VARIANT_SPMV_TILED) == [512, 1024, 2048, 4096]
    m.close()


def test_a_matrix_takes_the_scratch_back():
    """Column-major products keep scratch; a matrix that needs the memory gets it."""
    a, w = W.c3_matrix(90), W.gen_csr(W.GEN_FIXED, 300000, 300000, seed=2, p0=4)
    nv = 64
    d = [D.DeviceArray.from_numpy(v) for v in (w.rowPtr, np.zeros(1, np.int32), w.colIdx, w.values)]
    B, out = D.DeviceArray.zeros(w.nc * nv), D.DeviceArray.zeros(w.nr * nv)
    assert D.lib().dspmm_release_scratch() == 0
    D.synchronize()
    free = D.device_info()["free_mem"]
    assert D.launch("spmm_csr_scalar_col", w.nr, w.nc, w.nnz, nv, *d, B, out) == 0
    D.synchronize()
    kept = free - D.device_info()["free_mem"]
    assert kept >= 128 << 20
    x = np.random.default_rng(1).uniform(-1, 1, a.nc).astype(np.float32)
    d_x, d_y = D.DeviceArray.from_numpy(x), D.DeviceArray.from_numpy(np.full(a.nr, np.nan, np.float32))
    taken = []
    try:
        step = 64 << 30
        while step >= 16 << 20:
            if D.device_info()["free_mem"] < LEFT + step:
                step //= 2
                continue
            taken.append(D.DeviceArray(step, np.uint8, (step,)))
        left = D.device_info()["free_mem"]
        note(f"scratch {kept >> 20} MiB, free {left >> 20} MiB, matrix {8 * a.nnz >> 20} MiB")
        assert left < 8 * a.nnz
        m = D.Matrix(a.nr, a.nc, a.rowPtr, a.colIdx, a.values)
        m.spmm(d_x, d_y, 1, config=D.make_config(D.VARIANT_SPMV_TILED, tile_nnz=1024))
        D.synchronize()
        m.close()
    finally:
        for t in taken:
            t.free()
    h32 = O.spmm_host32(RM, a.nr, a.nc, 1, a.rowPtr, a.colIdx, a.values, x).reshape(-1)
    c64, ab = O.spmm_fp64(RM, a.nr, a.nc, 1, a.rowPtr, a.colIdx, a.values, x)
    assert_fp32(d_y.numpy(), c64.reshape(-1), ab.reshape(-1), np.diff(a.rowPtr).astype(np.float64),
                "tiles", h32)


@pytest.mark.parametrize("nr,n,slices", [(64, 8, True), (63, 16, True), (128, 32, True), (1, 40, False), (65, 8, False),
                                         (64, 33, False)])
def test_which_bands_go_in_slices(nr, n, slices):
    """One slice and two, and what keeps a band out of them: padding, long rows.
    The path shows in the plan's bytes."""
    col = (np.arange(nr)[:, None] + 2 * np.arange(n)).astype(np.int32)
    rng = np.random.default_rng(n)
    val = rng.uniform(-1, 1, (nr, n)).astype(np.float32)
    x = rng.uniform(-1, 1, nr + 2 * n).astype(np.float32)
    rp = (np.arange(nr + 1) * n).astype(np.int32)
    m = D.Matrix(nr, x.size, rp, col.reshape(-1), val.reshape(-1))
    d_x, d_y = D.DeviceArray.from_numpy(x), D.DeviceArray.from_numpy(np.full(nr, np.nan, np.float32))
    before = m.describe()["hbm_bytes"]
    m.spmm(d_x, d_y, 1)
    D.synchronize()
    grown = m.describe()["hbm_bytes"] - before
    assert (grown >= 5 * nr * n) == slices, f"plan of {grown} bytes"
    h32 = O.spmm_host32(RM, nr, x.size, 1, rp, col.reshape(-1), val.reshape(-1), x).reshape(-1)
    c64, ab = O.spmm_fp64(RM, nr, x.size, 1, rp, col.reshape(-1), val.reshape(-1), x)
    if n <= 16:
        assert np.array_equal(d_y.numpy(), h32)
    else:
        assert_fp32(d_y.numpy(), c64.reshape(-1), ab.reshape(-1), np.full(nr, n, np.float64), "band", h32)
    m.close()
