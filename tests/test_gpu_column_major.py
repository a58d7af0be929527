"""Column-major products on row-major copies in scratch, and the kernels that
run them: default and other streams, a captured stream (in place), threads,
columns in slabs, accumulation; rows far longer than the others; COO input in
any order.  Operands are small integers, so every summation order is exact.
"""
import ctypes as C
import threading

import numpy as np
import pytest

import dspmm as D
from gpu_common import assert_bitwise, note
from test_gpu_compat_edges import float_case, int_case, row_lengths
from test_gpu_prepare import capture, hip, stream

pytestmark = pytest.mark.gpu

COL = ["spmm_csr_scalar_col", "spmm_csr_vector_col", "spmm_coo_scalar_col", "spmm_coo_vector_col"]


@pytest.fixture(scope="module")
def big():
    """Enough products for the copies from nv = 8 on, in place below."""
    rng = np.random.default_rng(21)
    lens = rng.integers(0, 100, 15011)
    lens[[3, 15010]] = 1700
    return int_case("big", lens, 20021, 65)


def launch(c, name, nv, st=None, d_C=None):
    s = D.launch(name, c.nr, c.nc, c.nnz, nv, c.d_rp, c.d_ri, c.d_ci, c.d_v, c.d_B,
                 d_C or c.d_C, st)
    assert s == 0, D.status_string(s)


@pytest.mark.parametrize("name", COL)
@pytest.mark.parametrize("nv", [2, 3, 8, 16, 33, 64, 65])
def test_copies_on_default_and_other_streams(big, name, nv):
    note(f"{name} nv={nv}")
    want = big.ref(D.DENSE_COL_MAJOR, nv)[0] + (2.0 if "coo" in name else 0.0)
    for st in (None, stream()):
        big.fill_output(2.0)                    # overwritten, or added to
        launch(big, name, nv, st)
        D.synchronize()
        assert_bitwise(big.output(nv) + 0.0, want + 0.0, f"{name} nv={nv}")
    assert D.lib().dspmm_release_scratch() == 0
    assert D.lib().dspmm_release_scratch() == 0


def test_captured_stream_runs_in_place(big):
    h, st, nv = hip(), stream(), 16
    big.fill_output(0.0)
    status, graph = capture(h, st, lambda: D.lib().spmm_csr_scalar_col(
        big.nr, big.nc, big.nnz, nv, big.d_rp.ptr, big.d_ri.ptr, big.d_ci.ptr, big.d_v.ptr,
        big.d_B.ptr, big.d_C.ptr, st))
    assert status == D.STATUS_SUCCESS, D.status_string(status)
    ex = C.c_void_p()
    assert h.hipGraphInstantiate(C.byref(ex), graph, None, None, 0) == 0
    for _ in range(3):
        big.fill_output(np.nan)
        assert h.hipGraphLaunch(ex, st) == 0
        D.synchronize()
        assert_bitwise(big.output(nv) + 0.0, big.ref(D.DENSE_COL_MAJOR, nv)[0] + 0.0, "replay")
    h.hipGraphExecDestroy(ex)
    h.hipGraphDestroy(graph)


def test_threads_share_no_scratch(big):
    """Two threads on the default stream, two on streams of their own."""
    widths, fails = [8, 64, 16, 33], []
    refs = [big.ref(D.DENSE_COL_MAJOR, nv)[0] + 0.0 for nv in widths]
    streams = [None, None, stream(), stream()]
    outs = [D.DeviceArray.zeros(big.nr * nv) for nv in widths]
    D.synchronize()

    def work(i):
        for k in range(6):
            launch(big, COL[k % 2], widths[i], streams[i], outs[i])
            D.check(D.lib().dspmm_stream_synchronize(streams[i]), "sync")
            if not np.array_equal(outs[i].numpy() + 0.0, refs[i]):
                fails.append((i, k))

    ts = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not fails, fails


@pytest.mark.parametrize("name", ["spmm_csr_vector_col", "spmm_coo_vector_col"])
def test_columns_in_slabs(name):
    """Copies of more than 256 MiB: B of 2.2 M rows, 32 columns in two slabs and
    25 with a narrower last one."""
    rng = np.random.default_rng(5)
    lens = np.full(40000, 5)
    c = int_case("slabs", lens, 2_200_000, 1)
    for nv in (32, 25):
        B = np.resize(rng.integers(-3, 4, 99991).astype(np.float32), c.nc * nv)
        c.B, c.d_B, c.maxnv, c._ref = B, D.DeviceArray.from_numpy(B), nv, {}
        c.d_C = D.DeviceArray.zeros(c.nr * nv)
        launch(c, name, nv)
        D.synchronize()
        assert_bitwise(c.output(nv) + 0.0, c.ref(D.DENSE_COL_MAJOR, nv)[0] + 0.0, f"{name} {nv}")


@pytest.mark.parametrize("kind", ["tiny", "uniform_100", "one_long", "many_long"])
def test_csr_long_rows(kind):
    lens = row_lengths(kind)
    c = int_case(kind, lens, 3000, 260)
    for nv in (1, 2, 3, 4, 5, 8, 16, 17, 33, 64, 65, 128, 257, 260):
        for name, layout in (("spmm_csr_vector_row", D.DENSE_ROW_MAJOR),
                             ("spmm_csr_vector_col", D.DENSE_COL_MAJOR)):
            note(f"{kind} {name} nv={nv}")
            c.fill_output(np.nan)
            launch(c, name, nv)
            D.synchronize()
            assert_bitwise(c.output(nv) + 0.0, c.ref(layout, nv)[0] + 0.0, f"{kind} {name} nv={nv}")


@pytest.mark.parametrize("kind", ["tiny", "one_long", "many_long"])
def test_csr_scalar_col_bit_exact(kind):
    """In place and on copies, floats of the host loop's order."""
    c = float_case(kind, row_lengths(kind), 3000, 260)
    for nv in (2, 3, 4, 7, 8, 9, 20, 257):
        c.fill_output(np.nan)
        launch(c, "spmm_csr_scalar_col", nv)
        D.synchronize()
        assert_bitwise(c.output(nv), c.ref(D.DENSE_COL_MAJOR, nv)[0], f"{kind} nv={nv}")


def test_coo_in_any_order():
    """Rows that come back after others: every visit is added once."""
    rng = np.random.default_rng(17)
    c = int_case("shuffled", rng.integers(0, 60, 700), 300, 65)
    row = c.rowIdx.copy()
    perm = np.arange(c.nnz)
    for at in range(0, c.nnz - 64, 64):          # few rows to a wavefront, in turns
        rng.shuffle(perm[at:at + 64])
    c.d_ri = D.DeviceArray.from_numpy(row[perm])
    c.d_ci = D.DeviceArray.from_numpy(c.colIdx[perm])
    c.d_v = D.DeviceArray.from_numpy(c.values[perm])
    for nv in (1, 2, 4, 8, 16, 32, 64, 65):
        for name, layout in (("spmm_coo_scalar_row", D.DENSE_ROW_MAJOR),
                             ("spmm_coo_scalar_col", D.DENSE_COL_MAJOR)):
            c.fill_output(0.0)
            launch(c, name, nv)
            D.synchronize()
            assert_bitwise(c.output(nv) + 0.0, c.ref(layout, nv)[0] + 0.0, f"{name} nv={nv}")


@pytest.mark.parametrize("kind", ["even_16", "ends_together", "sparse_runs"])
def test_coo_long_runs(kind):
    """Runs that several groups finish at once and at different steps, four
    columns to a lane."""
    rng = np.random.default_rng(3)
    lens = {"even_16": np.full(777, 16), "ends_together": np.tile([8, 24, 32, 8], 1500),
            "sparse_runs": rng.integers(0, 3, 5000) * 27}[kind]
    c = int_case(kind, lens, 400, 132)
    for nv in (4, 8, 12, 16, 20, 32, 48, 64, 68, 128, 132):
        c.fill_output(1.0)
        launch(c, "spmm_coo_vector_row", nv)
        D.synchronize()
        assert_bitwise(c.output(nv) + 0.0, c.ref(D.DENSE_ROW_MAJOR, nv)[0] + 1.0, f"{kind} nv={nv}")
