"""The server and SpMV on slices of diagonals, a second copy of the matrix:
counted as the cache's memory, not built where the cache has none left for them
or where the request does not run them."""
import numpy as np
import pytest

import dspmm as D
import oracle as O
import workloads as W
from gpu_common import assert_fp32, note

pytestmark = pytest.mark.gpu
RM = D.DENSE_ROW_MAJOR


def serve(a, cache_bytes, alone, plain=0):
    """y of one SpMV request, the cache's bytes before and after it, and the
    device memory that it took."""
    srv = D.Server(cache_bytes=cache_bytes, operand_bytes=256 << 20, max_inflight=1, max_batch=4,
                   plain=plain, alone_nnz=1 if alone else 0)
    mid = srv.add_matrix(a.nr, a.nc, a.rowPtr, a.colIdx, a.values, preload=True)
    w = W.gen_csr(W.GEN_FIXED, 500, 400, seed=3, p0=20)   # what the runtime loads on first use
    warm = srv.add_matrix(w.nr, w.nc, w.rowPtr, w.colIdx, w.values, preload=True)
    assert srv.submit(srv.request(0, warm, 1, 7)) == 0
    srv.drain()
    assert [c["status"] for c in srv.poll()] == [0]
    srv.release(0)
    used, free = srv.stats()["cache_used"], D.device_info()["free_mem"]
    assert srv.submit(srv.request(1, mid, 1, 99)) == 0
    srv.drain()
    (c,) = srv.poll()
    assert c["status"] == 0, c
    y = D.device_read(c["C"], (a.nr,)).copy()
    taken, now = free - D.device_info()["free_mem"], srv.stats()["cache_used"]
    srv.release(1)
    srv.close()
    x = D.seeded_uniform(99, a.nc)
    h32 = O.spmm_host32(RM, a.nr, a.nc, 1, a.rowPtr, a.colIdx, a.values, x).reshape(-1)
    c64, ab = O.spmm_fp64(RM, a.nr, a.nc, 1, a.rowPtr, a.colIdx, a.values, x)
    assert_fp32(y, c64.reshape(-1), ab.reshape(-1), np.diff(a.rowPtr).astype(np.float64), "y", h32)
    note(f"cache {used >> 20} -> {now >> 20} MiB, device {taken >> 20} MiB")
    return used, now, taken


def test_server_counts_slices():
    a = W.c3_matrix(80)                                   # slices of 75 MB
    est = 4 * (a.nr + 1) + 9 * a.nnz + a.nr + (1 << 20)
    used, now, taken = serve(a, 1 << 30, alone=True)
    assert now >= used + 5 * a.nnz
    used, now, taken = serve(a, est + (3 << 20), alone=True)
    assert now == used and taken < 2 * a.nnz
    used, now, taken = serve(a, est + (3 << 20), alone=False, plain=2)
    assert now == used and taken < 2 * a.nnz


def test_server_builds_no_slices_in_vain():
    a = W.c3_matrix(80)
    used, now, taken = serve(a, 1 << 30, alone=False)
    assert now == used and taken < 4 * a.nnz             # the batch's own tiles
