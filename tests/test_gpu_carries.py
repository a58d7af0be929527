"""Calls that have little room for the carries of split rows: AUTO without
allocation, a caller's small workspace, a server's small arena.  Where tiles of
16 nonzeros per lane fit, they run.
"""
import numpy as np
import pytest

import dspmm as D
import oracle as O
import workloads as W
from gpu_common import assert_bf16, assert_fp32, note

pytestmark = pytest.mark.gpu
RM, CM = D.DENSE_ROW_MAJOR, D.DENSE_COL_MAJOR
MIB = 1 << 20


@pytest.fixture(scope="module")
def power_law():
    """Rows of up to 5000 nonzeros; at nv = 256, 64 per tile need 79 MB of carries."""
    a = W.gen_csr(W.GEN_ZIPF, 262144, 262144, 17, 1.8, 1, 5000, W.VAL_NORMAL)
    m = D.Matrix(a.nr, a.nc, a.rowPtr, a.colIdx, a.values)
    yield a, m
    m.close()


def some_rows(a, B, got, what):
    """1500 rows, the longest among them, against 64 bits."""
    lens = np.diff(a.rowPtr)
    pick = np.unique(np.concatenate([np.argsort(lens)[-200:], np.arange(0, a.nr, a.nr // 1300)]))
    rp = np.concatenate([[0], np.cumsum(lens[pick])]).astype(np.int32)
    at = np.concatenate([np.arange(a.rowPtr[r], a.rowPtr[r + 1]) for r in pick])
    c64, ab = O.spmm_fp64(RM, pick.size, a.nc, B.shape[1], rp, a.colIdx[at], a.values[at], B)
    assert_bf16(got[pick].reshape(-1), c64.reshape(-1), ab.reshape(-1), what)


@pytest.mark.parametrize("layout", [RM, CM])
def test_noalloc_auto(power_law, layout):
    a, m = power_law
    nv = 256 if layout == RM else 24
    B = np.random.default_rng(2).uniform(-1, 1, (a.nc, nv)).astype(np.float32)
    d_B = D.to_bf16_device(D.DeviceArray.from_numpy(B if layout == RM else np.ascontiguousarray(B.T)))
    d_C = D.DeviceArray.from_numpy(np.full((a.nr, nv), np.nan, np.float32))
    bt = D.DSPMM_R_16BF
    m.prepare(d_B, d_C, nv, layout, btype=bt)
    note(f"workspace {m.workspace_size(nv, layout, bt) / MIB:.1f} MiB")
    ld = (nv, nv) if layout == RM else (a.nc, a.nr)
    st = D.lib().dspmm_spmm_ex_noalloc(m.handle, layout, nv, d_B.ptr, ld[0], bt, d_C.ptr, ld[1], None, None)
    assert st == 0, D.status_string(st)
    D.synchronize()
    got = d_C.numpy().reshape((a.nr, nv) if layout == RM else (nv, a.nr))
    some_rows(a, B, got if layout == RM else got.T, f"noalloc layout {layout}")


def test_small_workspace(power_law):
    """What 256 nonzeros per tile need is enough, one byte less is not."""
    a, m = power_law
    nv, bt = 128, D.DSPMM_R_16BF
    lens = np.diff(a.rowPtr)
    need = int(np.sum(-(-lens[lens > 256] // 256))) * nv * 4
    B = np.random.default_rng(3).uniform(-1, 1, (a.nc, nv)).astype(np.float32)
    d_B = D.to_bf16_device(D.DeviceArray.from_numpy(B))
    d_C = D.DeviceArray.from_numpy(np.full((a.nr, nv), np.nan, np.float32))
    ws = D.DeviceArray.zeros(need // 4)
    assert m.workspace_size(nv, btype=bt) > need
    m.spmm(d_B, d_C, nv, btype=bt, workspace=ws, workspace_bytes=need)
    D.synchronize()
    some_rows(a, B, d_C.numpy().reshape(a.nr, nv), "small workspace")
    st = D.lib().dspmm_spmm_ex(m.handle, RM, nv, d_B.ptr, nv, bt, d_C.ptr, nv, None, ws.ptr, need - 1, None)
    assert st == D.STATUS_WORKSPACE_TOO_SMALL


@pytest.mark.parametrize("alone", [False, True])
@pytest.mark.parametrize("nv,btype", [(1, D.DSPMM_R_32F), (32, D.DSPMM_R_16BF)])
def test_small_arena(alone, nv, btype):
    """An arena for the operands and the carries of 16 nonzeros per lane."""
    bf16 = btype == D.DSPMM_R_16BF
    a = W.gen_csr(W.GEN_ZIPF, 60000, 60000, 23, 1.6, 12, 2000, W.VAL_NORMAL)
    lens = np.diff(a.rowPtr)
    S = 16 if nv == 1 else 64                      # 16 per lane of 4 (BF16: 8) columns
    ld = -(-nv // 8) * 8
    up = lambda x: -(-x // 256) * 256
    size = (up(a.nc * nv * (2 if bf16 else 4)) + up(a.nr * nv * 4) +
            up(int(np.sum(-(-lens[lens > S] // S))) * ld * 4))
    srv = D.Server(cache_bytes=1 << 30, operand_bytes=size, max_inflight=1, max_batch=4, btype=btype,
                   alone_nnz=1 if alone else 0)
    mid = srv.add_matrix(a.nr, a.nc, a.rowPtr, a.colIdx, a.values)
    got = []
    for rid in (1, 2):
        assert srv.submit(srv.request(rid, mid, nv, 5)) == 0
        srv.drain()
        (c,) = srv.poll()
        assert c["status"] == 0, c
        got.append(D.device_read(c["C"], (a.nr * nv,)).copy())
        srv.release(rid)
    srv.close()
    assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32))
    B = D.seeded_uniform(5, a.nc * nv)
    Br = O.round_bf16(B) if bf16 else B
    h32 = O.spmm_host32(RM, a.nr, a.nc, nv, a.rowPtr, a.colIdx, a.values, Br).reshape(-1)
    c64, ab = O.spmm_fp64(RM, a.nr, a.nc, nv, a.rowPtr, a.colIdx, a.values, Br)
    assert_fp32(got[0], c64.reshape(-1), ab.reshape(-1), np.repeat(lens.astype(np.float64), nv), "served", h32)


def test_auto_keeps_short_tiles():
    """What no-alloc calls have for carries does not bound AUTO's: a product with
    room is no slower than with the tile of 16 nonzeros per lane."""
    a = W.gen_csr(W.GEN_ZIPF, 1000000, 1000000, 29, 1.6, 4, 2000, W.VAL_NORMAL)
    m = D.Matrix(a.nr, a.nc, a.rowPtr, a.colIdx, a.values)
    nv, bt = 64, D.DSPMM_R_16BF
    d_B = D.to_bf16_device(D.DeviceArray.from_numpy(
        np.random.default_rng(4).uniform(-1, 1, (a.nc, nv)).astype(np.float32)))
    d_C = D.DeviceArray.zeros(a.nr * nv)
    need = m.workspace_size(nv, btype=bt)
    ms = [min(m.benchmark(d_B, d_C, nv, btype=bt, config=c, warmup=2, reps=5, per_call=False)[0] for _ in range(3))
          for c in (None, D.make_config(D.VARIANT_NNZ_TILED))]
    note(f"{a.nnz} nonzeros, workspace {need / MIB:.0f} MiB: AUTO {ms[0]:.3f} ms, 16 per lane {ms[1]:.3f} ms")
    assert need > 64 * MIB and ms[0] <= 1.05 * ms[1]
    m.close()
