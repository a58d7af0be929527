"""Rounding error of whole results against 64 bits, no larger than that of the
summation order that a path replaced: the order is computed here in FP32 on
the CPU, and a path may be 5% above it (the spread of such a measure over the
few hundred thousand outputs used).  Rows are of one length, so that one order
describes them all.
"""
import numpy as np
import pytest

import dspmm as D
from gpu_common import note

pytestmark = pytest.mark.gpu
F = np.float32
MARGIN = 1.05


def fma(a, b, c):
    return (a.astype(np.float64) * b.astype(np.float64) + c.astype(np.float64)).astype(F)


def chain(a, b):
    """One FMA after the other along the last axis."""
    s = np.zeros(np.broadcast_shapes(a.shape, b.shape)[:-1], F)
    for i in range(a.shape[-1]):
        s = fma(a[..., i], b[..., i], s)
    return s


def pairwise(parts):
    while len(parts) > 1:
        h = len(parts) // 2
        parts = [parts[i] + parts[i + h] for i in range(h)]
    return parts[0]


def over_lanes(a, b, lanes):
    """Lane l sums nonzeros l, l + lanes, ...; then a tree over the lanes."""
    n = a.shape[-1]
    return pairwise([chain(a[..., l:n:lanes], b[..., l:n:lanes]) if l < n else
                     np.zeros(b.shape[:-1], F) for l in range(lanes)])


def error(got, exact):
    return float(np.sqrt(((got - exact) ** 2).mean() / (exact ** 2).mean()))


class Rows:
    """nr rows of n nonzeros over nc columns; B of maxnv columns, row-major."""

    def __init__(self, nr, n, nc, maxnv, seed=3):
        rng = np.random.default_rng(seed)
        self.nr, self.n, self.nc = nr, n, nc
        self.col = np.sort(np.argsort(rng.random((nr, nc), F), axis=1)[:, :n], axis=1).astype(np.int32)
        self.val = rng.standard_normal((nr, n)).astype(F)
        self.B = rng.uniform(-1, 1, (nc, maxnv)).astype(F)
        self.ptr = (np.arange(nr + 1) * n).astype(np.int32)

    def operands(self, nv, cols):
        """Values and gathered B of the first `cols` columns, nonzeros last."""
        b = self.B[:, :cols][self.col]                     # nr, n, cols
        return self.val[:, None, :], np.ascontiguousarray(b.transpose(0, 2, 1))

    def exact(self, a, b):
        return (a.astype(np.float64) * b).sum(-1)


@pytest.mark.parametrize("n,nv", [(40, 64), (100, 64), (256, 128)])
def test_column_major_vector(n, nv):
    """spmm_csr_vector_col adds each row over up to 64 lanes, also where it
    runs on row-major copies."""
    cols = 16
    m = Rows(4000 if n < 200 else 2000, n, 3000, nv)
    a, b = m.operands(nv, cols)
    exact = m.exact(a, b)
    d = [D.DeviceArray.from_numpy(x) for x in (m.ptr, np.repeat(np.arange(m.nr, dtype=np.int32), n),
                                               m.col, m.val, np.ascontiguousarray(m.B[:, :nv].T))]
    out = D.DeviceArray.from_numpy(np.full((nv, m.nr), np.nan, F))
    st = D.launch("spmm_csr_vector_col", m.nr, m.nc, m.nr * n, nv, *d, out)
    assert st == 0, D.status_string(st)
    D.synchronize()
    got = error(out.numpy().T[:, :cols], exact)
    ref = error(over_lanes(a, b, 64 if n > 64 else 32), exact)
    note(f"rows of {n}, nv={nv}: {got:.3g}, over the lanes {ref:.3g}")
    assert got <= MARGIN * ref


@pytest.mark.parametrize("n", [20, 64, 100, 200, 256])
def test_spmv_tiles(n):
    """Rows of 17 to 256 nonzeros of an SpMV tile: products over 64 lanes, then
    a tree."""
    m = Rows(3000, n, 2500, 1)
    a, b = m.operands(1, 1)
    exact = m.exact(a, b)[:, 0]
    h = D.Matrix(m.nr, m.nc, m.ptr, m.col.reshape(-1), m.val.reshape(-1))
    d_x, d_y = D.DeviceArray.from_numpy(m.B[:, 0].copy()), D.DeviceArray.zeros(m.nr)
    h.spmm(d_x, d_y, 1, config=D.make_config(D.VARIANT_SPMV_TILED, tile_nnz=1024))
    D.synchronize()
    prod = (a * b)[:, 0, :]
    lanes = []
    for lane in range(64):
        s = np.zeros(m.nr, F)
        for i in range(lane, n, 64):
            s = s + prod[:, i]
        lanes.append(s)
    got, ref = error(d_y.numpy(), exact), error(pairwise(lanes), exact)
    note(f"rows of {n}: {got:.3g}, 64 lanes {ref:.3g}")
    assert got <= MARGIN * ref
    h.close()


@pytest.mark.parametrize("n", [27, 32, 33, 64, 256])
def test_spmv_band(n):
    """A banded matrix, which may run in slices of diagonals, rounds no worse
    than the tiles' 64 sums, and takes no longer than a multiple of the tiles."""
    rng = np.random.default_rng(n)
    nr = 4000
    nc = nr + 3 * n
    col = (np.arange(nr)[:, None] + 3 * np.arange(n)).astype(np.int32)
    val = rng.standard_normal((nr, n)).astype(F)
    x = rng.uniform(-1, 1, nc).astype(F)
    prod = val * x[col]
    exact = (val.astype(np.float64) * x[col]).sum(1)
    lanes = [chain(val[:, i::64], x[col][:, i::64]) if i < n else np.zeros(nr, F) for i in range(64)]
    ptr = (np.arange(nr + 1) * n).astype(np.int32)
    h = D.Matrix(nr, nc, ptr, col.reshape(-1), val.reshape(-1))
    # the same rows on scattered columns: no diagonals
    t = D.Matrix(nr, nc, ptr, np.sort(rng.permutation(nc)[:nc][col % nc], 1).reshape(-1), val.reshape(-1))
    d_x, d_y = D.DeviceArray.from_numpy(x), D.DeviceArray.zeros(nr)
    ms = {}
    for name, mat in (("band", h), ("scattered", t)):
        ms[name] = min(mat.benchmark(d_x, d_y, 1, warmup=5, reps=40, per_call=False)[0] for _ in range(3))
    h.spmm(d_x, d_y, 1)
    D.synchronize()
    got, ref = error(d_y.numpy(), exact), error(pairwise(lanes), exact)
    note(f"rows of {n}: {got:.3g}, 64 lanes {ref:.3g}; {ms}")
    assert got <= 1.15 * ref                   # 4000 outputs spread by a few percent
    assert ms["band"] <= 1.5 * ms["scattered"] + 0.002
    h.close()
    t.close()


def chunks(a, b, S):
    """Chunks of S nonzeros, each in order with a rounded product, added in order."""
    s = np.zeros(np.broadcast_shapes(a.shape, b.shape)[:-1], F)
    prod = a * b
    for c in range(0, a.shape[-1], S):
        t = np.zeros_like(s)
        for i in range(c, min(c + S, a.shape[-1])):
            t = t + prod[..., i]
        s = s + t
    return s


@pytest.mark.parametrize("bf16,layout,n,nv,S", [
    (True, "row", 20, 8, 16), (True, "row", 100, 2, 16), (True, "row", 100, 16, 32), (True, "row", 100, 48, 128),
    (True, "col", 100, 32, 64), (True, "row", 200, 12, 32), (True, "row", 250, 64, 128),
    (False, "col", 100, 16, 64), (False, "col", 200, 48, 256), (False, "col", 250, 12, 64)])
def test_auto(bf16, layout, n, nv, S):
    """AUTO rounds no worse than tiles of S nonzeros in order do, 16 per lane."""
    cols = min(nv, 16)
    m = Rows(4000, n, 3000, nv)
    d_B = D.DeviceArray.from_numpy(m.B if layout == "row" else np.ascontiguousarray(m.B.T))
    if bf16:
        d_B = D.to_bf16_device(d_B)
        m.B = (((m.B.view(np.uint32) + 0x7fff + ((m.B.view(np.uint32) >> 16) & 1)) >> 16) << 16).view(F)
    a, b = m.operands(nv, cols)
    exact = m.exact(a, b)
    out = D.DeviceArray.from_numpy(np.full((m.nr, nv) if layout == "row" else (nv, m.nr), np.nan, F))
    h = D.Matrix(m.nr, m.nc, m.ptr, m.col.reshape(-1), m.val.reshape(-1))
    h.spmm(d_B, out, nv, D.DENSE_ROW_MAJOR if layout == "row" else D.DENSE_COL_MAJOR,
           btype=D.DSPMM_R_16BF if bf16 else D.DSPMM_R_32F)
    D.synchronize()
    got = error((out.numpy() if layout == "row" else out.numpy().T)[:, :cols], exact)
    ref = error(chunks(a, b, S), exact)
    note(f"{'bf16' if bf16 else 'fp32'} {layout} rows of {n}, nv={nv}: {got:.3g}, tiles of {S} {ref:.3g}")
    assert got <= MARGIN * ref
    h.close()


@pytest.mark.parametrize("nv", [3, 5, 8, 12, 16, 32])
def test_auto_stencil(nv):
    """A 27-point stencil on 48^3, FP32: AUTO against sums over 8 lanes."""
    g = np.arange(48 ** 3).reshape(48, 48, 48)
    d = np.array([(x * 48 + y) * 48 + z for x in (-1, 0, 1) for y in (-1, 0, 1) for z in (-1, 0, 1)])
    col = (g[1:-1, 1:-1, 1:-1].reshape(-1, 1) + d).astype(np.int32)
    nr, nc = col.shape[0], 48 ** 3
    rng = np.random.default_rng(nv)
    val = rng.standard_normal(col.shape).astype(F)
    B = rng.uniform(-1, 1, (nc, nv)).astype(F)
    ptr = (np.arange(nr + 1) * 27).astype(np.int32)
    h = D.Matrix(nr, nc, ptr, col.reshape(-1), val.reshape(-1))
    out = D.DeviceArray.from_numpy(np.full((nr, nv), np.nan, F))
    h.spmm(D.DeviceArray.from_numpy(B), out, nv)
    D.synchronize()
    pick = np.arange(0, nr, 7)
    a, b = val[pick][:, None, :], np.ascontiguousarray(B[:, :8][col[pick]].transpose(0, 2, 1))
    exact = (a.astype(np.float64) * b).sum(-1)
    # (four threads to a row of more than 16 columns: in order, as always)
    ref = error(over_lanes(a, b, 8) if nv <= 16 else chunks(a, b, 27), exact)
    got = error(out.numpy()[pick][:, :8], exact)
    note(f"stencil, nv={nv}: {got:.3g}, over the lanes {ref:.3g}")
    assert got <= MARGIN * ref
    h.close()


def test_auto_clustered_rows():
    """Long rows side by side: AUTO's first call on a power law sorted by length
    within twice its tiles' time."""
    rng = np.random.default_rng(1)
    lens = np.sort(np.minimum(4000, (3 / rng.random(60000) ** 0.7).astype(int)))[::-1].copy()
    ptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    h = D.Matrix(60000, 60000, ptr, rng.integers(0, 60000, ptr[-1]).astype(np.int32),
                 rng.standard_normal(ptr[-1]).astype(F))
    for nv in (3, 8):
        B, out = D.DeviceArray.from_numpy(rng.uniform(-1, 1, (60000, nv)).astype(F)), D.DeviceArray.zeros(60000 * nv)
        tiles = D.make_config(D.VARIANT_NNZ_TILED)
        ms = [min(h.benchmark(B, out, nv, config=c, warmup=5, reps=20, per_call=False)[0] for _ in range(3))
              for c in (None, tiles)]
        note(f"nv={nv}: AUTO {ms[0]:.4f} ms, tiles {ms[1]:.4f} ms")
        assert ms[0] <= 2 * ms[1] + 0.002
    h.close()


def scanned(prod, row, nr):
    """Chunks of 64 products, each scanned by rows over 64 lanes (1, 2, 4, ...
    apart), a row's chunks added in order."""
    pad = -len(prod) % 64
    s = np.concatenate([prod, np.zeros(pad, F)]).reshape(-1, 64)
    key = np.concatenate([row, np.full(pad, nr)]).reshape(-1, 64)
    d = 1
    while d < 64:
        t = s.copy()
        t[:, d:] += np.where(key[:, d:] == key[:, :-d], s[:, :-d], F(0))
        s, d = t, 2 * d
    tail = np.concatenate([key[:, 1:] != key[:, :-1], np.ones((len(key), 1), bool)], 1)
    y = np.zeros(nr + 1, F)
    np.add.at(y, key[tail], s[tail])
    return y[:nr]


@pytest.mark.parametrize("fn", ["spmv_coo_scalar", "spmv_coo_vector"])
@pytest.mark.parametrize("n", [20, 64, 100, 300])
def test_spmv_coo(fn, n):
    """A row that goes on in the next chunk adds to that chunk's sum."""
    nr, nc = 2000000 // n, 3000
    rng = np.random.default_rng(n)
    row = np.repeat(np.arange(nr, dtype=np.int32), n)
    col = rng.integers(0, nc, nr * n).astype(np.int32)
    val, x = rng.standard_normal(nr * n).astype(F), rng.uniform(-1, 1, nc).astype(F)
    exact = (val.astype(np.float64) * x[col]).reshape(nr, n).sum(1)
    ptr = (np.arange(nr + 1) * n).astype(np.int32)
    d = [D.DeviceArray.from_numpy(v) for v in (ptr, row, col, val, x)]
    out = D.DeviceArray.zeros(nr)
    st = D.launch(fn, nr, nc, nr * n, 1, *d, out)
    assert st == 0, D.status_string(st)
    D.synchronize()
    got, ref = error(out.numpy(), exact), error(scanned(val * x[col], row, nr), exact)
    note(f"{fn} rows of {n}: {got:.3g}, chunk by chunk {ref:.3g}")
    assert got <= MARGIN * ref


@pytest.mark.parametrize("bf16,nv", [(False, 1), (False, 2), (False, 4), (True, 1), (True, 8)])
def test_batch_long_rows(bf16, nv):
    """A narrow item of a batch: no worse than chunks of 16 added in order, in
    as many parts as lanes of a wavefront share a column."""
    m = Rows(4000, 256, 3000, nv)
    d_B = D.DeviceArray.from_numpy(m.B)
    if bf16:
        d_B = D.to_bf16_device(d_B)
        m.B = (((m.B.view(np.uint32) + 0x7fff + ((m.B.view(np.uint32) >> 16) & 1)) >> 16) << 16).view(F)
    a, b = m.operands(nv, nv)
    exact = m.exact(a, b)
    out = D.DeviceArray.from_numpy(np.full((m.nr, nv), np.nan, F))
    h = D.Matrix(m.nr, m.nc, m.ptr, m.col.reshape(-1), m.val.reshape(-1))
    batch = D.Batch([(h, nv, d_B, out)], btype=D.DSPMM_R_16BF if bf16 else D.DSPMM_R_32F)
    batch.run()
    D.synchronize()
    prod, parts, each = a * b, 64 // max(1, nv), []
    for c in range(0, 256, 16):
        t = np.zeros(prod.shape[:-1], F)
        for i in range(c, c + 16):
            t = t + prod[..., i]
        each.append(t)
    per = -(-len(each) // parts)
    ref = np.zeros_like(each[0])
    for p in range(0, len(each), per):
        t = np.zeros_like(ref)
        for c in each[p:p + per]:
            t = t + c
        ref = ref + t
    got, ref = error(out.numpy(), exact), error(ref, exact)
    note(f"{'bf16' if bf16 else 'fp32'} batch, rows of 256, nv={nv}: {got:.3g}, chunks of 16 {ref:.3g}")
    assert got <= MARGIN * ref
    batch.close()
    h.close()
