"""Row-major kernels whose lanes may start anywhere in a row: dense widths
that no vector divides, odd leading dimensions and operands off their natural
alignment equal the host loop bit for bit and leave the padding alone; and
AUTO's choices over matrices, widths, layouts and types pass the gates.
"""
import numpy as np
import pytest

import dspmm as D
import oracle as O
import workloads as W
from gpu_common import assert_bitwise, assert_fp32, note

pytestmark = pytest.mark.gpu
RM, CM = D.DENSE_ROW_MAJOR, D.DENSE_COL_MAJOR

KERNELS = {
    "nnz_tiled": D.make_config(D.VARIANT_NNZ_TILED, tile_nnz=16),
    "nnz_tiled_vec2": D.make_config(D.VARIANT_NNZ_TILED, vec=2, lanes=4, tile_nnz=16, unroll=4),
    "row_seq": D.make_config(D.VARIANT_CSR_SCALAR, unroll=4),
    "row_seq_sliced": D.make_config(D.VARIANT_CSR_SCALAR, unroll=8, tile_nnz=1),
    "row_blocked": D.make_config(D.VARIANT_ROW_BLOCKED, tile_nnz=4),
    "csr_scalar": D.make_config(D.VARIANT_CSR_SCALAR),
    "csr_vector": D.make_config(D.VARIANT_CSR_VECTOR),
}
WIDTHS = (2, 3, 5, 6, 7, 9, 13, 31, 37, 65, 67, 130, 257)


def operand(a, off, bf16):
    """Device copy of `a` (floats) whose first element lies `off` elements
    into its allocation; the BF16 one is rounded on the device."""
    flat = np.concatenate([np.full(off, np.nan, np.float32), a.reshape(-1)])
    d = D.DeviceArray.from_numpy(flat)
    if bf16:
        d = D.to_bf16_device(d)
    return d, d.ptr + off * (2 if bf16 else 4)


# (the parallel reference class takes FP32 B only)
@pytest.mark.parametrize("kernel,bf16", [(k, b) for k in KERNELS for b in (False, True)
                                         if not (b and k == "csr_vector")])
def test_any_width_and_alignment(kernel, bf16):
    a = W.gen_csr(W.GEN_BINOMIAL, 203, 150, 17, p0=5.0)      # rows of at most a tile
    assert np.diff(a.rowPtr).max() <= 16
    m = D.Matrix(a.nr, a.nc, a.rowPtr, a.colIdx, a.values)
    rng = np.random.default_rng(4)
    for nv in WIDTHS:
        for pad_b, pad_c, off in ((0, 0, 0), (1, 0, 1), (3, 5, 3), (0, 8 - nv % 8, 0)):
            note(f"{kernel} bf16={bf16} nv={nv} pads {pad_b},{pad_c} offset {off}")
            B = rng.uniform(-1, 1, (a.nc, nv + pad_b)).astype(np.float32)
            keep, pB = operand(B, off, bf16)
            C = np.full(off + a.nr * (nv + pad_c), -7.0, np.float32)
            d_C = D.DeviceArray.from_numpy(C)
            m.spmm(pB, d_C.ptr + 4 * off, nv, ldb=nv + pad_b, ldc=nv + pad_c,
                   config=KERNELS[kernel], btype=D.DSPMM_R_16BF if bf16 else D.DSPMM_R_32F)
            D.synchronize()
            out = d_C.numpy()
            assert np.all(out[:off] == -7.0)
            out = out[off:].reshape(a.nr, nv + pad_c)
            assert np.all(out[:, nv:] == -7.0), "padding written"
            Bn = np.ascontiguousarray(B[:, :nv])
            ref = (a.rowPtr, a.colIdx, a.values, O.round_bf16(Bn) if bf16 else Bn)
            h32 = O.spmm_host32(RM, a.nr, a.nc, nv, *ref).reshape(-1)
            got = np.ascontiguousarray(out[:, :nv]).reshape(-1)
            if kernel == "csr_vector":
                c64, ab = O.spmm_fp64(RM, a.nr, a.nc, nv, *ref)
                assert_fp32(got, c64.reshape(-1), ab.reshape(-1),
                            np.repeat(np.diff(a.rowPtr).astype(np.float64), nv), kernel, h32)
            else:
                assert_bitwise(got, h32, f"{kernel} nv={nv}")
    m.close()


MATRICES = {
    "uniform": (W.GEN_FIXED, 900, 700, dict(p0=12)),
    "long_uniform": (W.GEN_FIXED, 400, 900, dict(p0=100)),   # rows overflow a wavefront's window
    "skewed": (W.GEN_ZIPF, 3000, 3000, dict(p0=1.6, p1=1, p2=900)),
    "stencil": (W.GEN_STENCIL27, 1728, 1728, dict(p0=12)),
}


@pytest.mark.parametrize("name", MATRICES)
@pytest.mark.parametrize("layout", [RM, CM], ids=["RM", "CM"])
@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
def test_auto_over_widths(name, layout, bf16):
    kind, nr, nc, p = MATRICES[name]
    a = W.gen_csr(kind, nr, nc, 23, **p)
    m = D.Matrix(a.nr, a.nc, a.rowPtr, a.colIdx, a.values)
    lens = np.diff(a.rowPtr).astype(np.float64)
    rng = np.random.default_rng(5)
    for nv in (2, 3, 8, 9, 16, 20, 32, 33, 64, 100, 129):
        note(f"AUTO {name} layout={layout} bf16={bf16} nv={nv}")
        B = rng.uniform(-1, 1, a.nc * nv).astype(np.float32)
        d_B = D.DeviceArray.from_numpy(B)
        if bf16:
            d_B = D.to_bf16_device(d_B)
        d_C = D.DeviceArray.from_numpy(np.full(a.nr * nv, np.nan, np.float32))
        m.spmm(d_B, d_C, nv, layout=layout, btype=D.DSPMM_R_16BF if bf16 else D.DSPMM_R_32F)
        D.synchronize()
        ref = (a.rowPtr, a.colIdx, a.values, O.round_bf16(B) if bf16 else B)
        h32 = O.spmm_host32(layout, a.nr, a.nc, nv, *ref).reshape(-1)
        c64, ab = O.spmm_fp64(layout, a.nr, a.nc, nv, *ref)
        n = np.repeat(lens, nv) if layout == RM else np.tile(lens, nv)
        assert_fp32(d_C.numpy(), c64.reshape(-1), ab.reshape(-1), n, f"{name} nv={nv}", h32)
    m.close()


@pytest.mark.parametrize("mean", [4, 37, 150])
def test_auto_accepts_every_width(mean):
    """The static default's tiles fit its kernels whatever lanes the width
    leaves a row (integers: every order is exact)."""
    rng = np.random.default_rng(mean)
    nr, nc = 120_000 // mean, 900
    rp = np.arange(nr + 1) * mean
    ci = np.sort(rng.permuted(np.tile(np.arange(nc), (nr, 1)), axis=1)[:, :mean], axis=1).ravel() \
        if nr * nc < 1 << 24 else rng.integers(0, nc, nr * mean)
    v = rng.integers(-3, 4, nr * mean).astype(np.float32)
    m = D.Matrix(nr, nc, rp, ci, v)
    for nv in (2, 3, 4, 5, 8, 9, 10, 16, 17, 32, 33, 64, 65):
        for layout, bf16 in ((RM, False), (RM, True), (CM, False), (CM, True)):
            note(f"mean {mean} nv={nv} layout={layout} bf16={bf16}")
            B = rng.integers(-3, 4, nc * nv).astype(np.float32)
            d_B = D.DeviceArray.from_numpy(B)
            d_b = D.to_bf16_device(d_B) if bf16 else d_B
            d_C = D.DeviceArray.zeros(nr * nv)
            m.spmm(d_b, d_C, nv, layout, btype=D.DSPMM_R_16BF if bf16 else D.DSPMM_R_32F)
            D.synchronize()
            ref = O.spmm_host32(layout, nr, nc, nv, rp, ci, v, B).reshape(-1)
            assert_bitwise(d_C.numpy().reshape(-1) + 0.0, ref + 0.0, f"nv={nv}")


def test_auto_accepts_narrow_bf16_of_many_rows():
    """Enough nonzeros for the static default's longest tiles, one lane each."""
    rng = np.random.default_rng(8)
    nr, nc, mean = 1_200_000, 5000, 4
    ci = rng.integers(0, nc, nr * mean)
    v = rng.integers(-3, 4, nr * mean).astype(np.float32)
    m = D.Matrix(nr, nc, np.arange(nr + 1) * mean, ci, v)
    for nv in (2, 3, 5):
        B = rng.integers(-3, 4, (nc, nv)).astype(np.float32)
        d_b = D.to_bf16_device(D.DeviceArray.from_numpy(B))
        d_C = D.DeviceArray.zeros(nr * nv)
        m.spmm(d_b, d_C, nv, btype=D.DSPMM_R_16BF)
        D.synchronize()
        ref = (v[:, None] * B[ci]).reshape(nr, mean, nv).sum(1)
        assert_bitwise(d_C.numpy().reshape(nr, nv) + 0.0, ref + 0.0, f"nv={nv}")
