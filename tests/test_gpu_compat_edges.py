"""The reference-compatible kernels at the sizes where their blocking can go
wrong: the ends of a wavefront's nonzeros, groups with no work, rows that
cross groups, wavefronts and blocks, dense widths that no vector divides.
Operands are small integers, so every summation order gives the exact result.
"""
import numpy as np
import pytest

import dspmm as D
from gpu_common import Case, assert_bitwise, note

pytestmark = pytest.mark.gpu


def int_case(name, lens, nc, maxnv, seed=5):
    """Rows of the given lengths, |values| <= 3 and |B| <= 3 integers."""
    rng = np.random.default_rng(seed)
    lens = np.asarray(lens, np.int64)
    rp = np.concatenate([[0], np.cumsum(lens)])
    cols = rng.integers(0, nc, int(rp[-1]))
    vals = rng.integers(-3, 4, int(rp[-1])).astype(np.float32)
    B = rng.integers(-3, 4, nc * maxnv).astype(np.float32)
    return Case(name, len(lens), nc, rp, cols, vals, maxnv, B=B)


def check(c, name, nv, layout=D.DENSE_ROW_MAJOR):
    note(f"{c.name} {name} nv={nv}")
    coo = "coo" in name
    c.fill_output(0.0 if coo else np.nan)       # row-balanced kernels overwrite
    st = D.launch(name, c.nr, c.nc, c.nnz, nv, c.d_rp, c.d_ri, c.d_ci, c.d_v, c.d_B, c.d_C)
    assert st == 0, D.status_string(st)
    D.synchronize()
    # -0 (products of zeros) and +0 (the zeroed output) compare equal
    assert_bitwise(c.output(nv) + 0.0, c.ref(layout, nv)[0] + 0.0, f"{c.name} {name} nv={nv}")


LENGTHS = {
    "one": [1],
    "n63": [1] * 63,
    "n65": [65],
    "n257_one_row": [257],
    "n511_mixed": [1, 0, 0, 200, 7, 0, 300, 3],
    "n513_units": [1] * 513,
    "long_between": [3, 0, 5000, 1, 1, 0, 2, 700, 0],
    "empty_ends": [0, 0, 31, 33, 0, 64, 1, 0, 0],
}


@pytest.mark.parametrize("shape", LENGTHS, ids=list(LENGTHS))
def test_coo_row_major_edges(shape):
    c = int_case(shape, LENGTHS[shape], 37, 260)
    for nv in (1, 2, 3, 4, 8, 15, 16, 17, 32, 33, 64, 65, 96, 128, 257, 260):
        check(c, "spmm_coo_vector_row", nv)
    check(c, "spmv_coo_scalar", 1)
    check(c, "spmm_coo_scalar_row", 48)


def test_coo_row_major_large():
    """Enough nonzeros for the longest runs per group and for two chunks per
    wavefront at nv = 1, with rows longer than a wavefront's share."""
    rng = np.random.default_rng(9)
    lens = rng.integers(0, 40, 60000)
    lens[[0, 777, 59999]] = 3001
    c = int_case("large", lens, 5000, 64)
    for nv in (1, 2, 32, 64):
        check(c, "spmm_coo_vector_row", nv)


def float_case(name, lens, nc, maxnv, seed=6):
    rng = np.random.default_rng(seed)
    rp = np.concatenate([[0], np.cumsum(np.asarray(lens, np.int64))])
    n = int(rp[-1])
    return Case(name, len(lens), nc, rp, rng.integers(0, nc, n),
                rng.standard_normal(n).astype(np.float32), maxnv,
                B=rng.uniform(-1, 1, nc * maxnv).astype(np.float32))


def row_lengths(kind):
    rng = np.random.default_rng(11)
    if kind == "uniform_100":          # every row long against a window, none against the others
        return np.full(700, 100)
    if kind == "tiny":
        return np.array([1, 0, 70, 0, 2])
    lens = rng.integers(0, 12, 1300)   # three scouts' worth of rows
    if kind == "one_long":
        lens[5] = 5003
    elif kind == "many_long":
        at = rng.choice(1300, 40, replace=False)
        lens[at] = np.resize([95, 96, 97, 191, 255, 256, 257, 511, 512, 513, 1023, 1024, 1025, 1279,
                              1281, 2048, 63, 64, 65, 128], 40)
        lens[[0, 511, 512, 1299]] = 1100
    return lens


@pytest.mark.parametrize("kind", ["tiny", "uniform_100", "one_long", "many_long"])
def test_csr_scalar_long_rows_bit_exact(kind):
    """Rows summed by a lane, a group, a whole block and a scout equal the host
    loop bit for bit, whatever the number of columns."""
    c = float_case(kind, row_lengths(kind), 3000, 260)
    for nv in (1, 2, 3, 4, 5, 8, 9, 16, 17, 32, 33, 48, 64, 100, 128, 256, 260):
        name = "spmm_csr_scalar_row"
        note(f"{kind} {name} nv={nv}")
        c.fill_output(np.nan)
        st = D.launch(name, c.nr, c.nc, c.nnz, nv, c.d_rp, c.d_ri, c.d_ci, c.d_v, c.d_B, c.d_C)
        assert st == 0, D.status_string(st)
        D.synchronize()
        assert_bitwise(c.output(nv), c.ref(D.DENSE_ROW_MAJOR, nv)[0], f"{kind} nv={nv}")


def test_csr_scalar_many_rows_few_columns():
    """Enough rows for a lane group each at 5 to 8 columns, some of them long."""
    rng = np.random.default_rng(14)
    lens = rng.integers(0, 5, 98304)
    lens[[0, 511, 40000, 98303]] = [97, 1025, 300, 1300]
    c = float_case("many_rows", lens, 3000, 8)
    for nv in (4, 5, 6, 7, 8):
        c.fill_output(np.nan)
        st = D.launch("spmm_csr_scalar_row", c.nr, c.nc, c.nnz, nv, c.d_rp, c.d_ri, c.d_ci, c.d_v,
                      c.d_B, c.d_C)
        assert st == 0, D.status_string(st)
        D.synchronize()
        assert_bitwise(c.output(nv), c.ref(D.DENSE_ROW_MAJOR, nv)[0], f"many rows nv={nv}")
