"""Row-balanced kernels where the long rows are neighbours or all rows are long:
results as ever, and no longer than a small multiple of the time that the same
work takes in another order (one block on hundreds of long rows took 10 to 60
times that).  The time limits are wide: they tell a serial chain of rows from
a busy GPU, not one microsecond from another.
"""
import numpy as np
import pytest

import dspmm as D
from gpu_common import Case, assert_bitwise, assert_fp32, note

pytestmark = pytest.mark.gpu
RM = D.DENSE_ROW_MAJOR


def make(name, lens, nc=6000, maxnv=64, seed=6):
    rng = np.random.default_rng(seed)
    rp = np.concatenate([[0], np.cumsum(np.asarray(lens, np.int64))])
    n = int(rp[-1])
    return Case(name, len(lens), nc, rp, rng.integers(0, nc, n),
                rng.standard_normal(n).astype(np.float32), maxnv,
                B=rng.uniform(-1, 1, nc * maxnv).astype(np.float32))


def lengths(kind):
    rng = np.random.default_rng(4)
    if kind == "long_block":                   # 512 long rows side by side
        return np.where(np.arange(4096) < 512, 2000, 4)
    if kind == "sorted":                       # a power law, longest rows first
        return np.sort(np.minimum(3000, rng.pareto(0.8, 65536).astype(np.int64) + 1))[::-1]
    return np.full(2048, 2000)                 # "all_long"


def reference(kind, lens):
    """The same nonzeros as rows in random order, or cut into rows of 250."""
    if kind == "all_long":
        return np.full(len(lens) * 8, 250)
    return np.random.default_rng(5).permutation(lens)


@pytest.mark.parametrize("kind", ["long_block", "sorted", "all_long"])
def test_long_rows_side_by_side(kind):
    lens = lengths(kind)
    c, r = make(kind, lens), make(kind + " spread", reference(kind, lens))
    for nv in (1, 8, 16, 64):
        for alg, name in ((D.ALG_CSR_SCALAR, "spmm_csr_scalar_row"), (D.ALG_CSR_VECTOR, "spmm_csr_vector_row")):
            note(f"{kind} {name} nv={nv}")
            c.fill_output(np.nan)
            st = D.launch(name, c.nr, c.nc, c.nnz, nv, c.d_rp, c.d_ri, c.d_ci, c.d_v, c.d_B, c.d_C)
            assert st == 0, D.status_string(st)
            D.synchronize()
            h32, c64, ab = c.ref(RM, nv)
            if alg == D.ALG_CSR_SCALAR:
                assert_bitwise(c.output(nv), h32, f"{kind} nv={nv}")
            else:
                assert_fp32(c.output(nv), c64, ab, c.rowlen_flat(RM, nv), kind, h32)
            if nv == 1 and alg == D.ALG_CSR_SCALAR:
                continue                       # a wavefront adds its rows in order there
            t = min(c.problem().benchmark(RM, nv, alg, 3, 10) for _ in range(3))
            t0 = min(r.problem().benchmark(RM, nv, alg, 3, 10) for _ in range(3))
            note(f"{kind} {name} nv={nv}: {1e3 * t:.1f} us, spread {1e3 * t0:.1f} us")
            assert t < 5 * t0 + 0.02, f"{kind} {name} nv={nv}: {t} ms against {t0} ms"


@pytest.mark.parametrize("nv", [2, 4])
def test_uniformly_long_rows(nv):
    """Rows past the length from which the vector kernel may gather four at a
    time: above a launch's 3 us no more per nonzero than rows short of it."""
    ms = []
    rng = np.random.default_rng(7)
    for n in (440, 800):
        col = np.sort(rng.integers(0, 20000, (4800, n)), axis=1).reshape(-1)
        c = Case(f"rows of {n}", 4800, 20000, np.arange(4801) * n, col, rng.standard_normal(col.size).astype(np.float32),
                 4, B=rng.uniform(-1, 1, 20000 * 4).astype(np.float32))
        c.fill_output(np.nan)
        ms.append(min(c.problem().benchmark(RM, nv, D.ALG_CSR_VECTOR, 5, 30) for _ in range(5)))
        h32, c64, ab = c.ref(RM, nv)
        assert_fp32(c.output(nv), c64, ab, c.rowlen_flat(RM, nv), c.name, h32)
    note(f"nv={nv}: rows of 440 {ms[0]:.4f} ms, of 800 {ms[1]:.4f} ms")
    assert ms[1] <= 1.05 * (0.003 + (ms[0] - 0.003) * 800 / 440)
