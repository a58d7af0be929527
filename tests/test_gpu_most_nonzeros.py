"""The most nonzeros that 32-bit offsets allow, 2^31 - 1: windows and strides at
the end of the matrix stay inside it."""
import numpy as np
import pytest

import dspmm as D
from gpu_common import note

pytestmark = pytest.mark.gpu
NNZ, ROW = 2 ** 31 - 1, 8191


@pytest.fixture(scope="module")
def matrix():
    torch = pytest.importorskip("torch")
    if torch.cuda.mem_get_info()[0] < 40 << 30:
        pytest.skip("needs 40 GB")
    ptr = np.append(np.arange(0, NNZ, ROW, dtype=np.int64), NNZ).astype(np.int32)
    col = torch.ones(NNZ, dtype=torch.int32, device="cuda")
    val = torch.ones(NNZ, dtype=torch.float32, device="cuda")
    val[-1] = 3.0
    torch.cuda.synchronize()
    yield ptr, D.DeviceArray.from_numpy(ptr), col, val
    del col, val
    torch.cuda.empty_cache()


@pytest.mark.parametrize("name,nv", [("spmv_csr_scalar", 1), ("spmm_csr_scalar_row", 4), ("spmm_csr_scalar_row", 16),
                                     ("spmv_csr_vector", 1), ("spmm_csr_vector_row", 8)])
def test_offsets_up_to_the_limit(matrix, name, nv):
    ptr, d_ptr, col, val = matrix
    nr, nc = ptr.size - 1, 4
    B = (np.arange(nc * nv, dtype=np.float32) % 7).reshape(nc, nv)
    out = D.DeviceArray.from_numpy(np.full((nr, nv), np.nan, np.float32))
    note(f"{name} nv={nv}, {nr} rows")
    st = D.launch(name, nr, nc, NNZ, nv, d_ptr, d_ptr, col.data_ptr(), val.data_ptr(),
                  D.DeviceArray.from_numpy(B), out)
    assert st == 0, D.status_string(st)
    D.synchronize()
    sums = np.diff(ptr).astype(np.float64)
    sums[-1] += 2                              # whole numbers below 2^24: exact in any order
    assert np.array_equal(out.numpy().reshape(nr, nv), (sums[:, None] * B[1]).astype(np.float32))
