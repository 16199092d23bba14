"""The sort slots at row counts around which the radix sort's digits change
their number and width, with products on both sides of the one-workgroup sort,
against the FP64 oracle."""
import numpy as np
import pytest

import oracle
import spmspv_amd as sa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("per", [1, 9])
@pytest.mark.parametrize("m", [2, 255, 257, 511, 65535, 65537, 131072, 131073, 1 << 17 | 12345])
def test_sort_slots_row_counts(gpu, m, per):
    import scipy.sparse as sp
    n = 4001
    rng = np.random.default_rng(m + per)
    # every second column hits row 0 or m - 1 as well: long runs of one digit
    cols = np.repeat(np.arange(n), per)
    rows = rng.integers(0, m, cols.size)
    rows[::5] = 0
    rows[1::7] = m - 1
    R = sp.csr_matrix((np.ones(rows.size, np.float32), (rows, cols)), shape=(m, n))
    R.sort_indices()
    R.data = rng.uniform(0.1, 1, R.nnz).astype(np.float32)
    M = sa.Matrix(m, n, R.indptr.astype(np.int32), R.indices.astype(np.int32), R.data)
    cp, ri, cv = oracle.csr_to_csc(m, n, R.indptr, R.indices, R.data)
    key = np.arange(n, dtype=np.int32)
    val = rng.uniform(-1, 1, n).astype(np.float32)
    dk, dv = sa.DeviceArray.from_host(key, np.int32), sa.DeviceArray.from_host(val, np.float32)
    yk, yv = sa.DeviceArray(m, np.int32), sa.DeviceArray(m, np.float32)
    ek, ev, eb = oracle.spmspv_f64(m, cp, ri, cv, key, val)
    M.A.set_small_x_path(False)
    for slot in (sa.K_COL_NAIVE_SORT, sa.K_COL_LB_SORT):
        M.A.set_sparse_x(dk, dv, n)
        cnt = M.A.run(slot, y_key=yk, y_val=yv)
        np.testing.assert_array_equal(yk.to_host(cnt), ek)
        assert np.all(np.abs(yv.to_host(cnt).astype(np.float64) - ev) <= 1e-5 * eb + 1e-30)
