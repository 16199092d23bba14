"""A speculated sort slot covers a few times the products of the size class's
last call: calls of one class whose products grow and shrink by more than
that, with and without a count, each against the FP64 oracle."""
import numpy as np
import pytest

import oracle
import spmspv_amd as sa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("slot", [sa.K_COL_NAIVE_SORT, sa.K_COL_LB_SORT])
def test_products_outgrow_the_guess(gpu, slot):
    import scipy.sparse as sp
    m, n = 30011, 40000
    rng = np.random.default_rng(slot)
    # 20,000 columns of one entry, 20,000 of thirty
    per = np.where(np.arange(n) < n // 2, 1, 30)
    cols = np.repeat(np.arange(n), per)
    R = sp.csr_matrix((np.ones(cols.size, np.float32), (rng.integers(0, m, cols.size), cols)), shape=(m, n))
    R.sort_indices()
    R.data = rng.uniform(0.1, 1, R.nnz).astype(np.float32)
    M = sa.Matrix(m, n, R.indptr.astype(np.int32), R.indices.astype(np.int32), R.data)
    cp, ri, cv = oracle.csr_to_csc(m, n, R.indptr, R.indices, R.data)
    yk, yv = sa.DeviceArray(m, np.int32), sa.DeviceArray(m, np.float32)
    yd = sa.DeviceArray(m, np.float32)
    M.A.selector_mode(2, slot)
    M.A.set_small_x_path(False)
    k = 9000  # one size class throughout
    for i, heavy in enumerate([0, 0, k, k, 0, k, 4000, 0]):
        key = np.sort(np.concatenate([rng.choice(n // 2, k - heavy, replace=False),
                                      n // 2 + rng.choice(n // 2, heavy, replace=False)])).astype(np.int32)
        val = rng.uniform(-1, 1, k).astype(np.float32)
        dk, dv = sa.DeviceArray.from_host(key, np.int32), sa.DeviceArray.from_host(val, np.float32)
        M.A.set_sparse_x(dk, dv, k)
        dense = i % 3 == 2
        cnt, used = M.A.run_auto(y_dense=yd if dense else None, y_key=yk, y_val=yv)
        assert used == slot
        ek, ev, eb = oracle.spmspv_f64(m, cp, ri, cv, key, val)
        np.testing.assert_array_equal(yk.to_host(cnt), ek)
        assert np.all(np.abs(yv.to_host(cnt).astype(np.float64) - ev) <= 1e-5 * eb + 1e-30)
        if dense:
            ref = np.zeros(m)
            ref[ek] = ev
            assert np.all(np.abs(yd.to_host() - ref) <= 1e-5 * np.abs(ref).max() + 1e-30)
