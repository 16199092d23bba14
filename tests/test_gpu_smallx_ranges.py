"""The single-launch small-x path where its workgroups' row ranges end: row
counts around one workgroup's rows and around the number of workgroups, rows
at both ends of a range, rows with many products, special values, against the
FP64 oracle; and the same result bit for bit on a second call."""
import numpy as np
import pytest

import oracle
import spmspv_amd as sa

pytestmark = pytest.mark.gpu


def run_both(m, n, R, key, val):
    M = sa.Matrix(m, n, R.indptr.astype(np.int32), R.indices.astype(np.int32), R.data)
    dk, dv = sa.DeviceArray.from_host(key, np.int32), sa.DeviceArray.from_host(val, np.float32)
    yk, yv = sa.DeviceArray(m, np.int32), sa.DeviceArray(m, np.float32)
    out = []
    for how in ("auto", "auto", 0, 3):
        M.A.set_sparse_x(dk, dv, key.size)
        if how == "auto":
            cnt, used = M.A.run_auto(y_key=yk, y_val=yv)
            assert used == sa.K_COL_NAIVE_SORT
        else:
            cnt = M.A.run(how, y_key=yk, y_val=yv)
        out.append((yk.to_host(cnt), yv.to_host(cnt)))
    for k, v in out[1:]:
        np.testing.assert_array_equal(k, out[0][0])
        np.testing.assert_array_equal(v.view(np.int32), out[0][1].view(np.int32))
    return out[0]


@pytest.mark.parametrize("m", [1, 31, 33, 8191, 8192, 8193, 262143, 262145, (1 << 22) - 1, (1 << 22) + 1])
@pytest.mark.parametrize("per", [1, 40])
def test_row_ranges(gpu, m, per):
    import scipy.sparse as sp
    n = 270
    rng = np.random.default_rng(m + per)
    cols = np.repeat(np.arange(n), per)
    rows = rng.integers(0, m, cols.size)
    groups = max(min(32, -(-m // 8192)), -(-m // 131072))
    edge = -(-m // groups)  # rows per workgroup
    rows[::3] = np.clip(rng.integers(0, groups + 1, rows[::3].size) * edge - rng.integers(0, 2, rows[::3].size), 0, m - 1)
    rows[1::4] = m - 1
    R = sp.csr_matrix((np.ones(rows.size, np.float32), (rows, cols)), shape=(m, n))
    R.sort_indices()
    R.data = rng.uniform(-1, 1, R.nnz).astype(np.float32)
    cp, ri, cv = oracle.csr_to_csc(m, n, R.indptr, R.indices, R.data)
    key = np.arange(n, dtype=np.int32)
    # values over many orders of magnitude: each row's sum keeps its own scale
    val = (rng.uniform(0.5, 1, n) * 10.0 ** rng.integers(-20, 18, n)).astype(np.float32)
    ek, ev, eb = oracle.spmspv_f64(m, cp, ri, cv, key, val)
    k, v = run_both(m, n, R, key, val)
    np.testing.assert_array_equal(k, ek)
    assert np.all(np.abs(v.astype(np.float64) - ev) <= 1e-5 * eb + 1e-30)


def test_special_values(gpu):
    import scipy.sparse as sp
    m, n = 20000, 64
    rng = np.random.default_rng(5)
    cols = np.repeat(np.arange(n), 50)
    rows = rng.integers(0, m, cols.size)
    R = sp.csr_matrix((np.ones(rows.size, np.float32), (rows, cols)), shape=(m, n))
    R.sort_indices()
    R.data = rng.uniform(0.5, 1, R.nnz).astype(np.float32)
    cp, ri, cv = oracle.csr_to_csc(m, n, R.indptr, R.indices, R.data)
    key = np.arange(n, dtype=np.int32)
    val = rng.uniform(0.5, 1, n).astype(np.float32)
    val[3], val[10], val[20] = np.inf, np.nan, 0.0
    ek, ev, eb = oracle.spmspv_f64(m, cp, ri, cv, key, val)
    M = sa.Matrix(m, n, R.indptr.astype(np.int32), R.indices.astype(np.int32), R.data)
    dk, dv = sa.DeviceArray.from_host(key, np.int32), sa.DeviceArray.from_host(val, np.float32)
    yk, yv = sa.DeviceArray(m, np.int32), sa.DeviceArray(m, np.float32)
    M.A.set_sparse_x(dk, dv, n)
    cnt, _ = M.A.run_auto(y_key=yk, y_val=yv)
    k, v = yk.to_host(cnt), yv.to_host(cnt).astype(np.float64)
    np.testing.assert_array_equal(k, ek)
    np.testing.assert_array_equal(np.isnan(v), np.isnan(ev))
    np.testing.assert_array_equal(np.isinf(v), np.isinf(ev))
    fine = np.isfinite(ev)
    assert np.all(np.abs(v[fine] - ev[fine]) <= 1e-5 * eb[fine] + 1e-30)
