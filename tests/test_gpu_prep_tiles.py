"""The column scan at the edges of its tiles (1,024 keys) and of the look-back's
window of 64 tiles: bin_len and the longest column exactly, the load-balanced
product against the FP64 oracle."""
import numpy as np
import pytest

import oracle
import spmspv_amd as sa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [0, 1, 1023, 1024, 1025, 2049, 64 * 1024, 64 * 1024 + 1, 66 * 1024 - 1, 131073])
def test_scan_edges(gpu, k):
    scale = 18
    rp, col, val = sa.gen_rmat_csr(scale, 4, seed=3)
    n = 1 << scale
    M = sa.Matrix(n, n, rp, col, val)
    M.A.set_small_x_path(False)
    cp, ri, cv = oracle.csr_to_csc(n, n, rp, col, val)
    rng = np.random.default_rng(k)
    key = np.sort(rng.choice(n, k, replace=False)).astype(np.int32)
    xv = rng.uniform(-1, 1, k).astype(np.float32)
    dk = sa.DeviceArray.from_host(key if k else np.zeros(1, np.int32), np.int32)
    dv = sa.DeviceArray.from_host(xv if k else np.zeros(1, np.float32), np.float32)
    M.A.set_sparse_x(dk, dv, k)
    lens = np.diff(cp)[key]
    assert M.A.computeBinlen() == lens.sum()
    yk, yv = sa.DeviceArray(n, np.int32), sa.DeviceArray(n, np.float32)
    for slot in (sa.K_COL_LB_ATOMIC, sa.K_COL_LB_SORT, sa.K_COL_BUCKET):
        M.A.set_sparse_x(dk, dv, k)
        cnt = M.A.run(slot, y_key=yk, y_val=yv)
        ek, ev, eb = oracle.spmspv_f64(n, cp, ri, cv, key, xv)
        np.testing.assert_array_equal(yk.to_host(cnt), ek)
        assert np.all(np.abs(yv.to_host(cnt).astype(np.float64) - ev) <= 1e-5 * eb + 1e-30)
