"""The CSC of a matrix around the size from which its sort runs in wide tiles
(6 * 2^20 nonzeros, tiles of 6,144), with columns of one entry and columns of many:
products through the CSC against the FP64 oracle."""
import numpy as np
import pytest

import oracle
import spmspv_amd as sa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("extra", [-1, 0, 1, 6143, 6145])
@pytest.mark.parametrize("n", [900, 70001])
def test_csc_around_the_wide_tiles(gpu, n, extra):
    nnz, per = (6 << 20) + extra, 16
    m = nnz // per + 700
    lens = np.zeros(m, np.int64)
    lens[: nnz // per] = per
    lens[nnz // per] = nnz % per
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    rng = np.random.default_rng(extra & 0xffff)
    start = rng.integers(0, n // 2, m)
    col = start[:, None] + np.cumsum(rng.integers(1, max(2, n // 36), (m, per)), axis=1)
    col = np.minimum(col, n - per + np.arange(per)).astype(np.int32).ravel()[:nnz]
    val = rng.uniform(0.1, 1, nnz).astype(np.float32)
    M = sa.Matrix(m, n, rp, col, val)
    M.A.set_small_x_path(False)
    csc = oracle.csr_to_csc(m, n, rp, col, val)
    yk, yv = sa.DeviceArray(m, np.int32), sa.DeviceArray(m, np.float32)
    for key in (np.arange(n), np.arange(3, n, 97), np.array([0, n // 2, n - 1])):
        key = key.astype(np.int32)
        x = rng.uniform(-1, 1, key.size).astype(np.float32)
        dk, dv = sa.DeviceArray.from_host(key, np.int32), sa.DeviceArray.from_host(x, np.float32)
        M.A.set_sparse_x(dk, dv, key.size)
        cnt = M.A.run(sa.K_COL_LB_SORT, y_key=yk, y_val=yv)
        ek, ev, eb = oracle.spmspv_f64(m, *csc, key, x)
        np.testing.assert_array_equal(yk.to_host(cnt), ek)
        assert np.all(np.abs(yv.to_host(cnt).astype(np.float64) - ev) <= 1e-5 * eb + 1e-30)
