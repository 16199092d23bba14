"""Radix passes whose scatter sums the digit counts itself: item counts at the
edges of a tile (3,072), of a chunk of 16 tiles and past the largest size of
that path, on one handle in an order that leaves the larger sort's counts
behind, for keys of 1 to 3 digits. Against the FP64 oracle."""
import numpy as np
import pytest

import oracle
import spmspv_amd as sa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("slot", [sa.K_COL_NAIVE_SORT, sa.K_COL_LB_SORT])
@pytest.mark.parametrize("m", [250, 40000, 700001, 3000001])
def test_count_edges(gpu, m, slot):
    import scipy.sparse as sp
    rng = np.random.default_rng(m)
    wide, ones = 300000, 64  # columns of 16 entries, then of one
    n = wide + ones
    cols = np.concatenate([np.repeat(np.arange(wide), 16), wide + np.arange(ones)])
    R = sp.csr_matrix((np.ones(cols.size, np.float32), (rng.integers(0, m, cols.size), cols)), shape=(m, n))
    R.sum_duplicates()
    R.sort_indices()
    R.data = rng.uniform(0.1, 1, R.nnz).astype(np.float32)
    M = sa.Matrix(m, n, R.indptr.astype(np.int32), R.indices.astype(np.int32), R.data)
    M.A.set_small_x_path(False)
    cp, ri, cv = oracle.csr_to_csc(m, n, R.indptr, R.indices, R.data)
    deg = np.diff(cp)
    yk, yv = sa.DeviceArray(m, np.int32), sa.DeviceArray(m, np.float32)
    for want in (49152, 3072, 4500000, 49153, 3073, 1000000, 49151, 2 * 49152 + 1, 6145, 4500000, 700003):
        # whole columns up to the size, single entries for the rest
        k = int(np.searchsorted(np.cumsum(deg[:wide]), want, side="right"))
        rest = want - int(deg[:k].sum())
        key = np.r_[np.arange(k), wide + np.arange(min(rest, ones))].astype(np.int32)
        xv = rng.uniform(-1, 1, key.size).astype(np.float32)
        dk, dv = sa.DeviceArray.from_host(key, np.int32), sa.DeviceArray.from_host(xv, np.float32)
        M.A.set_sparse_x(dk, dv, key.size)
        cnt = M.A.run(slot, y_key=yk, y_val=yv)
        ek, ev, eb = oracle.spmspv_f64(m, cp, ri, cv, key, xv)
        np.testing.assert_array_equal(yk.to_host(cnt), ek)
        assert np.all(np.abs(yv.to_host(cnt).astype(np.float64) - ev) <= 1e-5 * eb + 1e-30)
