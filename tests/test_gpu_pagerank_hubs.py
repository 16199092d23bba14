"""PageRank on a graph whose columns lie around the length at which a column's
weights are summed by a whole workgroup, and whose active sets end around the
push kernel's tile, against the FP64 restatement; fixed and learned slots
agree."""
import numpy as np
import pytest

import oracle
import spmspv_amd as sa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2047, 2048, 2049, 9001])
def test_pagerank_hub_columns(gpu, n):
    import scipy.sparse as sp
    rng = np.random.default_rng(n)
    cols, rows = [], []
    for j, d in enumerate([1023, 1024, 1025, 1500, 0, 1]):  # the first columns
        rows.append(rng.choice(n, size=min(d, n), replace=False))
        cols.append(np.full(min(d, n), j))
    for j in range(6, n):
        d = int(rng.integers(0, 6))
        rows.append(rng.choice(n, size=d, replace=False))
        cols.append(np.full(d, j))
    rows, cols = np.concatenate(rows), np.concatenate(cols)
    R = sp.csr_matrix((rng.uniform(0.1, 1, rows.size).astype(np.float32), (rows, cols)), shape=(n, n))
    R.sort_indices()
    M = sa.Matrix(n, n, R.indptr.astype(np.int32), R.indices.astype(np.int32), R.data)
    cp, ri, cv = oracle.csr_to_csc(n, n, R.indptr, R.indices, R.data)
    ref = oracle.pagerank_f64(n, cp, ri, cv, 0.85, 1e-6, 400)[0]
    rank = sa.DeviceArray(n, np.float32)
    for policy in (-1, 2, 3, 5):
        st, sizes = M.A.pagerank(rank, damping=0.85, eps=1e-6, max_iter=400, policy=policy)
        got = rank.to_host().astype(np.float64)
        # residuals end below eps * (1 - d) / n each, in either precision
        assert np.abs(got - ref).sum() <= 2 * 1e-6 * 0.85 + 1e-5 * ref.sum()
        assert sizes[0] == n and int(st[3]) == 0
