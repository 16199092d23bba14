"""Formats built from a CSR (the CSC transpose, the CSR5 copy) where the
building kernels' tiles end: row lengths around a tile, long runs of empty
rows, nonzero counts around a tile's multiples; products on each format
against the FP64 oracle."""
import numpy as np
import pytest

import oracle
import spmspv_amd as sa

pytestmark = pytest.mark.gpu


def csr_of_lengths(lengths, n, seed):
    rng = np.random.default_rng(seed)
    lengths = np.asarray(lengths)
    rp = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    col = np.empty(rp[-1], np.int32)
    for r in np.nonzero(lengths)[0]:
        col[rp[r]:rp[r + 1]] = np.sort(rng.choice(n, size=lengths[r], replace=False))
    return rp, col, rng.uniform(0.1, 1, rp[-1]).astype(np.float32)


SHAPES = {
    "one": ([1], 1),
    "tile": ([2304], 5000),
    "tile-1": ([2303], 5000),
    "tile+1": ([2304, 1], 5000),
    "empty-runs": ([0] * 3000 + [3] + [0] * 9000 + [2303, 1] + [0] * 2500 + [5] * 40 + [0] * 5000, 4000),
    "sparse-rows": ([1 if r % 300 == 7 else 0 for r in range(200000)], 3000),
    "short-rows": ([r % 3 for r in range(30011)], 70000),
    "windows": ([6143, 6144, 6145, 1, 6144, 6144, 0, 12287, 2, 20000, 6145], 30000),
    "half-windows": ([3071, 3072, 3073, 1, 3072, 3072, 0, 6143, 2, 6144, 3073], 30000),
    "long-and-short": ([9000] + [r % 5 for r in range(9001)] + [15000, 1, 0, 7000], 66000),
}


@pytest.mark.parametrize("shape", sorted(SHAPES))
def test_formats_of_row_lengths(gpu, shape):
    lengths, n = SHAPES[shape]
    m = len(lengths)
    rp, col, val = csr_of_lengths(lengths, n, m)
    M = sa.Matrix(m, n, rp, col, val)
    cp, ri, cv = oracle.csr_to_csc(m, n, rp, col, val)
    rng = np.random.default_rng(n)
    key = np.arange(n, dtype=np.int32)
    x = rng.uniform(-1, 1, n).astype(np.float32)
    dk, dv = sa.DeviceArray.from_host(key, np.int32), sa.DeviceArray.from_host(x, np.float32)
    yk, yv = sa.DeviceArray(m, np.int32), sa.DeviceArray(m, np.float32)
    ek, ev, eb = oracle.spmspv_f64(m, cp, ri, cv, key, x)
    for sigma in (8, 16, 24, 32):
        M.A.set_spmv_type(1)
        M.A.set_sigma(sigma)
        M.A.csr5_preprocess()
        for slot in (sa.K_COL_LB_SORT, sa.K_SPMV_LB):
            M.A.set_sparse_x(dk, dv, n)
            cnt = M.A.run(slot, y_key=yk, y_val=yv)
            np.testing.assert_array_equal(yk.to_host(cnt), ek, err_msg=f"sigma {sigma} slot {slot}")
            assert np.all(np.abs(yv.to_host(cnt).astype(np.float64) - ev) <= 1e-5 * eb + 1e-30)
        # a dense y, every row written (rows through several tiles, empty rows)
        yd = sa.DeviceArray.from_host(np.full(m, np.nan, np.float32), np.float32)
        M.A.set_sparse_x(dk, dv, n)
        M.A.run(sa.K_SPMV_LB, y_dense=yd, want_nnz=False)
        ref, bound = np.zeros(m), np.zeros(m)
        ref[ek], bound[ek] = ev, eb
        assert np.all(np.abs(yd.to_host() - ref) <= 1e-5 * bound + 1e-30), f"sigma {sigma} dense"
