"""The small-x launch's own gather: calls whose products outgrow the sorted
result's LDS and whose slot is an atomic one, around the limits (LDS
capacity, products per workgroup of the gather, one key, the most keys),
with the sizes of one class changing from call to call so that the queued
compaction is used, missed and run alone. Against the FP64 oracle."""
import numpy as np
import pytest

import oracle
import spmspv_amd as sa

pytestmark = pytest.mark.gpu


def matrix(m, lens, seed):
    """Columns of the given lengths on distinct random rows."""
    rng = np.random.default_rng(seed)
    n = len(lens)
    cp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    ri = np.concatenate([np.sort(rng.choice(m, k, replace=False)) for k in lens]).astype(np.int32)
    cv = rng.uniform(-1, 1, ri.size).astype(np.float32)
    rp, col, val = oracle.csr_to_csc(n, m, cp, ri, cv)  # the transpose's columns are A's rows
    return sa.Matrix(m, n, rp, col, val), (cp, ri, cv)


def check(M, csc, key, xv, run, want):
    dk, dv = sa.DeviceArray.from_host(key, np.int32), sa.DeviceArray.from_host(xv, np.float32)
    M.A.set_sparse_x(dk, dv, key.size)
    yk, yv = sa.DeviceArray(M.m, np.int32), sa.DeviceArray(M.m, np.float32)
    cnt, used = run(yk, yv)
    assert want is None or used == want
    ek, ev, eb = oracle.spmspv_f64(M.m, *csc, key, xv)
    np.testing.assert_array_equal(yk.to_host(cnt), ek)
    assert np.all(np.abs(yv.to_host(cnt).astype(np.float64) - ev) <= 1e-5 * eb + 1e-30)


@pytest.mark.parametrize("m", [16384, 300001])
@pytest.mark.parametrize("slot", [sa.K_COL_NAIVE_ATOMIC, sa.K_COL_LB_ATOMIC, sa.K_COL_NAIVE_SORT, None])
def test_sizes_around_the_limits(gpu, m, slot):
    # 4,096 columns of 3, 16 hub columns whose sums cross the gather's limit
    lens = np.concatenate([np.full(4096, 3), np.full(16, min(m, 100000)), [11264, 11265]])
    M, csc = matrix(m, lens, m)
    rng = np.random.default_rng(1)
    if slot is None:
        M.A.selector_mode(1)  # the rule tree chooses
    else:
        M.A.selector_mode(2, slot)
    h = 4096
    sets = [[h + 16], [h + 17], [h], np.arange(4096), np.r_[np.arange(1, 4096), h], [h + 17], [h + 16],
            np.arange(h, h + 5), np.arange(h, h + 6), np.arange(h, h + 16), np.r_[np.arange(4080), np.arange(h, h + 16)],
            np.arange(h, h + 5), np.arange(h, h + 6)]
    for s in sets:
        key = np.asarray(s, np.int32)
        xv = rng.uniform(-1, 1, key.size).astype(np.float32)
        # a call that fits reports the sort-based slot of the single launch
        small = int(lens[key].sum()) <= 11264
        want = None if slot is None or (small and slot != sa.K_COL_NAIVE_SORT) else slot
        check(M, csc, key, xv, lambda a, b: M.A.run_auto(y_key=a, y_val=b), want)
        if slot is not None:
            check(M, csc, key, xv, lambda a, b: (M.A.run(slot, y_key=a, y_val=b), slot), slot)
    # nothing is left behind for a dense result
    yd = sa.DeviceArray(m, np.float32)
    key, xv = np.arange(64, dtype=np.int32), np.ones(64, np.float32)
    dk, dv = sa.DeviceArray.from_host(key, np.int32), sa.DeviceArray.from_host(xv, np.float32)
    M.A.set_sparse_x(dk, dv, 64)
    M.A.run_auto(y_dense=yd)
    ek, ev, eb = oracle.spmspv_f64(m, *csc, key, xv)
    ref = np.zeros(m)
    ref[ek] = ev
    assert np.all(np.abs(yd.to_host() - ref) <= 1e-5 * np.abs(ref).max() + 1e-30)
