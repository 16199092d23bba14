"""Batches of more keys than the reserved workspace scans at a time: groups of
vectors, vectors that are scanned alone, and no allocation after the buffers
are reserved; every vector against the FP64 oracle."""
import ctypes

import numpy as np
import pytest

import oracle
import spmspv_amd as sa

pytestmark = pytest.mark.gpu


def free_bytes():
    sa.synchronize()
    free, total = ctypes.c_size_t(0), ctypes.c_size_t(0)
    assert ctypes.CDLL("libamdhip64.so.7").hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("slot", [sa.K_COL_LB_ATOMIC, sa.K_COL_NAIVE_SORT, sa.K_COL_LB_SORT])
@pytest.mark.parametrize("scale,per,sizes", [
    # three groups, the second vector of a group and the last one at its end
    (18, 2, [250000] * 17 + [1, 0, 200000, 131072] + [250000] * 5),
    # vectors around the places of a group, between small ones
    (22, 1, [50, 2097150, 30000, 2097151, 2097152, 2500000, 60000, 0, 2000000, 97150]),
])
def test_groups(gpu, scale, per, sizes, slot):
    n = 1 << scale
    rp, col, val = sa.gen_rmat_csr(scale, per, seed=3)
    M = sa.Matrix(n, n, rp, col, val)
    csc = oracle.csr_to_csc(n, n, rp, col, val)
    M.A.selector_mode(2, slot)
    xs = [sa.gen_sparse_vector(n, k, 11 + i) for i, k in enumerate(sizes)]
    need = [int(min(n, np.diff(csc[0])[k].sum())) for k, _ in xs]
    vptr = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    yoff = np.concatenate([[0], np.cumsum(need)]).astype(np.int64)
    assert vptr[-1] > 1 << 21
    d = [sa.DeviceArray.from_host(vptr), sa.DeviceArray.from_host(np.concatenate([k for k, _ in xs]).astype(np.int32)),
         sa.DeviceArray.from_host(np.concatenate([v for _, v in xs]).astype(np.float32)), sa.DeviceArray.from_host(yoff)]
    yk, yv, yn = sa.DeviceArray(yoff[-1], np.int32), sa.DeviceArray(yoff[-1], np.float32), sa.DeviceArray(len(xs), np.int32)
    before = free_bytes()
    M.A.run_batched(*d, yk, yv, yn)
    # the scans of all the keys at once would take 8 bytes per key; the runtime
    # itself takes a few MiB for its copies and first launches
    assert before - free_bytes() < 4 * int(vptr[-1])
    cnt = yn.to_host()
    for v, (k, x) in enumerate(xs):
        ek, ev, eb = oracle.spmspv_f64(n, *csc, k, x)
        assert cnt[v] == ek.size, f"vector {v}"
        np.testing.assert_array_equal(yk.to_host_range(yoff[v], cnt[v]), ek, err_msg=f"vector {v}")
        err = np.abs(yv.to_host_range(yoff[v], cnt[v]).astype(np.float64) - ev)
        assert np.all(err <= 1e-5 * eb + 1e-30), f"vector {v}"
