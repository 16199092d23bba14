"""Bucket slot at the edges of the accumulate kernel's rounds (4,096
products) and chunks (16,384), with odd and even bin counts (two bins share
a cursor word), in bins of many rows and in hub rows that are bins of their
own, against the FP64 oracle."""
import ctypes

import numpy as np
import pytest

import oracle
import spmspv_amd as sa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("per_bin", [32, 4096, 8192, 16384])
@pytest.mark.parametrize("extra", [-1, 0, 1])
@pytest.mark.parametrize("hubs", [0, 1, 2])
def test_round_and_chunk_edges(gpu, per_bin, extra, hubs):
    rng = np.random.default_rng(per_bin + 10 * extra + hubs)
    n = 40000
    lens = np.full(128, per_bin // 32)
    lens[-1] += extra
    lens = np.concatenate([np.full(hubs, per_bin + extra), lens, np.zeros(5, int)])
    m = lens.size
    col = np.concatenate([np.sort(rng.choice(n, k, replace=False)) for k in lens]).astype(np.int32)
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    val = rng.uniform(-1, 1, col.size).astype(np.float32)
    M = sa.Matrix(m, n, rp, col, val)
    cp, ri, cv = oracle.csr_to_csc(m, n, rp, col, val)
    key = np.arange(n, dtype=np.int32)
    xv = rng.uniform(-1, 1, n).astype(np.float32)
    dk, dv = sa.DeviceArray.from_host(key, np.int32), sa.DeviceArray.from_host(xv, np.float32)
    M.A.set_sparse_x(dk, dv, n)
    yk, yv = sa.DeviceArray(m, np.int32), sa.DeviceArray(m, np.float32)
    ek, ev, eb = oracle.spmspv_f64(m, cp, ri, cv, key, xv)
    for buckets in (2, 4, 8):  # the second and third call meet cleared cursors
        c = ctypes.c_int(-1)
        assert sa.lib().spmspv_csc_bucket(M.A.h, 1.0, ctypes.byref(c), yk.ptr, yv.ptr, buckets) == 0
        np.testing.assert_array_equal(yk.to_host(c.value), ek)
        assert np.all(np.abs(yv.to_host(c.value).astype(np.float64) - ev) <= 1e-5 * eb + 1e-30)
