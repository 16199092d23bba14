"""Batches whose workspace grows and is used again: few vectors, thousands of
them, vectors of several selector tiles and of sampled size, key arrays that
start past the first vector; every vector against the FP64 oracle and the
single-vector selector."""
import os

import numpy as np
import pytest

import oracle
import spmspv_amd as sa

pytestmark = pytest.mark.gpu
WEIGHTS = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "spmspv-adaptive_amd", "selector_weights.npy")


@pytest.fixture(scope="module")
def graph(gpu):
    scale = 17
    n = 1 << scale
    rp, col, val = sa.gen_rmat_csr(scale, 4, seed=71)
    M = sa.Matrix(n, n, rp, col, val)
    M.A.selector_set_weights(np.load(WEIGHTS).astype(np.float32))
    M.A.set_bucket_range(100_000, 400_000)
    return n, M, oracle.csr_to_csc(n, n, rp, col, val)


def run(graph, sizes, seed, skip=0):
    n, M, (cp, ri, cv) = graph
    rng = np.random.default_rng(seed)
    keys = [np.sort(rng.choice(n, k, replace=False)).astype(np.int32) for k in sizes]
    vals = [rng.uniform(-1, 1, k).astype(np.float32) for k in sizes]
    vptr = (skip + np.concatenate([[0], np.cumsum(sizes)])).astype(np.int32)
    need = [int(min(n, np.diff(cp)[k].sum())) for k in keys]
    yoff = np.concatenate([[0], np.cumsum(need)]).astype(np.int64)
    pad = [np.zeros(skip + 1, np.int32)]
    d = [sa.DeviceArray.from_host(vptr, np.int32),
         sa.DeviceArray.from_host(np.concatenate([pad[0][:skip]] + keys + [pad[0][:1]]), np.int32),
         sa.DeviceArray.from_host(np.concatenate([np.zeros(skip, np.float32)] + vals + [np.zeros(1, np.float32)]), np.float32),
         sa.DeviceArray.from_host(yoff, np.int64)]
    yk, yv, yn = sa.DeviceArray(yoff[-1], np.int32), sa.DeviceArray(yoff[-1], np.float32), sa.DeviceArray(len(sizes), np.int32)
    used = M.A.run_batched(*d, yk, yv, yn)
    cnt, hk, hv = yn.to_host(), yk.to_host(), yv.to_host()
    look = range(len(sizes)) if len(sizes) < 40 else rng.choice(len(sizes), 40, replace=False)
    for v in look:
        ek, ev, eb = oracle.spmspv_f64(n, cp, ri, cv, keys[v], vals[v])
        assert cnt[v] == ek.size, f"vector {v} slot {used[v]}"
        o = yoff[v]
        np.testing.assert_array_equal(hk[o:o + cnt[v]], ek)
        assert np.all(np.abs(hv[o:o + cnt[v]].astype(np.float64) - ev) <= 1e-5 * eb + 1e-30), f"vector {v} slot {used[v]}"
        if sizes[v]:
            dk, dv = sa.DeviceArray.from_host(keys[v], np.int32), sa.DeviceArray.from_host(vals[v], np.float32)
            M.A.set_sparse_x(dk, dv, int(sizes[v]))
            want = M.A.select()  # the network's choice, without the bucket rule
            if used[v] == sa.K_COL_BUCKET:
                assert want in (2, 3, 5, 7), f"vector {v}"
            else:
                assert want == used[v], f"vector {v}"
    return used


def test_batch_sizes(graph):
    n = graph[0]
    few = [0, 1, 2047, 2048, 2049, 4097, 20000, 65536, 65537, 100001, n]
    run(graph, few, 1)
    run(graph, [3] * 4500 + [2500, 0, 70000], 2)  # more vectors than are reserved
    run(graph, few[::-1], 3, skip=12345)
