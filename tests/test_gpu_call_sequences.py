"""Calls that follow one another on one handle without x being set again:
what one call leaves behind must not change the next one's result. Index sets
and counts exact, values within 1e-5 * sum|a_ij x_j| of the FP64 oracle."""
import numpy as np
import pytest

import oracle
import spmspv_amd as sa

pytestmark = pytest.mark.gpu
SCAN_SLOTS = [sa.K_COL_LB_ATOMIC, sa.K_COL_LB_SORT, sa.K_COL_BUCKET, sa.K_COL_TWO_LAYER_ATOMIC]


class Graph:
    """R-MAT on a handle, x of k keys, and the product's reference."""

    def __init__(self, scale, k, seed=5, per=8):
        self.n = n = 1 << scale
        rp, col, val = sa.gen_rmat_csr(scale, per, seed=seed)
        self.csr = rp, col, val
        self.M = sa.Matrix(n, n, rp, col, val)
        self.A = self.M.A
        self.csc = oracle.csr_to_csc(n, n, rp, col, val)
        self.yk, self.yv = sa.DeviceArray(n, np.int32), sa.DeviceArray(n, np.float32)
        self.set_x(k, seed)

    def set_x(self, k, seed):
        self.key, self.val = sa.gen_sparse_vector(self.n, k, seed)
        self.dk, self.dv = sa.DeviceArray.from_host(self.key, np.int32), sa.DeviceArray.from_host(self.val, np.float32)
        self.A.set_sparse_x(self.dk, self.dv, k)
        self.ref = oracle.spmspv_f64(self.n, *self.csc, self.key, self.val)

    def check(self, cnt, tag):
        ek, ev, eb = self.ref
        np.testing.assert_array_equal(self.yk.to_host(cnt), ek, err_msg=tag)
        assert np.all(np.abs(self.yv.to_host(cnt).astype(np.float64) - ev) <= 1e-5 * eb + 1e-30), tag

    def run(self, slot, tag):
        print(tag, "slot", slot, flush=True)
        self.check(self.A.run(slot, y_key=self.yk, y_val=self.yv), f"{tag}, slot {slot}")


@pytest.mark.parametrize("slot", SCAN_SLOTS)
@pytest.mark.parametrize("graphs", [0, 1])
def test_product_after_bfs(gpu, slot, graphs):
    """The column scan of x is made again after a BFS has scanned its
    frontiers into the same arrays."""
    g = Graph(15, 9000)
    lev = sa.DeviceArray(g.n, np.int32)
    g.run(slot, "before")
    for src in (0, 77):
        g.A.bfs(src, lev, policy=2, use_graphs=graphs)
        g.run(slot, f"after the BFS from {src}")
        assert g.A.computeBinlen() == int(np.diff(g.csc[0])[g.key].sum())


@pytest.mark.parametrize("slot", SCAN_SLOTS)
def test_product_after_sampled_selection(gpu, slot):
    """A selection from a sample of a large x (more than 65,536 keys, a row
    slot guessed from the call before) leaves no estimate in the place of the
    exact size that an earlier scan of the same x left."""
    g = Graph(17, 70000)
    g.A.selector_mode(2, sa.K_ROW_LB)
    g.check(g.A.run_auto(y_key=g.yk, y_val=g.yv)[0], "first, no guess yet")
    g.set_x(80000, 6)
    size = int(np.diff(g.csc[0])[g.key].sum())
    g.run(slot, "scans x")
    g.check(g.A.run_auto(y_key=g.yk, y_val=g.yv)[0], "selected from a sample")
    g.run(slot, "after the selection")
    g.check(g.A.run_auto(y_key=g.yk, y_val=g.yv)[0], "selected from a sample")
    assert g.A.computeBinlen() == size


@pytest.mark.parametrize("slot", SCAN_SLOTS)
def test_product_after_matrix_features(gpu, slot):
    """The matrix features, computed at their first use, need the array that
    holds the column scan of x."""
    g = Graph(13, 6000)
    A = sa.SpmspvHandle(g.n, g.n, g.csr[1].size)
    d = [sa.DeviceArray.from_host(a) for a in g.csr]
    A.InputCSR(g.csr[1].size, *d)
    A.ToCSC()
    A.set_sparse_x(g.dk, g.dv, g.key.size)
    g.A = A
    g.run(slot, "scans x")
    A.computeMatFeature()
    g.run(slot, "after the features")


class Captured:
    """A handle's calls on a stream of their own, captured into a graph."""

    def __init__(self, A):
        import ctypes
        self.ct, self.A = ctypes, A
        sa.lib()
        self.hip = ctypes.CDLL("libamdhip64.so.7")
        self.stream, self.graph, self.exec = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
        assert self.hip.hipStreamCreateWithFlags(ctypes.byref(self.stream), 1) == 0  # non-blocking
        assert sa.lib().spmspv_set_stream(A.h, self.stream) == 0

    def capture(self, call):
        c = self.ct
        assert self.hip.hipStreamBeginCapture(self.stream, 1) == 0  # thread-local
        call()
        assert self.hip.hipStreamEndCapture(self.stream, c.byref(self.graph)) == 0
        assert self.hip.hipGraphInstantiate(c.byref(self.exec), self.graph, None, None, c.c_size_t(0)) == 0

    def replay(self):
        assert self.hip.hipGraphLaunch(self.exec, self.stream) == 0
        assert self.hip.hipStreamSynchronize(self.stream) == 0
        out = np.empty(1, np.int32)
        p = self.ct.c_void_p(sa.lib().spmspv_ynnz_device(self.A.h))
        assert sa.lib().spmspv_memcpy_d2h(out.ctypes.data_as(self.ct.c_void_p), p, 4) == 0
        return int(out[0])

    def close(self):
        assert sa.lib().spmspv_set_stream(self.A.h, None) == 0
        if self.exec:
            self.hip.hipGraphExecDestroy(self.exec)
            self.hip.hipGraphDestroy(self.graph)
        self.hip.hipStreamDestroy(self.stream)


@pytest.mark.parametrize("known", [False, True])
@pytest.mark.parametrize("slot", [0, 1, 2, 3, sa.K_COL_BUCKET])
def test_captured_call_on_new_x(gpu, slot, known):
    """A call without a count, captured once and replayed on other contents of
    x's arrays, with eager calls between the replays: x that ends in the
    single launch (16 row ranges here) and, for the slots that try it, x of
    the same number of keys that does not (the heaviest columns)."""
    k = 600 if slot < 4 else 20000
    g = Graph(17, k)
    order = np.argsort(-np.diff(g.csc[0]), kind="stable")
    xs = [sa.gen_sparse_vector(g.n, k, 100 + i) for i in range(4)]
    heavy = np.sort(order[:k]).astype(np.int32)
    xs.insert(2, (heavy, np.random.default_rng(7).uniform(-1, 1, k).astype(np.float32)))
    if slot < 4:
        assert int(np.diff(g.csc[0])[heavy].sum()) > 11264 >= max(int(np.diff(g.csc[0])[x[0]].sum()) for x in xs if x[0] is not heavy)
    g.set_x(k, 100)
    g.run(slot, "eager")
    cap = Captured(g.A)
    g.A.set_sparse_x(g.dk, g.dv, k)
    if known and slot < 4:
        g.A.computeBinlen()
    cap.capture(lambda: g.A.run(slot, y_key=g.yk, y_val=g.yv, want_nnz=False))
    keep = g.dk, g.dv
    for rep in range(2):
        for i, (key, val) in enumerate(xs):
            keep[0].upload(key)
            keep[1].upload(val)
            sa.synchronize()
            g.ref = oracle.spmspv_f64(g.n, *g.csc, key, val)
            print(f"slot {slot} replay {rep} {i}", flush=True)
            g.check(cap.replay(), f"slot {slot} replay {rep} x {i}")
            if i % 2:
                g.set_x(k, 50 + i)
                g.run(slot, "eager between replays")
    cap.close()


@pytest.mark.parametrize("csr5", [0, 1])
@pytest.mark.parametrize("slot", [sa.K_COL_LB_ATOMIC, sa.K_ROW_LB, sa.K_SPMV_NAIVE, sa.K_SPMV_LB])
@pytest.mark.parametrize("x", ["sparse", "dense"])
def test_product_after_buffers_were_given_back(gpu, slot, csr5, x):
    """What the handle derived from x lies in its buffers: after they are
    given back and reserved again it is made again, x being the caller's."""
    g = Graph(13, 3000)
    g.A.set_spmv_type(csr5)
    if x == "dense":
        d = np.zeros(g.n, np.float32)
        d[g.key] = g.val
        dx = sa.DeviceArray.from_host(d)
        A = sa.SpmspvHandle(g.n, g.n, g.csr[1].size)  # no sparse arrays lent
        m = [sa.DeviceArray.from_host(a) for a in g.csr]
        A.InputCSR(g.csr[1].size, *m)
        A.ToCSC()
        A.set_spmv_type(csr5)
        A.set_vector_type(sa.SPMSPV_VEC_DENSE)
        A.set_x(dx)
        g.A = A
    for rep in range(3):
        g.run(slot, f"{x} x, buffers reserved {rep} times again")
        g.A.deallocPreBuffer()
        if rep:
            g.A.allocPreBuffer()


def test_product_after_outer_conversion(gpu):
    """An outer conversion of a vector longer than the result takes the
    handle's bit array of x as scratch: x's bits are made again."""
    import scipy.sparse as sp
    m, n = 500, 4000
    R = sp.random(m, n, density=0.01, format="csr", random_state=3, dtype=np.float32)
    R.sort_indices()
    M = sa.Matrix(m, n, R.indptr.astype(np.int32), R.indices.astype(np.int32), R.data)
    key, val = sa.gen_sparse_vector(n, 300, 9)
    d = np.zeros(n, np.float32)
    d[key] = val
    dx, yk, yv = sa.DeviceArray.from_host(d), sa.DeviceArray(n, np.int32), sa.DeviceArray(n, np.float32)
    ek, ev, eb = oracle.spmspv_f64(m, *oracle.csr_to_csc(m, n, M.h_row_ptr, M.h_col, M.h_val), key, val)
    M.A.set_vector_type(sa.SPMSPV_VEC_DENSE)
    M.A.set_x(dx)
    for rep in range(2):
        cnt = M.A.run(sa.K_ROW_NAIVE, y_key=yk, y_val=yv)
        np.testing.assert_array_equal(yk.to_host(cnt), ek, err_msg=f"call {rep}")
        assert np.all(np.abs(yv.to_host(cnt).astype(np.float64) - ev) <= 1e-5 * eb + 1e-30)
        assert M.A.dense2sparse_outer(n, dx, yk, yv) == key.size
        np.testing.assert_array_equal(yk.to_host(key.size), key)


@pytest.mark.parametrize("csr5", [0, 1])
@pytest.mark.parametrize("slot", [sa.K_ROW_LB, sa.K_SPMV_NAIVE, sa.K_SPMV_LB])
def test_lent_bit_array_is_filled(gpu, slot, csr5):
    """A bit array lent with set_bitvector holds a dense x's support after the
    products that fill it (the plain merge-path product reads none)."""
    g = Graph(12, 1500)
    A, n = g.A, g.n
    A.set_spmv_type(csr5)
    d = np.zeros(n, np.float32)
    d[g.key] = g.val
    d[g.val.size:g.val.size + 5] = -0.0
    dx, yd = sa.DeviceArray.from_host(d), sa.DeviceArray(n, np.float32)
    bits = sa.DeviceArray.from_host(np.full((n + 31) // 32, 0x5A5A5A5A, np.int32))
    A.set_bitvector(bits, bits.count)
    A.set_vector_type(sa.SPMSPV_VEC_DENSE)
    A.set_x(dx)
    if slot == sa.K_SPMV_LB and csr5:
        A.run(slot, y_dense=yd, want_nnz=False)
    else:
        A.run(slot, y_key=g.yk, y_val=g.yv)
    got = np.unpackbits(bits.to_host().view(np.uint8), bitorder="little")[:n]
    np.testing.assert_array_equal(got, (d != 0).astype(np.uint8))


@pytest.mark.parametrize("m", [256, 20011])
@pytest.mark.parametrize("slot", [0, 1, 2, 3])
def test_finite_rows_beside_special_ones(gpu, m, slot):
    """Rows without an Inf or NaN among their products have the same bits in
    every call, and the bits they have where the other rows' special entries
    are finite; the other rows are Inf or NaN as the sum in any order is."""
    import scipy.sparse as sp
    rng = np.random.default_rng(m)
    n, k, per = 4000, 650, 16
    rows = np.concatenate([rng.choice(min(m, 400), per, replace=False) for _ in range(n)]) * (m // min(m, 400))
    R = sp.csr_matrix((rng.uniform(-1, 1, n * per).astype(np.float32), (rows, np.repeat(np.arange(n), per))), shape=(m, n))
    R.sort_indices()
    M = sa.Matrix(m, n, R.indptr.astype(np.int32), R.indices.astype(np.int32), R.data)
    cp, ri, cv = oracle.csr_to_csc(m, n, M.h_row_ptr, M.h_col, M.h_val)
    key, val = sa.gen_sparse_vector(n, k, 3)
    odd = val.copy()
    odd[[5, 300]], odd[77], odd[400] = np.inf, -np.inf, np.nan
    yk, yv = sa.DeviceArray(m, np.int32), sa.DeviceArray(m, np.float32)
    dk = sa.DeviceArray.from_host(key, np.int32)

    def product(v):
        dv = sa.DeviceArray.from_host(v, np.float32)
        M.A.set_sparse_x(dk, dv, k)
        cnt = M.A.run(slot, y_key=yk, y_val=yv)
        return yk.to_host(cnt), yv.to_host(cnt)

    ek, plain = product(val)
    dense = np.zeros(n)
    dense[key] = odd
    with np.errstate(invalid="ignore"):
        want = np.zeros(m)
        for c in key:
            want[ri[cp[c]:cp[c + 1]]] += cv[cp[c]:cp[c + 1]].astype(np.float64) * dense[c]
    want = want[ek]
    finite = np.isfinite(want)
    assert 40 < finite.sum() < ek.size
    for rep in range(8):
        gk, got = product(odd)
        np.testing.assert_array_equal(gk, ek)
        np.testing.assert_array_equal(got[finite].view(np.uint32), plain[finite].view(np.uint32), err_msg=f"call {rep}")
        np.testing.assert_array_equal(got[~finite], want[~finite].astype(np.float32))


@pytest.mark.parametrize("policy", [2, 3, 5])
def test_bfs_after_queued_products(gpu, policy):
    """Products without a count are still running on the handle's (null) stream
    when a BFS starts on its own one: both use the handle's buffers."""
    g = Graph(18, 100000, per=16)
    lev = sa.DeviceArray(g.n, np.int32)
    ref, _ = oracle.bfs(g.n, g.csc[0], g.csc[1], 5)
    for slot in (sa.K_COL_LB_ATOMIC, sa.K_COL_BUCKET):
        cnt = g.A.run(slot, y_key=g.yk, y_val=g.yv)
        for rep in range(20):
            g.A.set_sparse_x(g.dk, g.dv, g.key.size)
            g.A.run(slot, y_key=g.yk, y_val=g.yv, want_nnz=False)
        g.A.bfs(5, lev, policy=policy)
        np.testing.assert_array_equal(lev.to_host(), ref)
        g.check(cnt, f"slot {slot} before the BFS")


@pytest.mark.parametrize("slot", [sa.K_COL_NAIVE_SORT, sa.K_COL_LB_SORT])
@pytest.mark.parametrize("out", ["count", "no count", "dense"])
def test_products_fall_below_the_guess(gpu, slot, out):
    """A sort slot queued behind the selector after a call of more than 24,576
    products leaves out the single-workgroup sort: an x of the same size class
    with at most 3,072 products (none among them) is sorted by a second run."""
    import ctypes
    import scipy.sparse as sp
    m, n, k = 30011, 40000, 9000
    rng = np.random.default_rng(slot)
    # 15,000 empty columns, 5,000 of one entry, 20,000 of thirty
    per = np.repeat([0, 1, 30], [15000, 5000, 20000])
    cols = np.repeat(np.arange(n), per)
    R = sp.csr_matrix((np.ones(cols.size, np.float32), (rng.integers(0, m, cols.size), cols)), shape=(m, n))
    R.sort_indices()
    R.data = rng.uniform(0.1, 1, R.nnz).astype(np.float32)
    M = sa.Matrix(m, n, R.indptr.astype(np.int32), R.indices.astype(np.int32), R.data)
    csc = oracle.csr_to_csc(m, n, M.h_row_ptr, M.h_col, M.h_val)
    yk, yv, yd = sa.DeviceArray(m, np.int32), sa.DeviceArray(m, np.float32), sa.DeviceArray(m, np.float32)
    M.A.selector_mode(2, slot)
    M.A.set_small_x_path(False)
    last = None
    for ones, thirties in [(0, k), (0, k), (0, 0), (0, k), (3000, 0), (3000, 0), (500, k - 500), (0, 0), (0, 0), (3071, 0), (0, k)]:
        key = np.sort(np.concatenate([rng.choice(15000, k - ones - thirties, replace=False),
                                      15000 + rng.choice(5000, ones, replace=False),
                                      20000 + rng.choice(20000, thirties, replace=False)])).astype(np.int32)
        val = rng.uniform(-1, 1, k).astype(np.float32)
        dk, dv = sa.DeviceArray.from_host(key, np.int32), sa.DeviceArray.from_host(val, np.float32)
        M.A.set_sparse_x(dk, dv, k)
        products = int(np.diff(csc[0])[key].sum())
        before = M.A.speculation_stats()[1]
        if out == "no count":
            used = ctypes.c_int(-1)
            assert sa.lib().spmspv_run_auto(M.A.h, 1.0, None, yk.ptr, yv.ptr, None, ctypes.byref(used)) == 0
            sa.synchronize()
            c = np.empty(1, np.int32)
            p = ctypes.c_void_p(sa.lib().spmspv_ynnz_device(M.A.h))
            assert sa.lib().spmspv_memcpy_d2h(c.ctypes.data_as(ctypes.c_void_p), p, 4) == 0
            cnt = int(c[0])
        else:
            cnt, _ = M.A.run_auto(y_dense=yd if out == "dense" else None, y_key=yk, y_val=yv)
        missed = M.A.speculation_stats()[1] - before
        if last is not None and last > 8 * 3072 and products <= 3072:
            assert missed == 1, (last, products)
        ek, ev, eb = oracle.spmspv_f64(m, *csc, key, val)
        assert cnt == ek.size
        np.testing.assert_array_equal(yk.to_host(cnt), ek)
        assert np.all(np.abs(yv.to_host(cnt).astype(np.float64) - ev) <= 1e-5 * eb + 1e-30)
        if out == "dense":
            ref, bound = np.zeros(m), np.zeros(m)
            ref[ek], bound[ek] = ev, eb
            assert np.all(np.abs(yd.to_host() - ref) <= 1e-5 * bound + 1e-30)
        last = products


def test_lent_sparse_arrays_keep_their_size(gpu):
    """A dense x that a column slot turns into a sparse one is written into
    the caller's arrays where it fits the entries that were lent, else into the
    handle's own; arrays lent to a batch are never written."""
    n = 1 << 12
    rp, col, val = sa.gen_rmat_csr(12, 8, seed=2)
    M = sa.Matrix(n, n, rp, col, val)
    csc = oracle.csr_to_csc(n, n, rp, col, val)
    yk, yv = sa.DeviceArray(n, np.int32), sa.DeviceArray(n, np.float32)
    # room for all of x, of which ten entries are lent
    key, xv = np.full(n, -7, np.int32), np.full(n, 9.0, np.float32)
    key[:10], xv[:10] = np.arange(10) * 300, 1.0
    dk, dv = sa.DeviceArray.from_host(key), sa.DeviceArray.from_host(xv)

    def product(x, tag):
        dx = sa.DeviceArray.from_host(x)
        M.A.set_vector_type(sa.SPMSPV_VEC_DENSE)
        M.A.set_x(dx)
        cnt = M.A.run(sa.K_COL_LB_ATOMIC, y_key=yk, y_val=yv)
        nz = np.nonzero(x)[0].astype(np.int32)
        ek, ev, eb = oracle.spmspv_f64(n, *csc, nz, x[nz])
        np.testing.assert_array_equal(yk.to_host(cnt), ek, err_msg=tag)
        assert np.all(np.abs(yv.to_host(cnt).astype(np.float64) - ev) <= 1e-5 * eb + 1e-30), tag
        return nz

    rng = np.random.default_rng(1)
    large, small = np.zeros(n, np.float32), np.zeros(n, np.float32)
    large[rng.choice(n, 2000, replace=False)] = rng.uniform(0.5, 1, 2000)
    small[rng.choice(n, 10, replace=False)] = rng.uniform(0.5, 1, 10)
    M.A.set_sparse_x(dk, dv, 10)
    product(large, "past the lent entries")
    np.testing.assert_array_equal(dk.to_host(), key)
    np.testing.assert_array_equal(dv.to_host(), xv)
    M.A.set_sparse_x(dk, dv, 10)
    nz = product(small, "as many as were lent")
    np.testing.assert_array_equal(dk.to_host(10), nz)
    np.testing.assert_array_equal(dv.to_host(10), small[nz])
    np.testing.assert_array_equal(dk.to_host()[10:], key[10:])
    # a batch whose last vector has ten entries
    dk.upload(key)
    dv.upload(xv)
    vptr, yoff = sa.DeviceArray.from_host(np.array([0, 10], np.int32)), sa.DeviceArray.from_host(np.array([0, n], np.int64))
    M.A.run_batched(vptr, dk, dv, yoff, yk, yv, sa.DeviceArray(1, np.int32))
    for x, tag in ((small, "after a batch"), (large, "after a batch, large")):
        product(x, tag)
        np.testing.assert_array_equal(dk.to_host(), key)
        np.testing.assert_array_equal(dv.to_host(), xv)
    rank = sa.DeviceArray(n, np.float32)
    M.A.pagerank(rank)
    product(large, "after PageRank")
