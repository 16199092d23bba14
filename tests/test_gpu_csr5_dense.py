"""CSR5 products of a dense x: the plain product (values alone in the copy's
column order) followed and preceded by calls that need x's support, zeros of
either sign and special values in x, against the FP64 oracle."""
import numpy as np
import pytest

import oracle
import spmspv_amd as sa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", ["plain-first", "support-first"])
def test_plain_then_support(gpu, order):
    n = 1 << 12
    rp, col, val = sa.gen_rmat_csr(12, 16, seed=23)
    M = sa.Matrix(n, n, rp, col, val)
    cp, ri, cv = oracle.csr_to_csc(n, n, rp, col, val)
    A = M.A
    A.set_spmv_type(1)
    A.csr5_preprocess()
    rng = np.random.default_rng(2)
    dx, yd = sa.DeviceArray(n, np.float32), sa.DeviceArray(n, np.float32)
    yk, yv = sa.DeviceArray(n, np.int32), sa.DeviceArray(n, np.float32)
    for rep in range(3):
        x = rng.uniform(-1, 1, n).astype(np.float32)
        x[rng.random(n) < 0.4] = 0.0
        x[rng.random(n) < 0.1] = -0.0
        dx.upload(x)
        key = np.nonzero(x)[0].astype(np.int32)
        ek, ev, eb = oracle.spmspv_f64(n, cp, ri, cv, key, x[key])
        ref, bound = np.zeros(n), np.zeros(n)
        ref[ek], bound[ek] = ev, eb

        def plain():
            A.run(sa.K_SPMV_LB, y_dense=yd, want_nnz=False)
            assert np.all(np.abs(yd.to_host() - ref) <= 1e-5 * bound + 1e-30)

        def support(slot):
            cnt = A.run(slot, y_key=yk, y_val=yv)
            np.testing.assert_array_equal(yk.to_host(cnt), ek)
            assert np.all(np.abs(yv.to_host(cnt) - ev) <= 1e-5 * eb + 1e-30)

        A.set_vector_type(sa.SPMSPV_VEC_DENSE)
        A.set_x(dx)
        if order == "plain-first":
            plain()
            support(sa.K_ROW_LB)
            support(sa.K_SPMV_LB)
            plain()
        else:
            support(sa.K_SPMV_LB)
            plain()
            support(sa.K_ROW_LB)
        A.set_x(None)
        A.set_vector_type(sa.SPMSPV_VEC_SPARSE)
        dk, dv = sa.DeviceArray.from_host(key, np.int32), sa.DeviceArray.from_host(x[key], np.float32)
        A.set_sparse_x(dk, dv, key.size)
        support(sa.K_ROW_LB)
