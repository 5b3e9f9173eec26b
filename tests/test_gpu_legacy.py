"""GPU parity of the legacy typed entry points (csrmv, CsrmvEx, csrmm, csrmm2) against the CPU
oracle, through the C ABI.  Same tolerance as the generic path."""
import ctypes

import numpy as np
import pytest

from mcsparse_amd import api
from mcsparse_amd import workloads as wl

from gpu_util import assert_within, dev

pytestmark = pytest.mark.gpu


def mat_descr(lib, base):
    d = ctypes.c_void_p()
    assert lib.mcsparseCreateMatDescr(ctypes.byref(d)) == 0
    assert lib.mcsparseSetMatIndexBase(d, base) == 0
    return d


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("base", [0, 1])
@pytest.mark.parametrize("entry", ["csrmv", "csrmv_opT_is_ignored", "CsrmvEx"])
def test_csrmv(torch_gpu, handle, oracle, lib, dtype, base, entry):
    a = wl.power_law(m=6000, max_len=4000, dtype=dtype).with_base(base)
    rng = np.random.default_rng(1)
    x = rng.uniform(-1, 1, a.n).astype(dtype)
    y0 = rng.uniform(-1, 1, a.m).astype(dtype)
    alpha, beta = 1.5, -0.5
    ct = api.maca_type(dtype)
    sc = ctypes.c_float if dtype == np.float32 else ctypes.c_double
    pa, pb = sc(alpha), sc(beta)
    d = mat_descr(lib, base)
    d_ptr, d_col, d_val, d_x, d_y = (dev(torch_gpu, v) for v in (a.ptr, a.col, a.val, x, y0))
    if entry.startswith("csrmv"):
        fn = lib.mcsparseScsrmv if dtype == np.float32 else lib.mcsparseDcsrmv
        op = api.OP_T if entry.endswith("ignored") else api.OP_N  # the reference never reads transA
        st = fn(handle.ptr, op, a.m, a.n, a.nnz, ctypes.addressof(pa), d, d_val.data_ptr(), d_ptr.data_ptr(),
                d_col.data_ptr(), d_x.data_ptr(), ctypes.addressof(pb), d_y.data_ptr())
    else:
        size = ctypes.c_size_t()
        common = (api.OP_N, a.m, a.n, a.nnz, ctypes.addressof(pa), ct, d, d_val.data_ptr(), ct, d_ptr.data_ptr(),
                  d_col.data_ptr(), d_x.data_ptr(), ct, ctypes.addressof(pb), ct, d_y.data_ptr(), ct, ct)
        assert lib.mcsparseCsrmvEx_bufferSize(handle.ptr, 0, *common, ctypes.byref(size)) == 0
        buf = torch_gpu.empty(size.value, dtype=torch_gpu.uint8, device="cuda")
        st = lib.mcsparseCsrmvEx(handle.ptr, 0, *common, buf.data_ptr())
    torch_gpu.cuda.synchronize()
    assert st == 0
    y_ref, bound = oracle.spmv(False, a.m, a.n, base, a.ptr, a.col, a.val, alpha, beta, x, y0)
    assert_within(d_y.cpu().numpy(), y_ref, bound, dtype, what=entry)
    lib.mcsparseDestroyMatDescr(d)


def rows_of(lens, n, dtype, seed):
    rng = np.random.default_rng(seed)
    ptr = np.concatenate([[0], np.cumsum(lens)])
    return wl.Csr(len(lens), n, ptr.astype(np.int32), rng.integers(0, n, ptr[-1]).astype(np.int32),
                  rng.uniform(-1, 1, ptr[-1]).astype(dtype))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("mean,m,longest", [(5, 280_001, 3000), (7, 500_003, 5000), (12, 160_001, 3000)])
def test_csrmv_knows_nothing_of_its_rows(torch_gpu, handle, oracle, lib, dtype, mean, m, longest):
    """Many short rows with a few long ones among them, and the bits of its first rows by themselves: no row-length analysis
    is there to say that rows may share lanes, so it is a lane group to a row, however many rows there are."""
    rng = np.random.default_rng(mean)
    lens = rng.integers(mean - 2, mean + 2, m)
    lens[100::m // 20] = longest
    a = rows_of(lens, 50_021, dtype, 3)
    x = rng.uniform(-1, 1, a.n).astype(dtype)
    sc = ctypes.c_float if dtype == np.float32 else ctypes.c_double
    pa, pb = sc(1.25), sc(0.0)
    d = mat_descr(lib, 0)
    d_ptr, d_col, d_val, d_x = (dev(torch_gpu, v) for v in (a.ptr, a.col, a.val, x))
    fn = lib.mcsparseScsrmv if dtype == np.float32 else lib.mcsparseDcsrmv
    out = []
    for rows in (m, 100_000):
        d_y = dev(torch_gpu, np.full(rows, 7, dtype))
        assert fn(handle.ptr, api.OP_N, rows, a.n, int(a.ptr[rows]), ctypes.addressof(pa), d, d_val.data_ptr(), d_ptr.data_ptr(),
                  d_col.data_ptr(), d_x.data_ptr(), ctypes.addressof(pb), d_y.data_ptr()) == 0
        torch_gpu.cuda.synchronize()
        out.append(d_y.cpu().numpy())
    y_ref, bound = oracle.spmv(False, m, a.n, 0, a.ptr, a.col, a.val, 1.25, 0.0, x, np.zeros(m, dtype))
    assert_within(out[0], y_ref, bound, dtype, what="csrmv")
    assert np.array_equal(out[0][:100_000], out[1])
    lib.mcsparseDestroyMatDescr(d)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("trans_b", [api.OP_N, api.OP_T])
@pytest.mark.parametrize("n", [1, 8, 33])
def test_csrmm2(torch_gpu, handle, oracle, lib, dtype, trans_b, n):
    base = 1
    a = wl.random_ragged(900, 700, 11, dtype=dtype, seed=n).with_base(base)
    rng = np.random.default_rng(2)
    k = a.n
    B = rng.uniform(-1, 1, (k, n)).astype(dtype)       # op(B)
    C0 = rng.uniform(-1, 1, (a.m, n)).astype(dtype)
    alpha, beta = -2.0, 0.75
    pad = 3
    if trans_b == api.OP_N:   # B stored k x n column-major
        ldb = k + pad
        img = np.zeros((n, ldb), dtype)
        img[:, :k] = B.T
        b_row_image = False
    else:                     # B stored n x k column-major = op(B) row-major
        ldb = n + pad
        img = np.zeros((k, ldb), dtype)
        img[:, :n] = B
        b_row_image = True
    ldc = a.m + pad
    cimg = np.full((n, ldc), 99.0, dtype)
    cimg[:, :a.m] = C0.T
    sc = ctypes.c_float if dtype == np.float32 else ctypes.c_double
    pa, pb = sc(alpha), sc(beta)
    d = mat_descr(lib, base)
    d_ptr, d_col, d_val, d_B, d_C = (dev(torch_gpu, v) for v in (a.ptr, a.col, a.val, img, cimg))
    fn = lib.mcsparseScsrmm2 if dtype == np.float32 else lib.mcsparseDcsrmm2
    st = fn(handle.ptr, api.OP_N, trans_b, a.m, n, k, a.nnz, ctypes.addressof(pa), d, d_val.data_ptr(),
            d_ptr.data_ptr(), d_col.data_ptr(), d_B.data_ptr(), ldb, ctypes.addressof(pb), d_C.data_ptr(), ldc)
    torch_gpu.cuda.synchronize()
    assert st == 0
    out = d_C.cpu().numpy()
    assert (out[:, a.m:] == 99.0).all()
    c_ref, bound = oracle.spmm(a.m, n, base, a.ptr, a.col, a.val, alpha, beta, img.ravel(), ldb, b_row_image,
                               np.ascontiguousarray(C0).ravel(), n, True)
    assert_within(np.ascontiguousarray(out[:, :a.m].T), c_ref, bound, dtype, what="csrmm2")
    if trans_b == api.OP_N:   # csrmm is csrmm2 with transB = N
        d_C2 = dev(torch_gpu, cimg)
        fn1 = lib.mcsparseScsrmm if dtype == np.float32 else lib.mcsparseDcsrmm
        st = fn1(handle.ptr, api.OP_N, a.m, n, k, a.nnz, ctypes.addressof(pa), d, d_val.data_ptr(), d_ptr.data_ptr(),
                 d_col.data_ptr(), d_B.data_ptr(), ldb, ctypes.addressof(pb), d_C2.data_ptr(), ldc)
        torch_gpu.cuda.synchronize()
        assert st == 0 and np.array_equal(d_C2.cpu().numpy(), out)
    lib.mcsparseDestroyMatDescr(d)
