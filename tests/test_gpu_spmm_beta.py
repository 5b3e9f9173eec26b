"""C = alpha * op(A) * op(B) + beta * C is rounded alike whichever kernel writes an element of C: alpha times the sum is rounded,
and beta * C is added to it in one fused operation.  So rows of one product, and products of one matrix along different ways
(row kernels, long rows in pieces, schedules, diagonals, transposes), agree to the bit where their sums do."""
import numpy as np
import pytest

from mcsparse_amd import api
from mcsparse_amd import workloads as wl

from test_gpu_spmm import run_spmm
from test_gpu_spmm_long_rows import rows_of_lengths

pytestmark = pytest.mark.gpu


def one_of_each_row(a, seed):
    """The same structure with a single 1 in a row, all else 0: every order of summation gives one element of op(B)."""
    val = np.zeros(a.nnz, a.val.dtype)
    lengths = a.row_lengths()
    rows = np.flatnonzero(lengths)
    val[a.ptr[rows] - a.base + np.random.default_rng(seed).integers(0, lengths[rows])] = 1
    return wl.Csr(a.m, a.n, a.ptr, a.col, val, base=a.base)


MATRICES = {
    "ragged": lambda dtype: wl.random_ragged(1201, 907, 14, dtype=dtype, seed=5),
    "stencil": lambda dtype: wl.stencil_27pt(24, dtype=dtype),
    "long rows": lambda dtype: rows_of_lengths([3, 1024, 1025, 0, 4097, 7, 0, 8193, 1, 20000, 5, 40] * 3, 30011, dtype, seed=6),
    "one line": lambda dtype: wl.laplacian_5pt(150, dtype=dtype),
}


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("matrix", MATRICES)
@pytest.mark.parametrize("b_order", [api.ORDER_ROW, api.ORDER_COL])
@pytest.mark.parametrize("c_order", [api.ORDER_ROW, api.ORDER_COL])
def test_every_kernel_rounds_alike(torch_gpu, handle, dtype, matrix, b_order, c_order):
    a = one_of_each_row(MATRICES[matrix](dtype), 7)
    exact = np.longdouble if dtype == np.float64 else np.float64
    # beta and C of half a significand: beta * C is exact, and so is its sum with alpha * b, once that is rounded, in the wider
    # type (2^-2 to 2^2 each), which is then rounded once
    half = 26 if dtype == np.float64 else 12
    rng = np.random.default_rng(8)
    alpha, beta = dtype(1.0) + dtype(rng.uniform(0.2, 0.8)), dtype(-1.375)
    for n in (1, 2, 3, 5, 8, 16, 24, 33, 64, 100):
        B = rng.uniform(1, 2, (a.n, n)).astype(dtype)
        C0 = np.round(rng.uniform(1, 2, (a.m, n)) * 2.0 ** (half - 5)).astype(dtype) * dtype(2.0 ** (5 - half))
        product = np.zeros((a.m, n), dtype)
        ones = np.flatnonzero(a.val)
        rows = np.repeat(np.arange(a.m), a.row_lengths())[ones]
        product[rows] = alpha * B[a.col[ones] - a.base]
        want = (product.astype(exact) + exact(beta) * C0.astype(exact)).astype(dtype)
        for preprocess in (False, True):
            st, got, _ = run_spmm(torch_gpu, handle, a, B, C0, alpha, beta, b_order=b_order, c_order=c_order, preprocess=preprocess)
            assert st == 0
            differ = got != want
            assert not differ.any(), (n, preprocess, int(differ.sum()), differ.size)
