"""The SpMM kernels without a schedule at the edges of their workgroups: rows dealt to the XCDs in stretches, and
column-major products written by the kernel that forms the sums, and widths that are no whole vectors.  Parity against the CPU oracle within
8*u*(|alpha| * (|A||B|)_ij + |beta*C_ij|)."""
import numpy as np
import pytest

from mcsparse_amd import api
from mcsparse_amd import workloads as wl

from test_gpu_spmm import check

pytestmark = pytest.mark.gpu


# rows: one, a workgroup and its neighbours, the last stretch of a round full, begun and short of one row
@pytest.mark.parametrize("m", [1, 63, 65, 4096, 8191, 16385])
@pytest.mark.parametrize("n", [4, 16, 40])
def test_rows_in_stretches(torch_gpu, handle, oracle, m, n):
    a = wl.random_ragged(m, 907, 6, dtype=np.float32, seed=m + n)
    check(torch_gpu, handle, oracle, a, n, -1.5, 0.75)


# widths: one lane, the first and last width of every lane count of the columns kernel, the first one past it
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("m,n", [(1, 12), (63, 16), (64, 17), (65, 5), (4097, 9), (700, 4), (700, 8), (700, 31), (700, 32),
                                 (700, 33), (700, 64), (700, 65)])
def test_column_major_product(torch_gpu, handle, oracle, m, n, dtype):
    a = wl.random_ragged(m, 530, 9, dtype=dtype, seed=m + n).with_base(1)
    for b_order in (api.ORDER_COL, api.ORDER_ROW):
        check(torch_gpu, handle, oracle, a, n, 1.5, 0.0, b_order=b_order, c_order=api.ORDER_COL, pad_b=1, pad_c=3)
        check(torch_gpu, handle, oracle, a, n, 1.5, -0.5, b_order=b_order, c_order=api.ORDER_COL)


# widths that are no multiple of a 16-byte vector: the last lane's vector reaches back over columns of the lane before;
# rows of op(B) and C that begin at any element
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [1, 2, 3, 5, 6, 7, 9, 15, 17, 31, 33, 63, 67, 129, 261])
def test_ragged_widths(torch_gpu, handle, oracle, n, dtype):
    a = wl.random_ragged(611, 530, 9, dtype=dtype, seed=n)
    for pad_b, pad_c in ((0, 0), (3, 1), (1, 2)):
        check(torch_gpu, handle, oracle, a, n, 1.5, 0.0, pad_b=pad_b, pad_c=pad_c)
        check(torch_gpu, handle, oracle, a, n, 1.5, -0.5, pad_b=pad_b, pad_c=pad_c)
        check(torch_gpu, handle, oracle, a, n, 1.5, -0.5, op_b=api.OP_T, b_order=api.ORDER_COL, c_order=api.ORDER_COL,
              pad_b=pad_b, pad_c=pad_c)
