"""The SpMM kernels without a schedule at the edges of their workgroups: rows dealt to the XCDs in stretches, and
column-major products written by the kernel that forms the sums.  Parity against the CPU oracle within
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
