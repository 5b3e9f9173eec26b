"""The SpMM kernels without a schedule at the edges of their workgroups: rows dealt to the XCDs in
stretches.  Parity against the CPU oracle within
8*u*(|alpha| * (|A||B|)_ij + |beta*C_ij|)."""
import numpy as np
import pytest

from mcsparse_amd import workloads as wl

from test_gpu_spmm import check

pytestmark = pytest.mark.gpu


# rows: one, a workgroup and its neighbours, the last stretch of a round full, begun and short of one row
@pytest.mark.parametrize("m", [1, 63, 65, 4096, 8191, 16385])
@pytest.mark.parametrize("n", [4, 16, 40])
def test_rows_in_stretches(torch_gpu, handle, oracle, m, n):
    a = wl.random_ragged(m, 907, 6, dtype=np.float32, seed=m + n)
    check(torch_gpu, handle, oracle, a, n, -1.5, 0.75)
