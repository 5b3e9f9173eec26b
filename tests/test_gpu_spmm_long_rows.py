"""mcsparseSpMM on matrices with rows far longer than the rest: rows above 256 to 1024 nonzeros (four times the mean)
are cut into pieces of 4096 that a workgroup each takes (one piece: the row of C written directly; several: partial sums added in the order
of the pieces).  Parity against the CPU oracle within 8*u*(|alpha| * (|A||B|)_ij + |beta*C_ij|), bits that repeat
from run to run, and the time of a call."""
import numpy as np
import pytest

from mcsparse_amd import api
from mcsparse_amd import workloads as wl

from gpu_util import assert_within, dev
from test_gpu_spmm import check, run_spmm

pytestmark = pytest.mark.gpu


def rows_of_lengths(lengths, n_cols, dtype, seed, base=0):
    """CSR matrix whose row i holds lengths[i] nonzeros in distinct, sorted, random columns."""
    rng = np.random.default_rng(seed)
    ptr = np.zeros(len(lengths) + 1, np.int64)
    ptr[1:] = np.cumsum(lengths)
    col = np.empty(ptr[-1], np.int32)
    for i, length in enumerate(lengths):
        col[ptr[i]:ptr[i + 1]] = np.sort(rng.choice(n_cols, size=length, replace=False))
    val = rng.uniform(-1, 1, ptr[-1]).astype(dtype)
    return wl.Csr(len(lengths), n_cols, ptr.astype(np.int32) + base, col + base, val, base=base)


# lengths around the two limits (1024: taken apart from the row kernels; 4096: one piece), empty rows between long ones
LENGTHS = [3, 1024, 1025, 0, 4095, 4096, 4097, 7, 0, 8192, 8193, 12289, 1, 2000, 0, 20000, 5, 1500, 16, 0]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [1, 3, 8, 16, 33, 64, 100, 260])
def test_rows_around_the_limits(torch_gpu, handle, oracle, n, dtype):
    a = rows_of_lengths(LENGTHS * 3, 30011, dtype, seed=n)
    check(torch_gpu, handle, oracle, a, n, 1.0, 0.0)
    check(torch_gpu, handle, oracle, a, n, -1.5, 0.75, seed=1)


@pytest.mark.parametrize("op_b", [api.OP_N, api.OP_T])
@pytest.mark.parametrize("b_order", [api.ORDER_ROW, api.ORDER_COL])
@pytest.mark.parametrize("c_order", [api.ORDER_ROW, api.ORDER_COL])
def test_layouts_and_padding(torch_gpu, handle, oracle, op_b, b_order, c_order):
    a = rows_of_lengths(LENGTHS, 25013, np.float32, seed=4, base=1)
    check(torch_gpu, handle, oracle, a, 24, 0.5, -2.0, op_b=op_b, b_order=b_order, c_order=c_order, pad_b=3, pad_c=5)
    check(torch_gpu, handle, oracle, a, 7, 0.5, 0.0, op_b=op_b, b_order=b_order, c_order=c_order, pad_b=1, pad_c=2)


def test_long_rows_among_many_short_ones(torch_gpu, handle, oracle):
    """The matrix of the mixed SpMV workload, smaller: 20,000 rows of 16 and 8 rows of 30,000."""
    a = wl.mixed_rows(m=20000, per_row=16, long_rows=8, long_len=30000, dtype=np.float32)
    for n in (8, 16, 64, 128):
        check(torch_gpu, handle, oracle, a, n, 1.25, 0.5, seed=n)


def test_preprocess_leaves_such_a_matrix_to_the_row_kernels(torch_gpu, handle, oracle):
    a = wl.mixed_rows(m=20000, per_row=16, long_rows=8, long_len=30000, dtype=np.float32)
    check(torch_gpu, handle, oracle, a, 64, 1.0, 0.0, preprocess=True, expect_schedule=1)
    check(torch_gpu, handle, oracle, a, 16, 1.0, 0.5, preprocess=True, expect_schedule=1)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_bits_repeat_from_run_to_run(torch_gpu, handle, dtype):
    a = rows_of_lengths(LENGTHS * 2, 30011, dtype, seed=9)
    rng = np.random.default_rng(3)
    B = rng.uniform(-1, 1, (a.n, 40)).astype(dtype)
    C0 = rng.uniform(-1, 1, (a.m, 40)).astype(dtype)
    first = None
    for _ in range(3):
        st, got, _ = run_spmm(torch_gpu, handle, a, B, C0, 1.5, 0.25)
        assert st == 0
        if first is None:
            first = got.copy()
        assert np.array_equal(first, got)


@pytest.mark.parametrize("fmt", ["coo", "csc"])
def test_coo_and_csc_inputs(torch_gpu, handle, oracle, fmt):
    torch = torch_gpu
    a = rows_of_lengths(LENGTHS, 20011, np.float64, seed=11)
    n = 12
    rng = np.random.default_rng(12)
    B = rng.uniform(-1, 1, (a.n, n))
    C0 = rng.uniform(-1, 1, (a.m, n))
    d_B, d_C = dev(torch, B), dev(torch, C0)
    if fmt == "coo":
        rows = np.repeat(np.arange(a.m, dtype=np.int32), np.diff(a.ptr))
        keep = [dev(torch, rows), dev(torch, a.col), dev(torch, a.val)]
        mat = api.SpMat(a.m, a.n, a.nnz, keep[0], keep[1], keep[2], fmt=api.FORMAT_COO)
    else:
        t_ptr, t_row, t_val = oracle.csr2csc(a.m, a.n, 0, a.ptr, a.col, a.val, method="counting")
        keep = [dev(torch, t_ptr.astype(np.int32)), dev(torch, t_row.astype(np.int32)), dev(torch, t_val)]
        mat = api.SpMat(a.m, a.n, a.nnz, keep[0], keep[1], keep[2], fmt=api.FORMAT_CSC)  # offsets, then indices
    mB, mC = api.DnMat(a.n, n, n, d_B), api.DnMat(a.m, n, n, d_C)
    st, size = api.spmm_buffer_size(handle, api.OP_N, api.OP_N, 2.0, mat, mB, -1.0, mC, api.R_64F)
    assert st == 0
    buf = torch.empty(size, dtype=torch.uint8, device="cuda")
    assert api.spmm(handle, api.OP_N, api.OP_N, 2.0, mat, mB, -1.0, mC, api.R_64F, buf) == 0
    torch.cuda.synchronize()
    c_ref, bound = oracle.spmm(a.m, n, 0, a.ptr, a.col, a.val, 2.0, -1.0, B.ravel(), n, True, C0.ravel(), n, True)
    assert_within(d_C.cpu().numpy(), c_ref, bound, np.float64, what="spmm long rows, %s input" % fmt)


def test_a_row_of_fifty_thousand_does_not_hold_the_call_up(torch_gpu, handle):
    """1 M power-law rows, the longest of 50,000 nonzeros, N = 16: 7.3 ms when that row was one lane group's work;
    the operands are 0.35 GB, so anything near a millisecond says the row is being walked alone again."""
    torch = torch_gpu
    a = wl.power_law(m=1 << 20, max_len=50000, dtype=np.float32)
    n = 16
    d = [dev(torch, v) for v in (a.ptr, a.col, a.val)]
    B = torch.rand((a.n, n), dtype=torch.float32, device="cuda")
    C = torch.zeros((a.m, n), dtype=torch.float32, device="cuda")
    mat = api.SpMat(a.m, a.n, a.nnz, d[0], d[1], d[2], base=a.base)
    mB, mC = api.DnMat(a.n, n, n, B), api.DnMat(a.m, n, n, C)
    st, size = api.spmm_buffer_size(handle, api.OP_N, api.OP_N, 1.0, mat, mB, 0.0, mC, api.R_32F)
    buf = torch.empty(size, dtype=torch.uint8, device="cuda")
    for _ in range(3):
        assert api.spmm(handle, api.OP_N, api.OP_N, 1.0, mat, mB, 0.0, mC, api.R_32F, buf) == 0
    torch.cuda.synchronize()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record()
    for _ in range(10):
        api.spmm(handle, api.OP_N, api.OP_N, 1.0, mat, mB, 0.0, mC, api.R_32F, buf)
    e1.record()
    torch.cuda.synchronize()
    ms = e0.elapsed_time(e1) / 10
    assert ms < 2.0, ms


# rows around the cut of a matrix that has longer ones (256, or four times the mean), widths of every lane count
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [2, 4, 9, 13, 17, 31, 50, 67, 130])
@pytest.mark.parametrize("short", [2, 100])
def test_rows_around_the_cut(torch_gpu, handle, oracle, n, dtype, short):
    cut = 256
    for _ in range(8):  # the cut is four times the mean row length, and its rows are part of the mean
        lengths = ([short] * 97 + [255, 256, 257, cut - 1, cut, cut + 1, 0, 1100]) * 2
        cut = max(256, 4 * (sum(lengths) // len(lengths) + 1))
    assert cut + 1 in lengths and cut < 1024
    a = rows_of_lengths(lengths, 5003, dtype, seed=n)
    check(torch_gpu, handle, oracle, a, n, 1.25, 0.0, pad_b=1)
    check(torch_gpu, handle, oracle, a, n, 1.25, -0.5, seed=1, c_order=api.ORDER_COL)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("c_order", [api.ORDER_ROW, api.ORDER_COL])
@pytest.mark.parametrize("n", [3, 8, 24, 40])
@pytest.mark.parametrize("longest", [700, 1024, 1025, 5000])
def test_every_way_to_a_product_gives_the_same_bits(torch_gpu, oracle, dtype, c_order, n, longest):
    """Rows between the cut (256 here) and 1024 are taken apart where there is a longer one, whether the call knows that
    from its analysis or finds out on the device: a capture that meets the matrix first, COO and CSC inputs, a plan that
    was set by the caller."""
    torch = torch_gpu
    side = torch.cuda.Stream()
    handle = api.Handle(stream=side.cuda_stream)
    a = rows_of_lengths([4] * 200 + [255, 256, 257, 600, 0, longest, 300] * 2, 7001, dtype, seed=n)
    rng = np.random.default_rng(5)
    B = dev(torch, rng.uniform(-1, 1, (a.n, n)).astype(dtype))
    start = dev(torch, rng.uniform(-1, 1, (a.m, n) if c_order == api.ORDER_ROW else (n, a.m)).astype(dtype))
    ct = api.maca_type(np.dtype(dtype))
    ptr, col, val = dev(torch, a.ptr), dev(torch, a.col), dev(torch, a.val)
    rows = dev(torch, np.repeat(np.arange(a.m, dtype=np.int32), np.diff(a.ptr)))
    t_ptr, t_row, t_val = oracle.csr2csc(a.m, a.n, 0, a.ptr, a.col, a.val, method="counting")
    t_ptr, t_row, t_val = dev(torch, t_ptr.astype(np.int32)), dev(torch, t_row.astype(np.int32)), dev(torch, t_val)
    torch.cuda.synchronize()

    def product(kind):
        if kind == "coo":
            mat = api.SpMat(a.m, a.n, a.nnz, rows, col, val, fmt=api.FORMAT_COO)
        elif kind == "csc":
            mat = api.SpMat(a.m, a.n, a.nnz, t_ptr, t_row, t_val, fmt=api.FORMAT_CSC)
        else:
            mat = api.SpMat(a.m, a.n, a.nnz, ptr, col, val)
        if kind == "forced":
            mat.set_plan(api.FAMILY_VECTOR)
        C = start.clone()
        mB, mC = api.DnMat(a.n, n, n, B), api.DnMat(a.m, n, n if c_order == api.ORDER_ROW else a.m, C, order=c_order)
        call = (handle, api.OP_N, api.OP_N, 1.25, mat, mB, -0.5, mC, ct)
        st, size = api.spmm_buffer_size(*call)
        assert st == 0
        buf = torch.empty(size, dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        if kind == "captured":
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=side):
                assert api.spmm(*call, buf) == 0
            for _ in range(3):
                C.copy_(start)
                torch.cuda.synchronize()
                graph.replay()
                torch.cuda.synchronize()
        else:
            assert api.spmm(*call, buf) == 0
            torch.cuda.synchronize()
        return C.cpu().numpy()

    want = product("csr")
    for kind in ("captured", "coo", "csc", "forced"):
        assert np.array_equal(product(kind), want), kind
    handle.destroy()


def banded_matrix(dtype, k=300000, base=0, seed=31):
    """20,000 short rows and 1,200 of 257 to 9,000 nonzeros, over a k large enough that the long ones are taken in bands of
    op(B) (16 MB from 54 bytes a row on)."""
    rng = np.random.default_rng(seed)
    lengths = np.concatenate([rng.integers(0, 8, 20000), rng.integers(257, 2200, 1150), rng.integers(4000, 9001, 50)])
    rng.shuffle(lengths)
    ptr = np.concatenate([[0], np.cumsum(lengths)])
    rows = np.repeat(np.arange(lengths.size), lengths)
    col = np.sort(rng.integers(0, k, rows.size) + rows * k) - rows * k  # ascending, now and then a column twice
    return wl.Csr(lengths.size, k, ptr, col, rng.uniform(-1, 1, rows.size).astype(dtype), 0).with_base(base)


@pytest.mark.parametrize("dtype,n,base", [(np.float32, 14, 0), (np.float32, 16, 1), (np.float32, 29, 0), (np.float32, 32, 0),
                                          (np.float64, 7, 1), (np.float64, 16, 0)])
def test_long_rows_in_bands_of_the_operand(torch_gpu, handle, oracle, dtype, n, base):
    a = banded_matrix(dtype, base=base)
    assert a.nnz >= 1 << 20 and a.n * n * a.val.itemsize >= 16 << 20
    check(torch_gpu, handle, oracle, a, n, 1.25, 0.0, pad_b=n % 3)
    check(torch_gpu, handle, oracle, a, n, 1.25, -0.5, seed=1, c_order=api.ORDER_COL)


@pytest.mark.parametrize("how", ["one row descends", "all columns in one band", "long rows name the ends of op(B)"])
def test_long_rows_whose_bands_are_unlike(torch_gpu, handle, oracle, how):
    a = banded_matrix(np.float32)
    long_rows = np.nonzero(a.row_lengths() > 256)[0]
    for r in long_rows[:1] if how == "one row descends" else long_rows:
        span = slice(a.ptr[r], a.ptr[r + 1])
        if how == "one row descends":
            a.col[span] = a.col[span][::-1]
        elif how == "all columns in one band":
            a.col[span] = 150000 + np.arange(span.stop - span.start) % 1000
            a.col[span].sort()
        else:
            a.col[span] = np.where(np.arange(span.stop - span.start) < 100, 0, a.n - 1)
    check(torch_gpu, handle, oracle, a, 32, -1.5, 0.5)


def test_long_rows_in_more_than_64_bands(torch_gpu, handle, oracle):
    a = banded_matrix(np.float32, k=4300000)
    check(torch_gpu, handle, oracle, a, 16, 1.25, -0.5)  # op(B): 275 MB, bands of 4 MB


def test_every_way_to_bands_gives_the_same_bits(torch_gpu, oracle):
    torch = torch_gpu
    side = torch.cuda.Stream()
    handle = api.Handle(stream=side.cuda_stream)
    a, n = banded_matrix(np.float32), 24
    rng = np.random.default_rng(5)
    B = dev(torch, rng.uniform(-1, 1, (a.n, n)).astype(np.float32))
    ptr, col, val = dev(torch, a.ptr), dev(torch, a.col), dev(torch, a.val)
    rows = dev(torch, np.repeat(np.arange(a.m, dtype=np.int32), a.row_lengths()))
    t_ptr, t_row, t_val = oracle.csr2csc(a.m, a.n, 0, a.ptr, a.col, a.val, method="counting")
    t_ptr, t_row, t_val = dev(torch, t_ptr.astype(np.int32)), dev(torch, t_row.astype(np.int32)), dev(torch, t_val)
    results = {}
    for kind in ("csr", "captured", "coo", "csc", "csr again"):
        if kind == "coo":
            mat = api.SpMat(a.m, a.n, a.nnz, rows, col, val, fmt=api.FORMAT_COO)
        elif kind == "csc":
            mat = api.SpMat(a.m, a.n, a.nnz, t_ptr, t_row, t_val, fmt=api.FORMAT_CSC)
        else:
            mat = api.SpMat(a.m, a.n, a.nnz, ptr, col, val)
        C = torch.full((a.m, n), 3.0, device="cuda")
        call = (handle, api.OP_N, api.OP_N, 1.25, mat, api.DnMat(a.n, n, n, B), 0.0, api.DnMat(a.m, n, n, C), api.R_32F)
        st, size = api.spmm_buffer_size(*call)
        assert st == 0
        buf = torch.full((size,), 0xFF, dtype=torch.uint8, device="cuda")  # (NaN wherever sums are read that were not written)
        torch.cuda.synchronize()
        if kind == "captured":
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=side):
                assert api.spmm(*call, buf) == 0
            for _ in range(3):
                C.fill_(9.0)
                torch.cuda.synchronize()
                graph.replay()
                torch.cuda.synchronize()
        else:
            assert api.spmm(*call, buf) == 0
            torch.cuda.synchronize()
        results[kind] = C.cpu().numpy()
    for kind, got in results.items():
        assert np.array_equal(got, results["csr"]), kind
    handle.destroy()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [5, 12, 16, 19, 32, 37, 64])  # four, eight and sixteen lanes to a row, whole vectors and ragged
@pytest.mark.parametrize("m", [64, 65, 200, 449])
def test_short_rows_are_taken_in_turns(torch_gpu, handle, oracle, n, dtype, m):
    """A wavefront's 64 rows where all are long, none, the last ones missing; lengths around what a group asks for at a time
    and around what it counts as long among them, empty rows, and one that keeps a group while the others take the rest."""
    edge = [0, 1, 2, 3, 4, 5, 7, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 65, 128, 255, 256]
    rng = np.random.default_rng(m + n)
    lengths = list(rng.choice(edge, m))
    lengths[0] = 256
    if m > 200:
        lengths[128:192] = [1100] * 64  # a wavefront without rows of its own
        lengths[192:256] = [1] * 64     # more rows than groups, all of one turn
    a = rows_of_lengths(lengths + [1100], 1501, dtype, seed=n, base=1)
    check(torch_gpu, handle, oracle, a, n, 1.25, 0.0, pad_b=2)
    check(torch_gpu, handle, oracle, a, n, 0.5, -1.5, seed=1, c_order=api.ORDER_COL)


@pytest.mark.parametrize("dtype,n", [(np.float32, 7), (np.float32, 16), (np.float32, 30), (np.float64, 4), (np.float64, 7), (np.float64, 16)])
def test_pieces_cut_beside_the_row_kernel(torch_gpu, handle, oracle, dtype, n):
    """op(B) beyond the L2s: rows of one piece, of as many as a workgroup has wavefronts, of one more and of many."""
    lengths = [3] * 3000
    for at, length in zip(range(5, 3000, 30), [300, 4096, 4097, 8193, 16384, 16385, 20481, 90001] * 8):
        lengths[at] = length
    a = rows_of_lengths(lengths, 400009, dtype, seed=2)
    assert a.nnz >= 1 << 20 and a.n * n * np.dtype(dtype).itemsize >= 10 << 20
    check(torch_gpu, handle, oracle, a, n, 1.25, -0.5)


def rows_about_a_limit(arrangement, lanes):
    """Row lengths about the one above which a row is taken by part of a wavefront: 16 times the lanes to a row, or six times the
    mean.  And that limit."""
    about = 16 * lanes
    for _ in range(8):  # its rows are part of the mean
        edge = [about - 1, about, about + 1, 63, 64, 65, 127, 128, 129, 191, 255, 256]
        if arrangement == "few":  # one, two and up to seven neighbours, so that parts of a wavefront are left without a row
            lengths = [1] * 70 + edge + [0, 2] * 40 + edge * 8 + [3] * 5 + [1025, 129]
            for count in range(1, 8):
                lengths += [1] * 300 + [200] * count
        elif arrangement == "sorted":
            lengths = [1025, 600] + sorted(edge * 20 + [3] * 4500, reverse=True)
        elif arrangement == "many":  # more rows than the wavefronts look at in one turn
            lengths = edge * 50 + [2] * 280000 + [900, 129] + [1] * 9
        else:  # most rows are above 16 times the lanes
            lengths = [25] * 1500 + edge * 4 + [1500] + [30] * 3
        limit = max(16 * lanes, 6 * (sum(lengths) // len(lengths) + 1))
        if arrangement != "alike" or about == limit:
            break
        about = limit
    assert limit < 256 and limit + 1 in lengths
    return lengths, limit


@pytest.mark.parametrize("dtype,n,lanes", [(np.float32, 9, 4), (np.float32, 16, 4), (np.float64, 8, 4), (np.float64, 9, 8),
                                           (np.float64, 15, 8), (np.float64, 16, 8)])
@pytest.mark.parametrize("arrangement", ["few", "sorted", "many", "alike"])
def test_rows_taken_by_part_of_a_wavefront(torch_gpu, handle, oracle, dtype, n, lanes, arrangement):
    """By a call that knows of the long row and by one that does not (COO), to the same bits; every row on its own tells rows left
    out, and rows taken twice with beta, from right ones."""
    lengths, limit = rows_about_a_limit(arrangement, lanes)
    assert (limit > 16 * lanes) == (arrangement == "alike")
    rng = np.random.default_rng(n)
    ptr = np.concatenate([[0], np.cumsum(lengths)])
    rows = np.repeat(np.arange(len(lengths)), lengths)
    col = np.sort(rng.integers(0, 3001, rows.size) + rows * 3001) - rows * 3001  # ascending, now and then a column twice
    a = wl.Csr(len(lengths), 3001, ptr, col, rng.uniform(-1, 1, rows.size).astype(dtype), 0).with_base(0)
    check(torch_gpu, handle, oracle, a, n, 1.25, 0.0, pad_b=1)
    check(torch_gpu, handle, oracle, a, n, 0.5, -1.5, seed=1, c_order=api.ORDER_COL)
    torch = torch_gpu
    B = dev(torch, np.random.default_rng(2).uniform(-1, 1, (a.n, n)).astype(dtype))
    ptr, col, val = dev(torch, a.ptr), dev(torch, a.col), dev(torch, a.val)
    rows = dev(torch, np.repeat(np.arange(a.m, dtype=np.int32), np.diff(a.ptr)))
    products = []
    for mat in (api.SpMat(a.m, a.n, a.nnz, ptr, col, val), api.SpMat(a.m, a.n, a.nnz, rows, col, val, fmt=api.FORMAT_COO)):
        C = torch.ones((a.m, n), dtype=B.dtype, device="cuda")
        call = (handle, api.OP_N, api.OP_N, 1.0, mat, api.DnMat(a.n, n, n, B), 0.5, api.DnMat(a.m, n, n, C), api.maca_type(np.dtype(dtype)))
        st, size = api.spmm_buffer_size(*call)
        assert st == 0
        assert api.spmm(*call, torch.empty(size, dtype=torch.uint8, device="cuda")) == 0
        torch.cuda.synchronize()
        products.append(C.cpu().numpy())
    assert np.array_equal(products[0], products[1])


def sorted_power_law(dtype, m=100000):
    """Power-law rows, the longest first."""
    a = wl.power_law(m=m, max_len=1500, dtype=dtype)
    lengths = np.sort(np.diff(a.ptr))[::-1]
    rng = np.random.default_rng(8)
    rows = np.repeat(np.arange(m), lengths)
    col = np.sort(rng.integers(0, m, rows.size) + rows * m) - rows * m
    return wl.Csr(m, m, np.concatenate([[0], np.cumsum(lengths)]), col, rng.uniform(-1, 1, rows.size).astype(dtype), 0).with_base(0)


@pytest.mark.parametrize("dtype,n", [(np.float32, 16), (np.float64, 8)])
def test_long_rows_that_lie_together(torch_gpu, dtype, n):
    """A matrix whose rows are sorted by their length takes no longer than twice what the same rows in random order do: 0.21
    and 0.058 ms where a wavefront had 64 adjacent rows, 0.050 and 0.047 now."""
    torch = torch_gpu
    stream = torch.cuda.current_stream()
    handle = api.Handle(stream=stream.cuda_stream)
    a = sorted_power_law(dtype)
    lengths = np.diff(a.ptr)
    order = np.random.default_rng(4).permutation(a.m)
    mixed_ptr = np.concatenate([[0], np.cumsum(lengths[order])])
    places = np.repeat(a.ptr[order] - mixed_ptr[:-1], lengths[order]) + np.arange(a.nnz)
    mixed = wl.Csr(a.m, a.n, mixed_ptr, a.col[places], a.val[places], 0).with_base(0)
    times = []
    for matrix in (a, mixed):
        rows = dev(torch, np.repeat(np.arange(a.m, dtype=np.int32), np.diff(matrix.ptr)))
        col, val = dev(torch, matrix.col), dev(torch, matrix.val)
        mat = api.SpMat(a.m, a.n, a.nnz, rows, col, val, fmt=api.FORMAT_COO)
        B, C = (torch.zeros((k, n), dtype=val.dtype, device="cuda") for k in (a.n, a.m))
        call = (handle, api.OP_N, api.OP_N, 1.0, mat, api.DnMat(a.n, n, n, B), 0.0, api.DnMat(a.m, n, n, C), api.maca_type(np.dtype(dtype)))
        st, size = api.spmm_buffer_size(*call)
        assert st == 0
        buf = torch.empty(size, dtype=torch.uint8, device="cuda")
        best = 1e9
        for _ in range(8):
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            for _ in range(5):
                assert api.spmm(*call, buf) == 0
            e1.record()
            torch.cuda.synchronize()
            best = min(best, e0.elapsed_time(e1) / 5)
        times.append(best)
    handle.destroy()
    assert times[0] < 2 * times[1], times


def launches_of(torch, call):
    """How many launches a call is, from a graph that has captured it."""
    import ctypes
    with open("/proc/self/maps") as maps:
        runtime = ctypes.CDLL(next(line.split()[-1] for line in maps if "libamdhip64" in line))
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph, stream=call[0]):
        assert call[1]() == 0
    nodes = ctypes.c_size_t()
    assert runtime.hipGraphGetNodes(ctypes.c_void_p(graph.raw_cuda_graph()), None, ctypes.byref(nodes)) == 0
    return nodes.value


@pytest.mark.parametrize("dtype,narrow,wide", [(np.float32, 16, 32), (np.float64, 16, 32), (np.float64, 8, 32)])
def test_rows_of_wavefronts_cost_no_launch_of_their_own(torch_gpu, dtype, narrow, wide):
    """A call that does not know whether there are long rows (COO): as many launches where rows are taken by parts of wavefronts as
    for wider operands, whose rows never are."""
    torch = torch_gpu
    side = torch.cuda.Stream()
    handle = api.Handle(stream=side.cuda_stream)
    a = wl.random_ragged(3000, 2000, 16, dtype=dtype, seed=1)
    rows = dev(torch, np.repeat(np.arange(a.m, dtype=np.int32), np.diff(a.ptr)))
    col, val = dev(torch, a.col), dev(torch, a.val)
    counts = []
    for n in (narrow, wide):
        mat = api.SpMat(a.m, a.n, a.nnz, rows, col, val, fmt=api.FORMAT_COO)
        B, C = (torch.zeros((k, n), dtype=val.dtype, device="cuda") for k in (a.n, a.m))
        call = (handle, api.OP_N, api.OP_N, 1.0, mat, api.DnMat(a.n, n, n, B), 0.0, api.DnMat(a.m, n, n, C), api.maca_type(np.dtype(dtype)))
        st, size = api.spmm_buffer_size(*call)
        assert st == 0
        buf = torch.empty(size, dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        counts.append(launches_of(torch, (side, lambda: api.spmm(*call, buf))))
    assert counts[0] == counts[1] > 0, counts
