"""mcsparseSpMM with column-major operands from the diagonals mcsparseSpMM_preprocess keeps (csrc/spmm_diagonals.hip): widths
around a wavefront's four columns, runs of diagonals shorter and longer than three, slices at the ends of op(B), holes,
leading dimensions, index types and bases, against the oracle within 8*u*(|alpha| * |A||B| + |beta*C|); what must not use them;
new values, other operands in between, infinities, an overwritten buffer, capture."""
import numpy as np
import pytest

from mcsparse_amd import api
from mcsparse_amd import workloads as wl

from gpu_util import assert_within, dev
from test_gpu_spmv_diagonals import BOX, CROSS, grid

pytestmark = pytest.mark.gpu


class Call:
    """A prepared product: op(B) (a.n x n) and C (a.m x n) held as the columns of arrays with leading dimensions."""

    def __init__(self, torch, handle, a, n, alpha=1.5, beta=-0.5, op_b=api.OP_N, pad_b=0, pad_c=0, index=np.int32, seed=21):
        rng = np.random.default_rng(seed)
        dt = a.val.dtype
        self.torch, self.a, self.n, self.alpha, self.beta = torch, a, n, alpha, beta
        self.B, self.C0 = rng.uniform(-1, 1, (a.n, n)).astype(dt), rng.uniform(-1, 1, (a.m, n)).astype(dt)
        image = np.full((n, a.n + pad_b), 55.0, dt)
        image[:, :a.n] = self.B.T
        self.c_image = np.full((n, a.m + pad_c), 99.0, dt)
        self.c_image[:, :a.m] = self.C0.T
        self.d_B, self.d_C, self.d_val = dev(torch, image), dev(torch, self.c_image), dev(torch, a.val)
        self.mat = api.SpMat(a.m, a.n, a.nnz, dev(torch, a.ptr.astype(index)), dev(torch, a.col.astype(index)), self.d_val,
                             base=a.base, **({} if index == np.int32 else {"index_type": api.INDEX_64I}))
        shape, order = ((a.n, n), api.ORDER_COL) if op_b == api.OP_N else ((n, a.n), api.ORDER_ROW)
        self.mB = api.DnMat(shape[0], shape[1], a.n + pad_b, self.d_B, order=order)
        self.mC = api.DnMat(a.m, n, a.m + pad_c, self.d_C, order=api.ORDER_COL)
        self.args = (handle, api.OP_N, op_b, alpha, self.mat, self.mB, beta, self.mC, api.maca_type(dt))
        st, size = api.spmm_buffer_size(*self.args)
        assert st == api.STATUS_SUCCESS
        self.buf = torch.empty(size, dtype=torch.uint8, device="cuda")
        assert api.spmm_preprocess(*self.args, self.buf) == api.STATUS_SUCCESS

    def run(self):
        self.d_C.copy_(self.torch.from_numpy(self.c_image))
        assert api.spmm(*self.args, self.buf) == api.STATUS_SUCCESS
        self.torch.cuda.synchronize()
        return self.d_C.cpu().numpy()

    def check(self, oracle, what=""):
        a = self.a
        got = self.run()
        assert (got[:, a.m:] == 99.0).all()
        ref, bound = oracle.spmm(a.m, self.n, a.base, a.ptr, a.col, a.val, self.alpha, self.beta, self.B.ravel(), self.n, True,
                                 self.C0, self.n, True)
        assert_within(got[:, :a.m].T, ref, bound, a.val.dtype, what=what)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("sides,reach,keep,base", [
    ((41, 37, 29), BOX, 1.0, 0), ((64, 32, 30), BOX, 1.0, 1), ((401, 403), CROSS, 1.0, 0), ((41, 37, 29), BOX, 0.85, 1),
    ((200003,), [(d,) for d in (-9, -8, -7, -6, -5, -1, 0, 2, 3, 300, 301, 302, 303)], 1.0, 0),  # runs of five, two, two, four
    ((20, 30, 60), [(0, 0, d) for d in range(-13, 14)], 1.0, 0),  # most slices name columns next to the ends of op(B)
])
def test_grids(torch_gpu, handle, oracle, dtype, sides, reach, keep, base):
    a = grid(sides, reach, dtype, 3, keep).with_base(base)
    for n in (1, 4, 7, 16, 17):
        call = Call(torch_gpu, handle, a, n, pad_b=3 * (n % 2), pad_c=n % 3)
        assert (call.mat.spmm_diagonals() != 0) == (dtype == np.float32 or n > 4)
        call.check(oracle, what=str((sides, keep, n)))


@pytest.mark.parametrize("how", [{"op_b": api.OP_T}, {"index": np.int64}, {"alpha": 1.0, "beta": 0.0}, {"alpha": 0.0, "beta": 2.0}])
@pytest.mark.parametrize("n", [5, 33])
def test_operations_scalars_and_indices(torch_gpu, handle, oracle, how, n):
    call = Call(torch_gpu, handle, grid((41, 37, 29), BOX, np.float64, 5, extra_columns=77), n, **how)
    assert call.mat.spmm_diagonals() != 0
    call.check(oracle, what=str(how))


def test_new_values_are_used(torch_gpu, handle, oracle):
    torch = torch_gpu
    call = Call(torch, handle, grid((41, 37, 29), BOX, np.float32, 7), 6)
    call.check(oracle)
    call.a.val[:] = np.random.default_rng(8).uniform(-1, 1, call.a.nnz).astype(np.float32)
    call.d_val.copy_(torch.from_numpy(call.a.val))
    call.check(oracle, what="values written after the preprocess call")


def test_row_major_call_in_between_leaves_them_alone(torch_gpu, handle, oracle):
    torch = torch_gpu
    call = Call(torch, handle, grid((41, 37, 29), BOX, np.float32, 7), 6)
    a = call.a
    d_B, d_C = dev(torch, call.B), torch.zeros((a.m, 6), dtype=torch.float32, device="cuda")
    other = (handle, api.OP_N, api.OP_N, 1.0, call.mat, api.DnMat(a.n, 6, 6, d_B), 0.0, api.DnMat(a.m, 6, 6, d_C), api.R_32F)
    st, size = api.spmm_buffer_size(*other)
    assert st == api.STATUS_SUCCESS and size <= call.buf.numel()
    assert api.spmm(*other, call.buf) == api.STATUS_SUCCESS
    torch.cuda.synchronize()
    ref, bound = oracle.spmm(a.m, 6, 0, a.ptr, a.col, a.val, 1.0, 0.0, call.B.ravel(), 6, True, None, 6, True)
    assert_within(d_C.cpu().numpy(), ref, bound, np.float32, what="row-major")
    call.check(oracle, what="column-major again")


def test_wider_operands_in_the_same_buffer_end_them(torch_gpu, handle, oracle):
    torch = torch_gpu
    a = grid((41, 37, 29), BOX, np.float32, 7)
    call, wide = Call(torch, handle, a, 6), Call(torch, handle, a, 30, seed=3)
    assert wide.buf.numel() > call.buf.numel()
    call.buf = wide.buf
    assert api.spmm_preprocess(*call.args, call.buf) == api.STATUS_SUCCESS
    call.check(oracle)
    args = list(wide.args)
    args[4] = call.mat  # the same matrix, the buffer that holds its diagonals
    wide.args = tuple(args)
    wide.check(oracle, what="wider")
    assert call.mat.spmm_diagonals() == 0
    call.check(oracle, what="narrow again")


def test_matrices_without_such_rows(torch_gpu, handle, oracle):
    a = grid((41, 37, 29), BOX, np.float64, 9)
    row = slice(int(a.ptr[20000]), int(a.ptr[20001]))
    unsorted = wl.Csr(a.m, a.n, a.ptr, a.col.copy(), a.val, 0)
    unsorted.col[row] = unsorted.col[row][::-1]
    wide = grid((7000,), [(d,) for d in range(-30, 31)], np.float64, 4)  # more values in a slice than LDS has room for
    for m, what in ((unsorted, "unsorted"), (grid((41, 37, 29), BOX, np.float64, 9, keep=0.5), "half empty"), (wide, "long rows"),
                    (wl.uniform_rows(m=30000, n=30000, per_row=9, dtype=np.float64), "uniform")):
        call = Call(torch_gpu, handle, m, 6)
        assert call.mat.spmm_diagonals() == 0, what
        call.check(oracle, what=what)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_infinite_elements_reach_only_the_rows_that_name_them(torch_gpu, handle, dtype):
    torch = torch_gpu
    call = Call(torch, handle, grid((41, 37, 29), BOX, dtype, 13, keep=0.9), 5, alpha=1.0, beta=0.0)
    assert call.mat.spmm_diagonals() != 0
    a, B = call.a, np.ones((call.a.n, 5), dtype)
    for j, at in enumerate((0, 5000, 30001, a.n - 1)):
        B[at, j] = (np.inf, np.nan, -np.inf, np.inf)[j]
    call.d_B.copy_(torch.from_numpy(np.ascontiguousarray(B.T)))
    got = call.run().T
    rows = np.repeat(np.arange(a.m), np.diff(a.ptr.astype(np.int64)))
    for j in range(5):
        touched = np.zeros(a.m, bool)
        touched[rows[~np.isfinite(B[a.col, j])]] = True
        assert np.array_equal(np.isfinite(got[:, j]), ~touched), j


def test_an_overwritten_buffer_stays_in_bounds(torch_gpu, handle, oracle):
    torch = torch_gpu
    call = Call(torch, handle, grid((41, 37, 29), BOX, np.float32, 15), 9)
    call.check(oracle)
    for fill in (0xFF, 0x55, 0x00):
        call.buf.fill_(fill)
        call.run()
    gen = torch.Generator(device="cuda").manual_seed(1)
    call.buf.copy_(torch.randint(0, 256, (call.buf.numel(),), dtype=torch.uint8, device="cuda", generator=gen))
    call.run()


def test_replays_in_a_graph(torch_gpu, oracle):
    torch = torch_gpu
    stream = torch.cuda.Stream()
    handle = api.Handle(stream=stream.cuda_stream)
    with torch.cuda.stream(stream):
        call = Call(torch, handle, grid((41, 37, 29), BOX, np.float64, 17), 5, alpha=1.0, beta=0.0)
        assert call.mat.spmm_diagonals() != 0
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            assert api.spmm(*call.args, call.buf) == api.STATUS_SUCCESS
    a = call.a
    for replay in range(3):
        B = np.random.default_rng(replay).uniform(-1, 1, (a.n, 5))
        call.d_B.copy_(torch.from_numpy(np.ascontiguousarray(B.T)))
        call.d_C.fill_(7.0)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        ref, bound = oracle.spmm(a.m, 5, 0, a.ptr, a.col, a.val, 1.0, 0.0, B.ravel(), 5, True, None, 5, True)
        assert_within(call.d_C.cpu().numpy().T, ref, bound, np.float64, what="replay %d" % replay)
    handle.destroy()


@pytest.mark.parametrize("n", [64, 63])  # columns of op(B) 6 MB apart: 64 are left to the blocks; 63 are not
@pytest.mark.parametrize("pad_c", [4, 1])  # 1: a C that the blocks do not write directly
def test_columns_on_the_same_sets_of_the_caches(torch_gpu, handle, oracle, n, pad_c):
    a = grid((64, 32, 16), BOX, np.float32, 31)
    call = Call(torch_gpu, handle, a, n, pad_b=(3 << 19) - a.n, pad_c=pad_c)
    assert call.mat.spmm_diagonals() > 0 and call.mat.spmm_schedule()[0] in (3, 4)
    call.check(oracle)
