"""The copy along the diagonals that mcsparseSpMV_preprocess tries for a direction that does not transpose
(csrc/spmv_diagonals.hip): rows around the edges of its slices, grid lines that end inside them, holes, every format and
index type that can be prepared, against the oracle within 8*u*(|alpha| * |A||x| + |beta*y|); matrices it must refuse; x
with infinities; an overwritten copy; capture."""
import numpy as np
import pytest

from mcsparse_amd import api
from mcsparse_amd import workloads as wl

from gpu_util import assert_within, dev

pytestmark = pytest.mark.gpu


def grid(sides, reach, dtype, seed, keep=1.0, extra_columns=0):
    """Every point of a grid with its neighbours of `reach` steps, values U[-1, 1]; a share 1 - keep of the entries left out."""
    rng = np.random.default_rng(seed)
    strides = np.cumprod([1] + list(sides[:-1]))
    m = int(np.prod(sides))
    at = [np.arange(m) // s % n for s, n in zip(strides, sides)]
    rows, cols = [], []
    for step in reach:
        ok = rng.random(m) < keep
        for p, n, d in zip(at, sides, step):
            ok &= (p + d >= 0) & (p + d < n)
        rows.append(np.nonzero(ok)[0])
        cols.append(rows[-1] + int(sum(d * s for d, s in zip(step, strides))))
    rows, cols = np.concatenate(rows), np.concatenate(cols)
    order = np.lexsort((cols, rows))
    ptr = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=m))])
    return wl.Csr(m, m + extra_columns, ptr, cols[order], rng.uniform(-1, 1, order.size).astype(dtype), 0)


BOX = [(dx, dy, dz) for dz in (-1, 0, 1) for dy in (-1, 0, 1) for dx in (-1, 0, 1)]
CROSS = [(0, -1), (-1, 0), (0, 0), (1, 0), (0, 1)]


def prepare(torch, handle, a, alpha, beta, x, y, alg=api.SPMV_ALG_DEFAULT, fmt=api.FORMAT_CSR, index=np.int32):
    ct = api.maca_type(a.val.dtype)
    ptr, ind = dev(torch, a.ptr.astype(index)), dev(torch, a.col.astype(index))
    op, shape = api.OP_N, (a.m, a.n)
    if fmt == api.FORMAT_COO:
        ptr = dev(torch, (np.repeat(np.arange(a.m), np.diff(a.ptr.astype(np.int64))) + a.base).astype(index))
    elif fmt == api.FORMAT_CSC:  # the same arrays, read as the CSC of the transpose, and transposed back
        op, shape = api.OP_T, (a.n, a.m)
    mat = api.SpMat(shape[0], shape[1], a.nnz, ptr, ind, dev(torch, a.val), base=a.base, fmt=fmt,
                    **({} if index == np.int32 else {"index_type": api.INDEX_64I}))
    vx, vy = api.DnVec(x), api.DnVec(y)
    call = (handle, op, alpha, mat, vx, beta, vy, ct)
    st, size = api.spmv_preprocess_buffer_size(*call, alg=alg)
    assert st == api.STATUS_SUCCESS
    buf = torch.empty(size, dtype=torch.uint8, device="cuda")
    assert api.spmv_preprocess(*call, buf, alg=alg) == api.STATUS_SUCCESS
    return call, mat, buf


def check(torch, handle, oracle, a, alpha=1.5, beta=-0.5, in_use=True, what="diagonals", **how):
    rng = np.random.default_rng(11)
    dt = a.val.dtype
    x, y = rng.uniform(-1, 1, a.n).astype(dt), rng.uniform(-1, 1, a.m).astype(dt)
    d_x, d_y = dev(torch, x), dev(torch, y)
    call, mat, buf = prepare(torch, handle, a, alpha, beta, d_x, d_y, **how)
    assert (mat.spmv_diagonals() != 0) == in_use, what
    y_ref, bound = oracle.spmv(False, a.m, a.n, a.base, a.ptr, a.col, a.val, alpha, beta, x, y)
    first = None
    for _ in range(2):
        d_y.copy_(torch.from_numpy(y))
        assert api.spmv(*call, buf, alg=how.get("alg", api.SPMV_ALG_DEFAULT)) == api.STATUS_SUCCESS
        torch.cuda.synchronize()
        got = d_y.cpu().numpy()
        assert_within(got, y_ref, bound, dt, what=what)
        assert not in_use or first is None or np.array_equal(first, got)  # the sums have an order
        first = got
    return call, mat, buf, d_x, d_y


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("sides,reach,keep,base", [
    ((101, 97, 45), BOX, 1.0, 0), ((30, 211, 64), BOX, 1.0, 1), ((128, 64, 50), BOX, 1.0, 0),
    ((1000003,), [(-1,), (0,), (1,)], 1.0, 0),  # slices end inside a lane's rows
    ((1601, 1203), CROSS, 1.0, 1), ((101, 97, 45), BOX, 0.85, 0),  # holes in every diagonal
    # offsets of many slices: the vectors of x would begin before it and end behind it in many of them
    ((20, 30, 1000), [(0, 0, d) for d in range(-40, 41, 2)], 1.0, 0),
])
def test_grids(torch_gpu, handle, oracle, dtype, sides, reach, keep, base):
    check(torch_gpu, handle, oracle, grid(sides, reach, dtype, 3, keep).with_base(base), what=str((sides, keep)))


@pytest.mark.parametrize("alpha,beta", [(1.0, 0.0), (0.0, 2.0), (-2.0, 1.0)])
def test_scalars_and_more_columns_than_rows(torch_gpu, handle, oracle, alpha, beta):
    check(torch_gpu, handle, oracle, grid((77, 85, 91), BOX, np.float64, 5, extra_columns=1001), alpha, beta)


@pytest.mark.parametrize("how", [{"fmt": api.FORMAT_COO}, {"fmt": api.FORMAT_CSC}, {"alg": api.SPMV_CSR_ALG2}, {"index": np.int64}])
def test_formats_and_algorithms(torch_gpu, handle, oracle, how):
    check(torch_gpu, handle, oracle, grid((101, 97, 45), BOX, np.float64, 7).with_base(1), what=str(how), **how)


def test_matrices_that_are_refused(torch_gpu, handle, oracle):
    a = grid((101, 97, 45), BOX, np.float64, 9)
    row = slice(int(a.ptr[200000]), int(a.ptr[200001]))
    unsorted = wl.Csr(a.m, a.n, a.ptr, a.col.copy(), a.val, 0)
    unsorted.col[row] = unsorted.col[row][::-1]
    check(torch_gpu, handle, oracle, unsorted, in_use=False, what="one row unsorted")
    twice = wl.Csr(a.m, a.n, a.ptr, a.col.copy(), a.val, 0)
    twice.col[row.start + 1] = twice.col[row.start]
    check(torch_gpu, handle, oracle, twice, in_use=False, what="one column twice")
    check(torch_gpu, handle, oracle, grid((101, 97, 45), BOX, np.float64, 9, keep=0.5), in_use=False, what="half empty")
    check(torch_gpu, handle, oracle, wl.uniform_rows(m=100000, n=100000, per_row=9, dtype=np.float32), in_use=False, what="uniform")
    check(torch_gpu, handle, oracle, wl.power_law(m=100000, max_len=50000, dtype=np.float32), in_use=False, what="power law")


def test_without_the_trial_there_is_no_such_copy(torch_gpu, handle, oracle):
    handle.set_spmv_preprocess_trial(False)
    check(torch_gpu, handle, oracle, grid((101, 97, 45), BOX, np.float64, 9), in_use=False, what="no trial")


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_infinite_x_reaches_only_the_rows_that_hold_its_column(torch_gpu, handle, dtype):
    torch = torch_gpu
    a = grid((101, 97, 45), BOX, dtype, 13, keep=0.9)
    x = np.ones(a.n, dtype)
    x[[0, 5000, 250001, a.n - 1]] = np.inf, np.nan, -np.inf, np.inf
    d_x, d_y = dev(torch, x), torch.zeros(a.m, dtype=getattr(torch, np.dtype(dtype).name), device="cuda")
    call, mat, buf = prepare(torch, handle, a, 1.0, 0.0, d_x, d_y)
    assert mat.spmv_diagonals() != 0
    assert api.spmv(*call, buf) == api.STATUS_SUCCESS
    torch.cuda.synchronize()
    touched = np.zeros(a.m, bool)
    rows = np.repeat(np.arange(a.m), np.diff(a.ptr.astype(np.int64)))
    touched[rows[~np.isfinite(x[a.col])]] = True
    assert np.array_equal(np.isfinite(d_y.cpu().numpy()), ~touched)


def test_an_overwritten_copy_stays_in_bounds(torch_gpu, handle, oracle):
    torch = torch_gpu
    a = grid((101, 97, 45), BOX, np.float32, 15)
    call, mat, buf, d_x, d_y = check(torch, handle, oracle, a)
    for fill in (0xFF, 0x55, 0x00):
        buf.fill_(fill)
        assert api.spmv(*call, buf) == api.STATUS_SUCCESS
        torch.cuda.synchronize()
    gen = torch.Generator(device="cuda").manual_seed(1)
    buf.copy_(torch.randint(0, 256, (buf.numel(),), dtype=torch.uint8, device="cuda", generator=gen))
    assert api.spmv(*call, buf) == api.STATUS_SUCCESS
    torch.cuda.synchronize()


def test_replays_in_a_graph(torch_gpu, oracle):
    torch = torch_gpu
    a = grid((101, 97, 45), BOX, np.float64, 17)
    stream = torch.cuda.Stream()
    handle = api.Handle(stream=stream.cuda_stream)
    rng = np.random.default_rng(1)
    with torch.cuda.stream(stream):
        d_x, d_y = dev(torch, rng.uniform(-1, 1, a.n)), torch.zeros(a.m, dtype=torch.float64, device="cuda")
        call, mat, buf = prepare(torch, handle, a, 1.0, 0.0, d_x, d_y)
        assert mat.spmv_diagonals() != 0
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            assert api.spmv(*call, buf) == api.STATUS_SUCCESS
    for replay in range(3):
        x = rng.uniform(-1, 1, a.n)
        d_x.copy_(torch.from_numpy(x))
        d_y.fill_(7.0)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        y_ref, bound = oracle.spmv(False, a.m, a.n, 0, a.ptr, a.col, a.val, 1.0, 0.0, x, np.zeros(a.m))
        assert_within(d_y.cpu().numpy(), y_ref, bound, np.float64, what="replay %d" % replay)
    handle.destroy()
