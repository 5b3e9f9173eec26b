"""GPU parity of what is built on the partition of tiles by key bits (csrc/partition.hip), at the sizes where it can go
wrong: entry counts around a tile, both tile sizes, keys concentrated in a few runs, empty rows.  The transposing
mcsparseSpMV without a preprocess call is compared exactly (integer-valued operands make any order of summation exact),
csr2csc and the index sorts bit for bit against the oracle."""
import ctypes

import numpy as np
import pytest

from mcsparse_amd import api
from mcsparse_amd import workloads as wl

from gpu_util import dev, run_spmv

pytestmark = pytest.mark.gpu

LARGE_FROM = 128 * 8192  # entries up to which the tiles hold 4096 entries, beyond 8192


def matrix(kind, m, n, nnz, dtype, seed):
    """A CSR matrix with exactly nnz nonzeros: columns drawn from all of them, from a band around the diagonal, or mostly
    from a few; a fifth of the rows empty in the first case."""
    rng = np.random.default_rng(seed)
    weights = rng.random(m) * (rng.random(m) > 0.2 if kind == "uniform" else 1.0)
    cuts = np.concatenate([[0], np.round(np.cumsum(weights) / weights.sum() * nnz)]).astype(np.int64)
    cuts[-1] = nnz
    rows = np.repeat(np.arange(m), np.diff(cuts))
    if kind == "uniform":
        col = rng.integers(0, n, nnz)
    elif kind == "band":
        col = np.clip(rows * n // m + rng.integers(-20, 21, nnz), 0, n - 1)
    else:
        col = np.where(rng.random(nnz) < 0.7, rng.integers(0, 5, nnz) * (n // 7), rng.integers(0, n, nnz))
    col = col[np.lexsort((col, rows))]
    return wl.Csr(m, n, cuts, col, rng.integers(-3, 4, nnz).astype(dtype), 0)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("kind,m,n,nnz", [
    ("uniform", 50, 40000, 1), ("uniform", 300, 40000, 4095), ("uniform", 300, 40000, 4096), ("uniform", 300, 40000, 4097),
    ("uniform", 30000, 20000, 300001), ("band", 50000, 70000, 700000), ("few", 60000, 200000, 900000),
    ("uniform", 400000, 1 << 22, LARGE_FROM), ("uniform", 400000, 300000, LARGE_FROM + 1),
    ("band", 200000, 150000, LARGE_FROM + 8191), ("few", 150000, 4000000, LARGE_FROM + 8192 * 30),
])
def test_transposed_product_exact(torch_gpu, handle, dtype, kind, m, n, nnz):
    a = matrix(kind, m, n, nnz, dtype, seed=nnz)
    rng = np.random.default_rng(3)
    x, y = rng.integers(-4, 5, m).astype(dtype), rng.integers(-8, 9, n).astype(dtype)
    want = 2 * (a.to_scipy().T.astype(np.float64) @ x.astype(np.float64)) - 3 * y
    st, got, _ = run_spmv(torch_gpu, handle, a, x, y, 2.0, -3.0, op=api.OP_T)
    assert st == api.STATUS_SUCCESS
    assert np.array_equal(got.astype(np.float64), want)


ONE_LEVEL_UPTO = 4300 << 11  # entries up to which one partition makes the buckets that are sorted in LDS


@pytest.mark.parametrize("dtype,action", [(np.float32, api.ACTION_NUMERIC), (np.float64, api.ACTION_NUMERIC),
                                          (np.float32, api.ACTION_SYMBOLIC)])
@pytest.mark.parametrize("kind,m,n,nnz,base", [
    ("uniform", 5, 1, 40, 0), ("uniform", 50, 200, 1, 1), ("uniform", 400, 256, 4097, 0), ("uniform", 300, 257, 20000, 1),
    ("uniform", 3000, 70000, 6145, 0), ("few", 50, 3, 30000, 0), ("few", 3000, 1 << 16, 400000, 1),
    ("band", 100000, 90000, 1000001, 0), ("uniform", 100000, 5000, LARGE_FROM, 0), ("few", 100000, 300000, LARGE_FROM + 1, 1),
    ("uniform", 300000, 1 << 20, ONE_LEVEL_UPTO, 0), ("uniform", 300000, (1 << 20) + 1, ONE_LEVEL_UPTO + 1, 1),
    ("few", 300000, 1 << 22, ONE_LEVEL_UPTO + 777, 0), ("band", 300000, 3000000, 2 * ONE_LEVEL_UPTO, 0),
    ("uniform", 20000, (1 << 24) + 1, 500000, 0),
    # two levels with keys short enough for 8 bits behind the first one
    ("uniform", 300000, 4000, ONE_LEVEL_UPTO + 1, 0), ("few", 300000, 1 << 14, ONE_LEVEL_UPTO + 777, 1),
])
def test_csr2csc_bit_exact(torch_gpu, handle, oracle, dtype, action, kind, m, n, nnz, base):
    torch = torch_gpu
    a = matrix(kind, m, n, nnz, dtype, seed=nnz).with_base(base)
    d_ptr, d_col, d_val = dev(torch, a.ptr), dev(torch, a.col), dev(torch, a.val)
    o_val = torch.full((nnz,), -9.0, dtype=d_val.dtype, device="cuda")
    o_ptr, o_row = (torch.full((k,), -9, dtype=torch.int32, device="cuda") for k in (n + 1, nnz))
    args = (handle, m, n, nnz, d_val, d_ptr, d_col, o_val, o_ptr, o_row, api.maca_type(np.dtype(dtype)), action, base)
    st, size = api.csr2csc_buffer_size(*args)
    assert st == api.STATUS_SUCCESS
    buf = torch.empty(size, dtype=torch.uint8, device="cuda")
    want_ptr, want_row, want_val = oracle.csr2csc(m, n, base, a.ptr, a.col, a.val, method="counting")
    for _ in range(2):
        assert api.csr2csc(*args, buf) == api.STATUS_SUCCESS
    torch.cuda.synchronize()
    assert np.array_equal(o_ptr.cpu().numpy().view(np.uint32), want_ptr)
    assert np.array_equal(o_row.cpu().numpy().view(np.uint32), want_row)
    if action == api.ACTION_NUMERIC:
        assert np.array_equal(o_val.cpu().numpy(), want_val)
    else:
        assert (o_val == -9.0).all()


@pytest.mark.parametrize("dtype,action", [(np.float32, api.ACTION_NUMERIC), (np.float64, api.ACTION_NUMERIC),
                                          (np.float32, api.ACTION_SYMBOLIC)])
@pytest.mark.parametrize("m,n,gap,base", [
    # a row every `gap` rows: with 2^22 columns the word behind the first partition has room for 2^17 rows of a tile
    ((1 << 24) - 1, 1 << 22, 131071, 0), ((1 << 24) - 1, 1 << 22, 131072, 1), ((1 << 24) - 1, 1 << 22, 1 << 20, 1),
    # one row more than a word holds beside eight bits of the column: rows and keys apart
    (1 << 24, 1 << 22, 131072, 1),
    # with 2^16 columns the room behind the first partition is 2^22 rows
    ((1 << 24) - 1, 1 << 16, (1 << 22) - 1, 0), ((1 << 24) - 1, 1 << 16, 1 << 22, 0),
])
def test_csr2csc_tiles_of_many_rows(torch_gpu, handle, oracle, dtype, action, m, n, gap, base):
    torch = torch_gpu
    nnz = ONE_LEVEL_UPTO + 12345
    full = np.arange(0, m, gap)
    rng = np.random.default_rng(gap)
    lengths = np.zeros(m, dtype=np.int64)
    lengths[full] = nnz // full.size
    lengths[full[-1]] += nnz - lengths.sum()
    ptr = np.concatenate([[0], np.cumsum(lengths)])
    a = wl.Csr(m, n, ptr, rng.integers(0, n, nnz), rng.integers(-3, 4, nnz).astype(dtype), 0).with_base(base)
    d_ptr, d_col, d_val = dev(torch, a.ptr), dev(torch, a.col), dev(torch, a.val)
    o_val = torch.full((nnz,), -9.0, dtype=d_val.dtype, device="cuda")
    o_ptr, o_row = (torch.full((k,), -9, dtype=torch.int32, device="cuda") for k in (n + 1, nnz))
    args = (handle, m, n, nnz, d_val, d_ptr, d_col, o_val, o_ptr, o_row, api.maca_type(np.dtype(dtype)), action, base)
    st, size = api.csr2csc_buffer_size(*args)
    assert st == api.STATUS_SUCCESS
    buf = torch.empty(size, dtype=torch.uint8, device="cuda")
    want_ptr, want_row, want_val = oracle.csr2csc(m, n, base, a.ptr, a.col, a.val, method="counting")
    assert api.csr2csc(*args, buf) == api.STATUS_SUCCESS
    torch.cuda.synchronize()
    assert np.array_equal(o_ptr.cpu().numpy().view(np.uint32), want_ptr)
    assert np.array_equal(o_row.cpu().numpy().view(np.uint32), want_row)
    if action == api.ACTION_NUMERIC:
        assert np.array_equal(o_val.cpu().numpy(), want_val)


@pytest.mark.parametrize("by", ["row", "column"])
@pytest.mark.parametrize("with_perm", [True, False])
@pytest.mark.parametrize("kind,m,n,nnz", [
    ("uniform", 3, 2, 1), ("uniform", 90, 3000000, 6144), ("uniform", 3000000, 90, 6145), ("few", 40, 50, 70000),
    ("few", 4000, 70000, 300000), ("band", 300000, 40000, 1000000), ("uniform", 1 << 23, 1 << 22, 100000),
    ("few", 100000, 1 << 22, ONE_LEVEL_UPTO), ("uniform", 1 << 22, 1 << 20, ONE_LEVEL_UPTO + 1),
    ("uniform", 1 << 24, 300, 50000), ("uniform", 5000, 100000, ONE_LEVEL_UPTO + 1),
    # what is left of the major key and the minor one: more than 32 bits, so that no word holds both, and one row in pieces;
    # 32 bits, where only the sort by column may have both in a word (the other could be all ones)
    ("few", 1 << 22, 1 << 22, 2000000), ("uniform", 1 << 22, (1 << 21) - 1, ONE_LEVEL_UPTO + 1),
])
def test_coosort_bit_exact(torch_gpu, handle, oracle, by, with_perm, kind, m, n, nnz):
    torch = torch_gpu
    a = matrix(kind, m, n, nnz, np.float32, seed=nnz)
    rng = np.random.default_rng(nnz)
    order = rng.permutation(nnz)
    rows = np.repeat(np.arange(m, dtype=np.int32), a.row_lengths())[order]
    cols, perm = a.col[order], rng.permutation(nnz).astype(np.int32)
    if kind == "few":  # and one row with a third of all entries
        rows[rng.random(nnz) < 0.33] = m // 2
    d_r, d_c, d_p = dev(torch, rows), dev(torch, cols), dev(torch, perm) if with_perm else None
    st, size = api.sort_buffer_size(handle, "coo", m, n, nnz, d_r, d_c)
    assert st == api.STATUS_SUCCESS
    buf = torch.empty(size, dtype=torch.uint8, device="cuda")
    sort = api.xcoosort_by_row if by == "row" else api.xcoosort_by_column
    assert sort(handle, m, n, nnz, d_r, d_c, d_p, buf) == api.STATUS_SUCCESS
    torch.cuda.synchronize()
    want = np.lexsort((cols, rows) if by == "row" else (rows, cols))  # stable
    assert np.array_equal(d_r.cpu().numpy(), rows[want])
    assert np.array_equal(d_c.cpu().numpy(), cols[want])
    if with_perm:
        assert np.array_equal(d_p.cpu().numpy(), perm[want])


@pytest.mark.parametrize("with_perm", [True, False])
@pytest.mark.parametrize("how", ["row", "column", "csr"])
@pytest.mark.parametrize("minor", [(1 << 24) - 2, (1 << 24) - 1, 1 << 24])
def test_index_sorts_with_minor_keys_of_24_bits(torch_gpu, handle, how, with_perm, minor):
    """Ten million entries in a million rows leave eight bits of the major key behind two partitions.  With a minor extent
    of 2^24 - 2 they share a word with the minor key, with 2^24 - 1 (one-based indices reach it) they are the only eight
    that travel by themselves, and 2^24 is beyond the partitions."""
    torch, major, nnz = torch_gpu, 1000000, 10000000
    gen = torch.Generator(device="cuda").manual_seed(minor)
    hi, lo = (torch.randint(0, k, (nnz,), generator=gen, dtype=torch.int32, device="cuda") for k in (major, minor))
    lo[:3] = minor - 1
    perm = torch.randperm(nnz, generator=gen, device="cuda").to(torch.int32)
    if how == "csr":
        hi = hi.sort().values
        ptr = torch.searchsorted(hi, torch.arange(major + 1, dtype=torch.int32, device="cuda")).to(torch.int32)
    want = torch.sort(hi.long() << 24 | lo, stable=True).indices
    d_hi, d_lo, d_p = hi.clone(), lo.clone(), perm.clone() if with_perm else None
    kind, arrays = ("csr", (ptr, d_lo)) if how == "csr" else ("coo", (d_hi, d_lo))
    m, n = (minor, major) if how == "column" else (major, minor)
    st, size = api.sort_buffer_size(handle, kind, m, n, nnz, *arrays)
    assert st == api.STATUS_SUCCESS
    buf = torch.empty(size, dtype=torch.uint8, device="cuda")
    if how == "csr":
        descr = ctypes.c_void_p()
        assert handle.lib.mcsparseCreateMatDescr(ctypes.byref(descr)) == 0
        assert api.xcsrsort(handle, m, n, nnz, descr, ptr, d_lo, d_p, buf) == api.STATUS_SUCCESS
        handle.lib.mcsparseDestroyMatDescr(descr)
    elif how == "row":
        assert api.xcoosort_by_row(handle, m, n, nnz, d_hi, d_lo, d_p, buf) == api.STATUS_SUCCESS
    else:
        assert api.xcoosort_by_column(handle, m, n, nnz, d_lo, d_hi, d_p, buf) == api.STATUS_SUCCESS
    torch.cuda.synchronize()
    assert torch.equal(d_lo, lo[want])
    assert how == "csr" or torch.equal(d_hi, hi[want])
    assert not with_perm or torch.equal(d_p, perm[want])


@pytest.mark.parametrize("longest", [3, 64, 65, 700])  # 64: up to there a bucket's entries are counted, not sorted in passes
@pytest.mark.parametrize("columns", [2, 70000])
def test_coosort_runs_and_equal_pairs(torch_gpu, handle, longest, columns):
    torch, rng, m, nnz = torch_gpu, np.random.default_rng(longest), 300000, 600001
    rows, cols = rng.integers(0, m, nnz, dtype=np.int32), rng.integers(0, columns, nnz, dtype=np.int32)
    rows[:longest] = m - 1  # in the last bucket, and in front of the places behind it
    cols[:longest] = rng.integers(69998, 70000, longest)
    order = rng.permutation(nnz)
    rows, cols, perm = rows[order], cols[order], np.arange(nnz, dtype=np.int32)
    d_r, d_c, d_p = dev(torch, rows), dev(torch, cols), dev(torch, perm)
    st, size = api.sort_buffer_size(handle, "coo", m, 70000, nnz, d_r, d_c)
    assert st == api.STATUS_SUCCESS
    buf = torch.full((size,), 255, dtype=torch.uint8, device="cuda")
    assert api.xcoosort_by_row(handle, m, 70000, nnz, d_r, d_c, d_p, buf) == api.STATUS_SUCCESS
    torch.cuda.synchronize()
    want = np.lexsort((cols, rows))  # stable
    assert np.array_equal(d_p.cpu().numpy(), want)
    assert np.array_equal(d_r.cpu().numpy(), rows[want])
    assert np.array_equal(d_c.cpu().numpy(), cols[want])


# buckets beyond what LDS holds: one chunk and an entry more, several of a bucket and of buckets in turn; the two keys in a word
# (of 9 to 32 bits, in one to four passes) and apart
@pytest.mark.parametrize("with_perm", [True, False])
@pytest.mark.parametrize("columns", [1, 200, 70000, (1 << 22) - 2, 1 << 24])
@pytest.mark.parametrize("popular", [[6145], [6144, 6145, 12289], [30000, 1, 100000]])
def test_coosort_of_popular_rows(torch_gpu, handle, popular, columns, with_perm):
    torch = torch_gpu
    m, rest = 3001, 40000
    gen = torch.Generator(device="cuda").manual_seed(columns)
    rows = torch.randint(0, m, (rest,), generator=gen, dtype=torch.int32, device="cuda")
    rows = torch.cat([rows] + [torch.full((c,), 17 + 900 * i, dtype=torch.int32, device="cuda") for i, c in enumerate(popular)])
    rows = rows[torch.randperm(rows.numel(), generator=gen, device="cuda")]
    cols = torch.randint(0, columns, (rows.numel(),), generator=gen, dtype=torch.int32, device="cuda")
    order = torch.sort(rows.long() * columns + cols, stable=True).indices
    perm = torch.arange(rows.numel(), dtype=torch.int32, device="cuda") if with_perm else None
    got_rows, got_cols = rows.clone(), cols.clone()
    st, size = api.sort_buffer_size(handle, "coo", m, columns, rows.numel(), rows, cols)
    assert st == 0
    buffer = torch.empty(size, dtype=torch.uint8, device="cuda")
    assert api.xcoosort_by_row(handle, m, columns, rows.numel(), got_rows, got_cols, perm, buffer) == 0
    torch.cuda.synchronize()
    assert torch.equal(got_rows, rows[order]) and torch.equal(got_cols, cols[order])
    assert perm is None or torch.equal(perm.long(), order)


@pytest.mark.parametrize("share", [0.3, 0.9])  # 0.9: one bucket with more tiles of the second step than the first has
def test_a_row_with_most_of_ten_million_entries(torch_gpu, handle, share):
    """Many more pieces of one bucket than workgroups that work on it, in every pass: what one workgroup writes is read
    by others of the same launch, on other XCDs."""
    torch = torch_gpu
    m, n, nnz = 1 << 22, 1 << 20, 10000000
    rng = np.random.default_rng(int(10 * share))
    rows = np.where(rng.random(nnz) < share, m // 3, rng.integers(0, m, nnz)).astype(np.int32)
    cols, perm = rng.integers(0, n, nnz).astype(np.int32), np.arange(nnz, dtype=np.int32)
    want = np.argsort(rows.astype(np.int64) * n + cols, kind="stable")
    st, size = api.sort_buffer_size(handle, "coo", m, n, nnz, dev(torch, rows), dev(torch, cols))
    assert st == api.STATUS_SUCCESS
    buf = torch.empty(size, dtype=torch.uint8, device="cuda")
    for _ in range(3):
        d_r, d_c, d_p = dev(torch, rows), dev(torch, cols), dev(torch, perm)
        assert api.xcoosort_by_row(handle, m, n, nnz, d_r, d_c, d_p, buf) == api.STATUS_SUCCESS
        torch.cuda.synchronize()
        assert np.array_equal(d_p.cpu().numpy(), perm[want])
        assert np.array_equal(d_r.cpu().numpy(), rows[want])
        assert np.array_equal(d_c.cpu().numpy(), cols[want])


def best_us(torch, call, repeats=5):
    """Shortest time of a few calls after one that is not looked at."""
    call()
    torch.cuda.synchronize()
    best = float("inf")
    for _ in range(repeats):
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        call()
        e1.record()
        e1.synchronize()
        best = min(best, e0.elapsed_time(e1) * 1e3)
    return best


def csr2csc_us(torch, handle, m, per_row, n, col):
    """Time of csr2csc on m rows of per_row nonzeros with these columns (device tensor), which is checked first."""
    nnz = m * per_row
    ptr = torch.arange(m + 1, dtype=torch.int32, device="cuda") * per_row
    val = torch.rand(nnz, dtype=torch.float32, device="cuda")
    o_ptr = torch.zeros(n + 1, dtype=torch.int32, device="cuda")
    o_row, o_val = torch.zeros(nnz, dtype=torch.int32, device="cuda"), torch.zeros_like(val)
    args = (handle, m, n, nnz, val, ptr, col, o_val, o_ptr, o_row, api.R_32F, api.ACTION_NUMERIC, api.BASE_ZERO)
    st, size = api.csr2csc_buffer_size(*args)
    assert st == api.STATUS_SUCCESS
    buf = torch.empty(size, dtype=torch.uint8, device="cuda")
    assert api.csr2csc(*args, buf) == api.STATUS_SUCCESS
    order = torch.sort(col, stable=True).indices
    assert torch.equal(o_val, val[order]) and torch.equal(o_row, (order // per_row).to(torch.int32))
    del order
    return best_us(torch, lambda: api.csr2csc(*args, buf))


def coosort_us(torch, handle, m, n, rows, cols):
    nnz = rows.numel()
    d_r, d_c, d_p = (torch.empty_like(rows) for _ in range(3))
    st, size = api.sort_buffer_size(handle, "coo", m, n, nnz, d_r, d_c)
    assert st == api.STATUS_SUCCESS
    buf = torch.empty(size, dtype=torch.uint8, device="cuda")

    def call():
        d_r.copy_(rows)
        d_c.copy_(cols)
        assert api.create_identity_permutation(handle, nnz, d_p) == api.STATUS_SUCCESS
        assert api.xcoosort_by_row(handle, m, n, nnz, d_r, d_c, d_p, buf) == api.STATUS_SUCCESS

    call()
    order = torch.sort(rows.long() * n + cols, stable=True).indices
    assert torch.equal(d_p, order.to(torch.int32)) and torch.equal(d_r, rows[order]) and torch.equal(d_c, cols[order])
    del order
    return best_us(torch, call)


@pytest.mark.parametrize("few", [16, 1000])
def test_few_keys_take_no_longer_than_many(torch_gpu, handle, few):
    """16.8 M entries with 16 or 1000 keys against as many with a million: keys that fill more than a bucket each go to
    the LSD passes (two to six times the time of many keys when they were sorted in buckets)."""
    torch = torch_gpu
    m, per_row, many = 1 << 20, 16, 1 << 20

    def drawn(k):
        gen = torch.Generator(device="cuda").manual_seed(k)
        return torch.randint(0, k, (m * per_row,), generator=gen, dtype=torch.int32, device="cuda")

    assert csr2csc_us(torch, handle, m, per_row, few, drawn(few)) < 1.4 * csr2csc_us(torch, handle, m, per_row, many, drawn(many))
    other = drawn(many - 1)
    assert coosort_us(torch, handle, few, many, drawn(few), other) < 2 * coosort_us(torch, handle, many, many, drawn(many), other)


def test_popular_keys_do_not_hold_a_sort_up(torch_gpu, handle):
    """Keys by Zipf's law against evenly spread ones: four fifths of the entries lie in buckets that do not fit LDS.
    csr2csc of 67 M nonzeros took 4.3 times as long, an index sort of 10 M triples 5.7 times, when those buckets were
    sorted chunk by chunk under device-wide fences; 1.7 and 2.9 times now."""
    torch = torch_gpu
    gen = torch.Generator(device="cuda").manual_seed(9)

    def zipf(n, count):
        cdf = torch.cumsum(1.0 / torch.arange(1, n + 1, dtype=torch.float64, device="cuda"), 0)
        draw = torch.rand(count, generator=gen, dtype=torch.float64, device="cuda") * cdf[-1]
        return torch.searchsorted(cdf, draw).clamp(max=n - 1).to(torch.int32)

    def even(n, count):
        return torch.randint(0, n, (count,), generator=gen, dtype=torch.int32, device="cuda")

    n, m, per_row = 1 << 22, 1 << 23, 8
    assert csr2csc_us(torch, handle, m, per_row, n, zipf(n, m * per_row)) < \
        2.5 * csr2csc_us(torch, handle, m, per_row, n, even(n, m * per_row))
    n, nnz = 1 << 20, 10000000
    cols = even(n, nnz)
    assert coosort_us(torch, handle, n, n, zipf(n, nnz), cols) < 4 * coosort_us(torch, handle, n, n, even(n, nnz), cols)
