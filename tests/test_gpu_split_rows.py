"""Kernels that split the work by values or by parts of a row instead of by
whole rows, at the sizes where that goes wrong: rows longer than a wave's
run of values, runs of empty rows, rows that end at a run's edge."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import _capi
from _util import storage, to_numpy, to_torch
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

DEV = "cuda"
VTYPES = ["float32", "float16", "bfloat16", "complex64"]


def _values(rng, shape, vtype):
    v = rng.standard_normal(shape)
    if vtype == "complex64":
        v = v + 1j * rng.standard_normal(shape)
    return storage(v, vtype)


def _csr(rng, lengths, n_cols, index_dtype=np.int32, bad=0.0):
    indptr = np.zeros(len(lengths) + 1, np.int64)
    np.cumsum(lengths, out=indptr[1:])
    indices = rng.integers(0, n_cols, int(indptr[-1]))
    if bad:
        indices[rng.random(indices.size) < bad] = -1
        indices[rng.random(indices.size) < bad] = n_cols
    return indices.astype(index_dtype), indptr.astype(index_dtype)


def _row_lengths(kind, rng):
    if kind == "one_row":
        return np.array([1000])
    if kind == "edges":  # rows that end on, before and after multiples of 64 and 256
        return np.array([64, 64, 128, 1, 63, 255, 1, 257, 0, 512, 0, 0])
    if kind == "empty_runs":  # more than 64 rows end inside 64 positions
        lengths = np.zeros(3000, np.int64)
        lengths[[0, 200, 201, 900, 2998]] = [3, 40, 700, 1, 20]
        return lengths
    lengths = rng.integers(0, 6, 2500)
    lengths[[0, 7, 1300, 2499]] = [5000, 300, 129, 2000]
    return lengths


@pytest.mark.parametrize("kind", ["one_row", "edges", "empty_runs", "skewed"])
@pytest.mark.parametrize("vtype", VTYPES)
def test_value_gradients_by_positions(kind, vtype):
    """Both value gradients equal the oracle bit for bit on every row
    structure, for column counts below, at and past a 16-byte load and a
    tile of 128 bytes, rows not aligned to 16 bytes included."""
    rng = np.random.default_rng(41)
    lengths = _row_lengths(kind, rng)
    n_rows, n_cols = len(lengths), 777
    index_dtype = np.int64 if kind == "edges" else np.int32
    indices, indptr = _csr(rng, lengths, n_cols, index_dtype, bad=0.02)
    nnz = indices.size
    x, cot = _values(rng, n_cols, vtype), _values(rng, n_rows, vtype)
    i, p = to_torch(indices, None, DEV), to_torch(indptr, None, DEV)
    print(f"value gradients {kind} {vtype}", flush=True)
    want = orc.csr_data_vjp(indices, indptr, x, cot, n_rows, n_cols, nnz, vtype=vtype)
    for plan in (None, _capi.Plan(p, n_rows, nnz, 64)):  # W = 64: rows past it are long
        got = _capi.spmv_data_vjp(i, p, to_torch(x, vtype, DEV), to_torch(cot, vtype, DEV), n_rows,
                                  n_cols, plan=plan)
        assert to_numpy(got).tobytes() == want.tobytes()
    for k in (1, 2, 3, 7, 16, 31, 32, 33, 100):
        X, C = _values(rng, (n_cols, k), vtype), _values(rng, (n_rows, k), vtype)
        got = _capi.spmm_data_vjp(i, p, to_torch(X, vtype, DEV), to_torch(C, vtype, DEV), n_rows,
                                  n_cols)
        want = orc.csr_data_vjp(indices, indptr, X, C, n_rows, n_cols, nnz, vtype=vtype)
        assert to_numpy(got).tobytes() == want.tobytes(), k


@pytest.mark.parametrize("longest", [96, 97, 513])
@pytest.mark.parametrize("vtype", VTYPES)
def test_value_gradients_around_the_split_rule(longest, vtype):
    """The vector's value gradient with the longest row at sixteen mean rows
    (lanes a row), one value above and far above (by positions), rows ending
    at the edges of a wave's 64 and 256 positions: the oracle's bits."""
    rng = np.random.default_rng(101)
    lengths = np.full(600, 6)
    lengths[:10] = [64, 64, 90, 1, 63, 0, 0, 33, 31, 90]
    lengths[300] = longest
    lengths[10:200] -= np.minimum(6, np.diff(np.linspace(0, lengths.sum() - 3650, 191).astype(int)))
    n_rows, n_cols = len(lengths), 777
    assert lengths.min() >= 0 and lengths.sum() // n_rows == 6 and lengths.max() == longest
    indices, indptr = _csr(rng, lengths, n_cols, np.int64, bad=0.02)
    nnz = indices.size
    x, cot = _values(rng, n_cols, vtype), _values(rng, n_rows, vtype)
    i, p = to_torch(indices, None, DEV), to_torch(indptr, None, DEV)
    plan = _capi.Plan(p, n_rows, nnz, 64)
    print(f"split rule {longest} {vtype}", flush=True)
    got = _capi.spmv_data_vjp(i, p, to_torch(x, vtype, DEV), to_torch(cot, vtype, DEV), n_rows,
                              n_cols, plan=plan)
    want = orc.csr_data_vjp(indices, indptr, x, cot, n_rows, n_cols, nnz, vtype=vtype)
    assert to_numpy(got).tobytes() == want.tobytes()
    plan.close()


@pytest.mark.parametrize("vtype,index_dtype,n_rows,n_cols,values", [
    ("float32", np.int32, 700_001, (4 << 20) // 4, 5 << 20),
    ("float32", np.int64, 900_003, (5 << 19) // 4, 12 << 20),
    ("bfloat16", np.int32, 900_001, (4 << 20) // 2 + 5, (5 << 20) + 3),
    ("float16", np.int64, 2_100_001, (4 << 20) // 2, 5 << 20),
    ("complex64", np.int32, 300_007, (4 << 20) // 8, 5 << 20),
])
def test_auto_panels_at_their_smallest_sizes(vtype, index_dtype, n_rows, n_cols, values):
    """The smallest matrices for which AUTO takes column panels: every short
    row equals the row blocks' bit for bit (unsorted and repeated columns,
    columns out of range and empty rows among them), long rows to their
    rounding, before and after new values; one value fewer keeps row blocks.
    Rows average at most 18 values: row blocks sum those in stored order,
    and only blocks averaging more than 32 in another."""
    rng = np.random.default_rng(5)
    # rows of any length up to twice the mean, two long ones, the count exact
    lengths = rng.multinomial(values - 1500, np.ones(n_rows) / n_rows)
    lengths[[3, n_rows - 2]] += [1000, 500]
    indices, indptr = _csr(rng, lengths, n_cols, index_dtype, bad=1e-4)
    nnz = indices.size
    assert nnz == values
    d = to_torch(_values(rng, nnz, vtype), vtype, DEV)
    x = to_torch(_values(rng, n_cols, vtype), vtype, DEV)
    i, p = to_torch(indices, None, DEV), to_torch(indptr, None, DEV)
    print(f"auto panels {vtype} {np.dtype(index_dtype).name} {n_rows}x{n_cols}", flush=True)
    auto = _capi.Plan(p, n_rows, nnz, data=d, indices=i, n_cols=n_cols)
    blocks = _capi.Plan(p, n_rows, nnz, data=d, indices=i, n_cols=n_cols,
                        slice_mode=_capi.SLICE_OFF)
    assert auto.info().n_panels > 0 and blocks.info().n_panels == 0
    for _ in range(2):
        got = _capi.spmv(d, i, p, x, n_rows, n_cols, auto)
        want = _capi.spmv(d, i, p, x, n_rows, n_cols, blocks)
        same = (got == want) | (got.isnan() & want.isnan())
        same[[3, n_rows - 2]] = True
        assert bool(same.all())
        # 1,000 products of two normals: 1e-5 of their magnitudes' sum (float32)
        scale = 1e-2 if vtype in ("float16", "bfloat16") else 1e-5
        for r in (3, n_rows - 2):
            assert abs(complex(got[r]) - complex(want[r])) <= scale * 1000
        d.mul_(0.5)
        auto.refresh(d)
    fewer = _capi.Plan(p, n_rows, nnz - 1, data=d[:-1], indices=i[:-1], n_cols=n_cols)
    if values in (5 << 20, 12 << 20):
        assert fewer.info().n_panels == 0
    for plan in (auto, blocks, fewer):
        plan.close()


@pytest.mark.parametrize("vtype", VTYPES)
@pytest.mark.parametrize("index_dtype", [np.int32, np.int64])
def test_spmm_long_rows_in_stored_order(vtype, index_dtype):
    """Long rows of a plan, a workgroup each, equal the oracle bit for bit at
    column counts around every tile width (16, 32, 64 columns) and below a
    16-byte load, rows a tile of products long, one value more and less
    among them; also where indptr changed after the plan was built (a row
    longer than it was then, and a listed row now short)."""
    rng = np.random.default_rng(43)
    lengths = rng.integers(0, 6, 2500)
    lengths[[0, 7, 900, 901, 1300, 2100, 2499]] = [5000, 257, 256, 255, 129, 1024, 2000]
    n_rows, n_cols = len(lengths), 3001
    indices, indptr = _csr(rng, lengths, n_cols, index_dtype, bad=0.01)
    nnz = indices.size
    data = _values(rng, nnz, vtype)
    d, i = to_torch(data, vtype, DEV), to_torch(indices, None, DEV)
    p = to_torch(indptr, None, DEV)
    plan = _capi.Plan(p, n_rows, nnz, 64, data=d, indices=i, n_cols=n_cols)
    assert plan.info().n_long_rows == 7
    # a column out of range adds nothing, as a zero does
    good = (indices >= 0) & (indices < n_cols)
    held, cols = np.where(good, data, np.zeros_like(data)), np.where(good, indices, 0)
    moved = indptr.copy()
    moved[8:901] = moved[901]  # row 7 takes the rows after it, rows 8 to 900 are empty
    for ptr in (indptr, moved):
        p.copy_(to_torch(ptr, None, DEV))
        for k in (1, 2, 3, 7, 16, 17, 32, 33, 63, 64, 65, 100, 130):
            X = _values(rng, (n_cols, k), vtype)
            print(f"spmm long rows {vtype} {np.dtype(index_dtype).name} k={k}", flush=True)
            got = _capi.spmm(d, i, p, to_torch(X, vtype, DEV), n_rows, n_cols, plan=plan)
            want = orc.csr_matmul(held, cols.astype(index_dtype), ptr, X, n_rows, vtype=vtype)
            assert to_numpy(got).tobytes() == want.tobytes(), k
    plan.close()


@pytest.mark.parametrize("vtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("n_cols", [32_700, 66_000, 140_000])
def test_spmm_narrow_16_bit_rows_of_scattered_matrices(vtype, n_cols):
    """16-bit X rows of one to four sixteen-byte vectors, X below 2 MB, about
    there and above (where the loads are taken apart at once): the oracle's
    bits."""
    rng = np.random.default_rng(97)
    lengths = rng.integers(0, 31, 2000)
    n_rows = len(lengths)
    indices, indptr = _csr(rng, lengths, n_cols)
    data = _values(rng, indices.size, vtype)
    d, i, p = to_torch(data, vtype, DEV), to_torch(indices, None, DEV), to_torch(indptr, None, DEV)
    plan = _capi.Plan(p, n_rows, indices.size, data=d, indices=i, n_cols=n_cols)
    assert 4 * plan.info().window_rows > n_cols
    for k in (8, 16, 24, 32):
        X = _values(rng, (n_cols, k), vtype)
        print(f"narrow 16-bit {vtype} {n_cols} k={k}", flush=True)
        got = _capi.spmm(d, i, p, to_torch(X, vtype, DEV), n_rows, n_cols, plan=plan)
        want = orc.csr_matmul(data, indices, indptr, X, n_rows, vtype=vtype)
        assert to_numpy(got).tobytes() == want.tobytes(), k
    plan.close()


@pytest.mark.parametrize("longest", [600, 9600, 9601])
def test_spmm_where_every_row_is_long(longest):
    """Rows of 600 values throughout, the longest at sixteen times the mean
    and one value above it (then a workgroup takes it): the oracle's bits."""
    rng = np.random.default_rng(83)
    lengths = np.full(3000, 600)
    lengths[1500] = longest
    lengths[:100] -= (longest - 600) // 100
    n_rows, n_cols = len(lengths), 2001
    assert lengths.sum() // n_rows == 600
    indices, indptr = _csr(rng, lengths, n_cols)
    data = _values(rng, indices.size, "float32")
    d, i, p = (to_torch(t, None, DEV) for t in (data, indices, indptr))
    plan = _capi.Plan(p, n_rows, indices.size, data=d, indices=i, n_cols=n_cols)
    assert plan.info().n_long_rows >= 2900
    for k in (1, 6, 32, 64):
        X = _values(rng, (n_cols, k), "float32")
        print(f"every row long {longest} k={k}", flush=True)
        got = _capi.spmm(d, i, p, to_torch(X, None, DEV), n_rows, n_cols, plan=plan)
        want = orc.csr_matmul(data, indices, indptr, X, n_rows, n_threads=8)
        assert to_numpy(got).tobytes() == want.tobytes(), k
    plan.close()


@pytest.mark.parametrize("k", [65535 * 64, 65535 * 64 + 1])
def test_spmm_long_row_with_more_column_tiles_than_a_grid_holds(k):
    """A long row at the last column count whose 64-column tiles fit a grid's
    y extent, and at the first that does not (small integers: exact)."""
    rng = np.random.default_rng(89)
    n_rows, n_cols = 40, 3
    lengths = np.zeros(n_rows, np.int64)
    lengths[[3, 7, 39]] = [600, 5, 1]
    indices, indptr = _csr(rng, lengths, n_cols)
    data = storage(rng.integers(-1, 2, indices.size).astype(np.float64), "float16")
    d, i, p = to_torch(data, "float16", DEV), to_torch(indices, None, DEV), to_torch(indptr, None, DEV)
    plan = _capi.Plan(p, n_rows, indices.size, data=d, indices=i, n_cols=n_cols)
    assert plan.info().n_long_rows == 1
    X = (torch.arange(n_cols * k, device=DEV) % 3 - 1).to(torch.float16).view(n_cols, k)
    dense = torch.zeros(n_rows, n_cols, device=DEV)
    rows = torch.repeat_interleave(torch.arange(n_rows, device=DEV), torch.from_numpy(lengths).to(DEV))
    dense.index_put_((rows, i.long()), d.float(), accumulate=True)
    print(f"spmm long row k={k}", flush=True)
    got = _capi.spmm(d, i, p, X, n_rows, n_cols, plan=plan)
    for r in (0, 3, 7, 39):
        want = (dense[r, :, None] * X.float()).sum(0)
        assert torch.equal(got[r].float(), want), r
    plan.close()


@pytest.mark.parametrize("vtype", VTYPES)
def test_spmm_rows_of_any_length_and_alignment(vtype):
    """Rows of X and Y that are no multiple of sixteen bytes, or start off
    one: every column equals the oracle's bit for bit and nothing is written
    past a row's end (rows of a wider buffer, first element skipped)."""
    rng = np.random.default_rng(47)
    lengths = rng.integers(0, 21, 700)
    lengths[[0, 1, 2, 3]] = [8, 9, 16, 17]
    n_rows, n_cols = len(lengths), 513
    indices, indptr = _csr(rng, lengths, n_cols)
    data = _values(rng, indices.size, vtype)
    d = to_torch(data, vtype, DEV)
    i, p = to_torch(indices, None, DEV), to_torch(indptr, None, DEV)
    for k in (1, 2, 3, 4, 5, 6, 7, 9, 12, 15, 20, 31, 33, 64, 100, 127, 257, 515):
        X = _values(rng, (n_cols, k), vtype)
        want = orc.csr_matmul(data, indices, indptr, X, n_rows, vtype=vtype)
        for pad, skip in ((0, 0), (3, 1)):
            wide = torch.zeros(n_cols, k + pad + skip, dtype=d.dtype, device=DEV)
            wide[:, skip:skip + k] = to_torch(X, vtype, DEV)
            out = torch.full((n_rows, k + pad + skip), 7, dtype=d.dtype, device=DEV)
            print(f"spmm ragged {vtype} k={k} pad={pad} skip={skip}", flush=True)
            _capi.spmm(d, i, p, wide[:, skip:skip + k], n_rows, n_cols, Y=out[:, skip:skip + k])
            got = out[:, skip:skip + k].contiguous()
            assert to_numpy(got).tobytes() == want.tobytes(), (k, pad)
            assert bool((out[:, :skip] == 7).all()) and bool((out[:, skip + k:] == 7).all())


@pytest.mark.parametrize("kind", ["short_rows", "banded_plan", "scattered"])
@pytest.mark.parametrize("vtype", VTYPES)
def test_spmm_ragged_rows_on_either_side_of_the_rule(kind, vtype):
    """Ragged and misaligned X rows where they are read sixteen bytes a lane
    (short rows; a plan with narrow column windows; 16-bit values) and where
    one column a lane: the oracle's bits, nothing written past a row's end."""
    rng = np.random.default_rng(71)
    n_rows, n_cols = 700, 40_000
    if kind == "short_rows":
        lengths = rng.integers(0, 13, n_rows)
    else:
        lengths = rng.integers(8, 21, n_rows)
    assert (lengths.sum() // n_rows < 8) == (kind == "short_rows")
    indices, indptr = _csr(rng, lengths, n_cols)
    if kind == "banded_plan":
        indices = (indices % 40 + np.repeat(np.arange(n_rows) * 50, lengths)).astype(np.int32)
    data = _values(rng, indices.size, vtype)
    d, i, p = to_torch(data, vtype, DEV), to_torch(indices, None, DEV), to_torch(indptr, None, DEV)
    plan = None
    if kind == "banded_plan":
        plan = _capi.Plan(p, n_rows, indices.size, data=d, indices=i, n_cols=n_cols)
        assert 0 < 4 * plan.info().window_rows <= n_cols
    for k in (2, 3, 4, 5, 7, 9, 13, 15, 17, 31, 33):
        X = _values(rng, (n_cols, k), vtype)
        want = orc.csr_matmul(data, indices, indptr, X, n_rows, vtype=vtype)
        print(f"spmm ragged {kind} {vtype} k={k}", flush=True)
        for pad, skip in ((0, 0), (2, 1)):
            wide = torch.zeros(n_cols, k + pad + skip, dtype=d.dtype, device=DEV)
            wide[:, skip:skip + k] = to_torch(X, vtype, DEV)
            out = torch.full((n_rows, k + pad + skip), 7, dtype=d.dtype, device=DEV)
            _capi.spmm(d, i, p, wide[:, skip:skip + k], n_rows, n_cols, plan=plan,
                       Y=out[:, skip:skip + k])
            got = out[:, skip:skip + k].contiguous()
            assert to_numpy(got).tobytes() == want.tobytes(), (k, pad)
            assert bool((out[:, :skip] == 7).all()) and bool((out[:, skip + k:] == 7).all())
    if plan is not None:
        plan.close()


@pytest.mark.parametrize("kind", ["one_row", "edges", "empty_runs", "skewed"])
@pytest.mark.parametrize("vtype", ["float32", "bfloat16", "complex64"])
def test_transposed_products_by_positions(kind, vtype):
    """The atomic transposed products on every row structure, k from 1 past a
    wave's lanes: small integers, so every order of additions is exact."""
    rng = np.random.default_rng(59)
    lengths = _row_lengths(kind, rng)
    n_rows, n_cols = len(lengths), 777
    index_dtype = np.int64 if kind == "edges" else np.int32
    indices, indptr = _csr(rng, lengths, n_cols, index_dtype, bad=0.02)
    small = lambda *shape: storage(rng.integers(-1, 2, shape).astype(np.float64), vtype)  # noqa: E731
    data = small(indices.size)
    good = (indices >= 0) & (indices < n_cols)
    held, cols = np.where(good, data, np.zeros_like(data)), np.where(good, indices, 0)
    d, i, p = to_torch(data, vtype, DEV), to_torch(indices, None, DEV), to_torch(indptr, None, DEV)
    for k in (0, 1, 2, 3, 5, 8, 33, 64, 70):
        X = small(n_rows, k) if k else small(n_rows)
        want = orc.csr_transpose_product(held, cols.astype(index_dtype), indptr, X, n_rows, n_cols,
                                         vtype=vtype)
        print(f"transposed products {kind} {vtype} k={k}", flush=True)
        f = _capi.spmm_transpose if k else _capi.spmv_transpose
        got = f(d, i, p, to_torch(X, vtype, DEV), n_rows, n_cols)
        np.testing.assert_array_equal(to_numpy(got), want)


@pytest.mark.parametrize("vtype", ["float32", "bfloat16", "complex64"])
def test_transposed_products_drop_columns_beyond_32_bits(vtype):
    """64-bit columns out of range whose low 32 bits are a valid column add
    nothing (small integers: every order of additions is exact)."""
    rng = np.random.default_rng(67)
    lengths = rng.integers(0, 12, 400)
    n_rows, n_cols = len(lengths), 777
    indices, indptr = _csr(rng, lengths, n_cols, np.int64)
    small = lambda *shape: storage(rng.integers(-1, 2, shape).astype(np.float64), vtype)  # noqa: E731
    data = small(indices.size)
    bad = rng.random(indices.size) < 0.2
    wide = indices + np.where(bad, rng.choice([-(1 << 31), -1, 1, 5], indices.size) << 32, 0)
    held = np.where(bad, np.zeros_like(data), data)
    d, i, p = to_torch(data, vtype, DEV), to_torch(wide, None, DEV), to_torch(indptr, None, DEV)
    for k in (0, 1, 4, 12, 20, 33, 64, 70, 130):  # every run of positions a wave takes
        X = small(n_rows, k) if k else small(n_rows)
        want = orc.csr_transpose_product(held, indices, indptr, X, n_rows, n_cols, vtype=vtype)
        print(f"columns beyond 32 bits {vtype} k={k}", flush=True)
        f = _capi.spmm_transpose if k else _capi.spmv_transpose
        got = f(d, i, p, to_torch(X, vtype, DEV), n_rows, n_cols)
        np.testing.assert_array_equal(to_numpy(got), want)


@pytest.mark.parametrize("solver", ["cg", "pcg", "minres", "bicgstab"])
@pytest.mark.parametrize("rows", [1, 2, 513, 1500, 2048, 2049, 4608])
def test_small_systems_in_one_workgroup(solver, rows):
    """Solves of small systems of up to about nine values a row, in one
    workgroup and in a kernel a pass (the limits: the next test), both index
    types and a budget that ends inside a launch: status and iterations as
    the oracle's, x within the tolerance's bound of the float64 solution
    (condition number at most 5)."""
    rng = np.random.default_rng(rows)
    dense = {}
    for i in range(rows):
        for j in rng.integers(0, rows, 4):
            if i != j:
                v = rng.uniform(-0.2, 0.2)
                dense[i, int(j)] = dense.get((i, int(j)), 0.0) + v
                if solver != "bicgstab":
                    dense[int(j), i] = dense[i, int(j)]
    near = np.zeros(rows)
    for (i, _), v in dense.items():
        near[i] += abs(v)
    for i in range(rows):
        dense[i, i] = 2.0 * max(near.max(), 0.5)
    keys = np.array(sorted(dense))
    data = np.array([dense[tuple(k)] for k in keys], np.float32)
    index_dtype = np.int64 if rows % 2 else np.int32
    indices = keys[:, 1].astype(index_dtype)
    indptr = np.searchsorted(keys[:, 0], np.arange(rows + 1)).astype(index_dtype)
    b = rng.standard_normal(rows).astype(np.float32)
    from scipy import sparse
    from scipy.sparse.linalg import spsolve
    exact = spsolve(sparse.csc_matrix((data.astype(np.float64), (keys[:, 0], keys[:, 1])),
                                      shape=(rows, rows)), b.astype(np.float64))
    d, i, p = (to_torch(t, None, DEV) for t in (data, indices, indptr))
    plan = _capi.Plan(p, rows, data.size, data=d, indices=i, n_cols=rows)
    bt, inv = to_torch(b, None, DEV), 1.0 / data[keys[:, 0] == keys[:, 1]]
    print(f"one workgroup {solver} {rows}", flush=True)
    for budget in (200, 2):
        if solver in ("cg", "pcg"):
            jac = to_torch(inv.astype(np.float32), None, DEV) if solver == "pcg" else None
            x, info, res, its = _capi.cg(d, i, p, bt, rtol=1e-5, maxiter=budget, plan=plan,
                                         inv_diag=jac)
            want = (orc.csr_pcg_jacobi(data, indices, indptr, b, inv.astype(np.float32), rtol=1e-5,
                                       maxiter=budget) if jac is not None else
                    orc.csr_cg(data, indices, indptr, b, rtol=1e-5, maxiter=budget))
        else:
            x, info, res, its = _capi.krylov(solver, d, i, p, bt, rtol=1e-5, maxiter=budget,
                                             plan=plan)
            f = orc.csr_minres if solver == "minres" else orc.csr_bicgstab
            want = f(data, indices, indptr, b, rtol=1e-5, maxiter=budget)
        assert info == want[1] and abs(its - want[3]) <= 1, (info, its, want[1:])
        if info == 0:
            # |x - exact| <= cond * rtol * |x|, cond <= (2 + 1) / (2 - 1) of the row sums' bound
            assert np.linalg.norm(to_numpy(x) - exact) <= 5e-5 * np.linalg.norm(exact)
    plan.close()


def _system(n, values, longest=None):
    """A symmetric diagonally dominant n x n system of exactly `values` stored
    values in rows of about the same length, as (data, indices, indptr, rows);
    with `longest`, row 0 has that many (diagonal entries split)."""
    rng = np.random.default_rng(n + values)
    pairs = (values - n) // 2
    i = np.arange(pairs) % n
    j = (i + 1 + np.arange(pairs) // n) % n
    v = rng.uniform(-0.2, 0.2, pairs)
    near = np.zeros(n)
    np.add.at(near, np.concatenate([i, j]), np.abs(np.concatenate([v, v])))
    diagonal = np.full(n, 2.0 * max(near.max(), 0.5))
    rows = np.concatenate([i, j, np.arange(n)])
    cols = np.concatenate([j, i, np.arange(n)])
    data = np.concatenate([v, v, diagonal])
    extra = values - rows.size if longest is None else longest - int((rows == 0).sum())
    assert extra >= 0
    if extra:  # row 0's diagonal entry in 1 + extra parts
        data[2 * pairs] /= 1 + extra
        rows, cols = np.append(rows, np.zeros(extra, int)), np.append(cols, np.zeros(extra, int))
        data = np.append(data, np.full(extra, data[2 * pairs]))
    order = np.lexsort((cols, rows))
    index_dtype = np.int64 if n % 2 else np.int32
    rows = rows[order]
    return (data[order].astype(np.float32), cols[order].astype(index_dtype),
            np.searchsorted(rows, np.arange(n + 1)).astype(index_dtype), rows)


@pytest.mark.parametrize("solver,rows,values,longest,inside", [
    case for solvers, cases in (
        (("cg", "pcg"), [(4608, 24576, None, True), (4608, 24577, None, False),
                         (4609, 24000, None, False), (2000, 24576, None, True),
                         (300, 8700, 32, True), (300, 8700, 33, False)]),
        (("minres", "minres_jacobi"), [(4608, 8192, None, True), (4608, 8193, None, False),
                                       (4609, 8000, None, False), (513, 8192, None, True),
                                       (250, 7250, 32, True), (250, 7250, 33, False)]),
        (("bicgstab", "bicgstab_jacobi"), [(2048, 8192, None, True), (2048, 8193, None, False),
                                           (2049, 8000, None, False), (513, 8192, None, True),
                                           (250, 7250, 32, True), (250, 7250, 33, False)]))
    for s in solvers for case in [(s, *c) for c in cases]])
def test_one_workgroup_solves_at_their_limits(solver, rows, values, longest, inside):
    """Systems at the most rows, values and values a row that a solver's
    one-workgroup loop takes, and one beyond each: the loop runs where it
    should, the status and (to one) the iterations are the oracle's, x within
    the tolerance's bound of the float64 solution (condition number at most
    5), also on a budget that ends inside a launch."""
    data, indices, indptr, row_of = _system(rows, values, longest)
    assert longest is not None or data.size == values
    assert longest is None or np.diff(indptr).max() == longest
    b = np.random.default_rng(rows).standard_normal(rows).astype(np.float32)
    from scipy import sparse
    from scipy.sparse.linalg import spsolve

    m = sparse.csc_matrix((data.astype(np.float64), (row_of, indices)), shape=(rows, rows))
    exact = spsolve(m, b.astype(np.float64))
    inv = (1.0 / m.diagonal()).astype(np.float32)
    d, i, p = (to_torch(t, None, DEV) for t in (data, indices, indptr))
    plan = _capi.Plan(p, rows, data.size, data=d, indices=i, n_cols=rows)
    kind = solver.replace("_jacobi", "").replace("pcg", "cg")
    assert _capi.one_workgroup(kind, plan) == inside
    jacobi = solver != kind
    bt, jac = to_torch(b, None, DEV), to_torch(inv, None, DEV) if jacobi else None
    print(f"limits {solver} {rows} {values} {longest}", flush=True)
    for budget in (200, 2):
        f = getattr(orc, {"cg": "csr_cg", "pcg": "csr_pcg_jacobi"}.get(solver, f"csr_{solver}"))
        pre = (inv,) if jacobi else ()
        want = f(data, indices, indptr, b, *pre, rtol=1e-5, maxiter=budget)
        if kind == "cg":
            x, info, _, its = _capi.cg(d, i, p, bt, rtol=1e-5, maxiter=budget, plan=plan,
                                       inv_diag=jac)
        else:
            x, info, _, its = _capi.krylov(kind, d, i, p, bt, rtol=1e-5, maxiter=budget, plan=plan,
                                           inv_diag=jac)
        assert info == want[1] and abs(its - want[3]) <= 1, (info, its, want[1:])
        if info == 0:
            assert np.linalg.norm(to_numpy(x) - exact) <= 5e-5 * np.linalg.norm(exact)
    plan.close()
