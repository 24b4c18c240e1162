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
