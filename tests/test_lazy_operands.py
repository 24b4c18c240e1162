"""Operands that torch keeps as a flag on another tensor's memory (conjugates,
some negations) count with the values they stand for."""

from __future__ import annotations

import pytest
import torch

import mlx_sparse as ms


@pytest.fixture(params=["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def device(request):
    ms.use_cpu() if request.param == "cpu" else ms.use_gpu()
    yield request.param
    if torch.cuda.is_available():
        ms.use_gpu()


def _ops(a):
    n = a.shape[0]
    return [
        lambda v: a @ v,
        lambda v: a @ torch.stack([v, 2 * v], 1),
        lambda v: ms.csr_batched_matvec(a, v.reshape(1, n)),
        lambda v: ms.csr_batched_matmul(a, v.reshape(1, n, 1)),
        lambda v: ms.csr_matvec_transpose(a, v),
        lambda v: ms.csr_matmul_transpose(a, v[:, None]),
    ]


@pytest.mark.parametrize("lazy", ["operand", "values", "both"])
def test_conjugates(device, lazy):
    gen = torch.Generator().manual_seed(3)
    n, nnz = 40, 130
    data = torch.randn(nnz, generator=gen, dtype=torch.complex64).to(device)
    x = torch.randn(n, generator=gen, dtype=torch.complex64).to(device)
    indices = torch.randint(n, (nnz,), generator=gen, dtype=torch.int32).to(device)
    indptr = torch.linspace(0, nnz, n + 1).to(torch.int32).to(device)
    d = data.conj() if lazy != "operand" else data
    v = x.conj() if lazy != "values" else x
    assert d.is_conj() or v.is_conj()
    a = ms.csr_array((d, indices, indptr), shape=(n, n))
    plain = ms.csr_array((d.resolve_conj(), indices, indptr), shape=(n, n))
    for f, g in zip(_ops(a), _ops(plain)):
        torch.testing.assert_close(f(v), g(v.resolve_conj()), rtol=1e-6, atol=1e-6)
    for other, want in ((a.T, plain.T), (a.H, plain.H), (a.conj(), plain.conj())):
        torch.testing.assert_close(other @ v, want @ v.resolve_conj(), rtol=1e-6, atol=1e-6)


def test_negations(device):
    gen = torch.Generator().manual_seed(5)
    n, nnz = 40, 130
    data = torch.randn(nnz, generator=gen).to(device)
    x = torch._neg_view(torch.randn(n, generator=gen).to(device))
    assert x.is_neg()
    indices = torch.randint(n, (nnz,), generator=gen, dtype=torch.int32).to(device)
    indptr = torch.linspace(0, nnz, n + 1).to(torch.int32).to(device)
    for d in (data, torch._neg_view(data)):
        a = ms.csr_array((d, indices, indptr), shape=(n, n))
        plain = ms.csr_array((d.resolve_neg(), indices, indptr), shape=(n, n))
        for f, g in zip(_ops(a), _ops(plain)):
            torch.testing.assert_close(f(x), g(x.resolve_neg()), rtol=1e-6, atol=1e-6)
