"""One matrix used from several streams and threads at once: the cached plan is
shared, the scratch of a product or a solve is not."""

from __future__ import annotations

import threading

import numpy as np
import pytest
import torch

import mlx_sparse as ms
from mlx_sparse import linalg, runtime

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.fixture(autouse=True)
def on_the_gpu():
    ms.use_gpu()


def _matrix(rng, lengths, n_cols):
    indptr = np.zeros(len(lengths) + 1, np.int32)
    np.cumsum(lengths, out=indptr[1:])
    nnz = int(indptr[-1])
    # small integers: every order of additions is exact
    data = torch.from_numpy(rng.integers(-2, 3, nnz).astype(np.float32)).to(DEV)
    indices = torch.from_numpy(rng.integers(0, n_cols, nnz).astype(np.int32)).to(DEV)
    return ms.csr_array((data, indices, torch.from_numpy(indptr).to(DEV)),
                        shape=(len(lengths), n_cols))


@pytest.mark.parametrize("mode,long_rows", [
    ("panels", False), ("panels", True), ("on", False), ("off", True)])
def test_products_and_value_gradients_on_two_streams(mode, long_rows):
    rng = np.random.default_rng(71)
    n_rows, n_cols = 400_000, 300_000
    lengths = rng.integers(2, 12, n_rows)
    if long_rows:
        lengths[[0, 1000, n_rows - 1]] = [60_000, 20_000, 9_000]
    a = _matrix(rng, lengths, n_cols)
    with runtime.context("gpu_slice", mode):
        info = a.plan().info()
    assert (info["n_panels"] > 0) == (mode == "panels") and (info["n_slices"] > 0) == (mode == "on")
    xs = [torch.from_numpy(rng.integers(-2, 3, n_cols).astype(np.float32)).to(DEV) for _ in range(2)]
    g = torch.from_numpy(rng.integers(-2, 3, n_rows).astype(np.float32)).to(DEV)
    wide = torch.repeat_interleave(torch.arange(n_rows, device=DEV),
                                   torch.from_numpy(lengths).to(DEV))
    want = [torch.zeros(n_rows, device=DEV, dtype=torch.float64).index_add_(
        0, wide, (a.data * x[a.indices.long()]).double()).float() for x in xs]
    want_g = [g[wide] * x[a.indices.long()] for x in xs]
    streams = [torch.cuda.Stream() for _ in range(2)]
    a.data.requires_grad_(True)
    torch.cuda.synchronize()
    print(f"two streams {mode} long={long_rows}", flush=True)
    got, grads = [[], []], [[], []]
    for _ in range(12):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                y = a @ xs[i]
                got[i].append(y.detach())
                grads[i].append(torch.autograd.grad(y, a.data, g)[0])
    torch.cuda.synchronize()
    for i in range(2):
        assert all(torch.equal(y, want[i]) for y in got[i])
        assert all(torch.equal(d, want_g[i]) for d in grads[i])


@pytest.mark.parametrize("mode", ["panels", "on", "off"])
def test_new_values_reach_a_product_on_another_stream(mode):
    """The values change on one stream; a product on another that waits for
    that change, and no more, uses them also where the copy that the plan
    holds is rewritten later, in the first stream's own time."""
    rng = np.random.default_rng(79)
    a = _matrix(rng, rng.integers(2, 12, 40_000), 30_000)
    with runtime.context("gpu_slice", mode):
        a.plan()
    x = torch.from_numpy(rng.integers(-2, 3, 30_000).astype(np.float32)).to(DEV)
    first, second = torch.cuda.Stream(), torch.cuda.Stream()
    old = a @ x
    torch.cuda.synchronize()
    print(f"new values {mode}", flush=True)
    for _ in range(3):
        old = 2 * old
        changed = torch.cuda.Event()
        with torch.cuda.stream(first):
            a.data.mul_(2)
            changed.record()
            torch.cuda._sleep(20_000_000)  # about 10 ms before the copy is rewritten
            y1 = a @ x
        with torch.cuda.stream(second):
            second.wait_event(changed)
            y2 = a @ x
        torch.cuda.synchronize()
        assert torch.equal(y1, old) and torch.equal(y2, old)


def test_solves_in_two_threads():
    rng = np.random.default_rng(73)
    n, per = 60_000, 6
    r = np.repeat(np.arange(n), per)
    c = rng.integers(0, n, n * per)
    from scipy import sparse

    m = sparse.coo_matrix((rng.uniform(-0.1, 0.1, n * per), (r, c)), shape=(n, n))
    m = (m + m.T + 4.0 * sparse.identity(n)).tocsr().astype(np.float32)
    a = ms.csr_array(tuple(torch.from_numpy(t).to(DEV) for t in (m.data, m.indices, m.indptr)),
                     shape=(n, n))
    with runtime.context("gpu_slice", "panels"):
        assert a.plan().info()["n_panels"] > 0
    bs = [torch.from_numpy(rng.standard_normal(n).astype(np.float32)).to(DEV) for _ in range(2)]
    alone = [linalg.cg(a, b, rtol=1e-6) for b in bs]
    torch.cuda.synchronize()
    print("two threads", flush=True)
    out = [[], []]

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(4):
                out[i].append(linalg.cg(a, bs[i], rtol=1e-6))
            torch.cuda.current_stream().synchronize()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i in range(2):
        for x, info in out[i]:
            assert int(info) == int(alone[i][1]) and torch.equal(x, alone[i][0])
