"""Panels that only many products repay: they wait for those, and until then -
and where torch does not count what is written to the values, or a graph
replays a product - the values are read as they are."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import _capi
import mlx_sparse as ms
from mlx_sparse import _csr

pytestmark = pytest.mark.gpu

DEV = "cuda"
N_ROWS, N_COLS, VALUES = 400_000, (4 << 20) // 4, 5 << 20  # the smallest that take panels


@pytest.fixture(autouse=True)
def on_the_gpu():
    ms.use_gpu()


@pytest.fixture(scope="module")
def buffers():
    rng = np.random.default_rng(83)
    indptr = np.zeros(N_ROWS + 1, np.int32)
    np.cumsum(rng.multinomial(VALUES, np.ones(N_ROWS) / N_ROWS), out=indptr[1:])
    # small integers: every order of additions is exact
    data = rng.integers(-2, 3, VALUES).astype(np.float32)
    indices = rng.integers(0, N_COLS, VALUES).astype(np.int32)
    return tuple(torch.from_numpy(t).to(DEV) for t in (data, indices, indptr))


def _array(buffers):
    data, indices, indptr = buffers
    return ms.csr_array((data.clone(), indices, indptr), shape=(N_ROWS, N_COLS))


def _want(a, x):
    rows = torch.repeat_interleave(torch.arange(N_ROWS, device=DEV), a.indptr.diff())
    out = torch.zeros(N_ROWS, dtype=torch.float64, device=DEV)
    return out.index_add_(0, rows, (a.data.detach() * x[a.indices]).double()).float()


def _panels(a):
    return a._cache[("plan", "cuda:0")][1].info()["n_panels"]


def _x(seed=1):
    rng = np.random.default_rng(seed)
    return torch.from_numpy(rng.integers(-2, 3, N_COLS).astype(np.float32)).to(DEV)


def test_panels_wait_for_the_products_that_repay_them(buffers):
    a, x = _array(buffers), _x()
    want = _want(a, x)
    print("late panels", flush=True)
    for _ in range(3):  # products with a matrix do not use them
        a @ x[:, None]
    for i in range(_csr._REPAID):
        assert torch.equal(a @ x, want)
        assert _panels(a) == 0, i
    assert torch.equal(a @ x, want) and _panels(a) > 0
    assert a.T._cache["kept"]  # used as often
    b = _array(buffers)
    b.plan()
    assert _panels(b) > 0 and torch.equal(b @ x, want)
    b.data.mul_(2)
    assert torch.equal(b @ x, 2 * want)


@pytest.mark.parametrize("planned", [False, True])
def test_uncounted_values_are_read_as_they_are(buffers, planned):
    x = _x()
    print(f"inference values planned={planned}", flush=True)
    with torch.inference_mode():
        a = _array(buffers)
        want = _want(a, x)
        if planned:
            a.plan()
        for _ in range(_csr._REPAID + 2):
            y = a @ x
        assert torch.equal(y, want)
        a.data.mul_(2)
        assert torch.equal(a @ x, 2 * want)


@pytest.mark.parametrize("long_rows", [False, True])
def test_replayed_products_read_the_values_as_they_are(buffers, long_rows):
    data, indices, indptr = buffers
    if long_rows:
        indptr = indptr.clone()
        indptr[1:1001] = indptr[1000].item()  # row 0 takes the values of the next 999
    a, x = _array((data, indices, indptr)), _x()
    a.plan()
    assert _panels(a) > 0
    want = _want(a, x)
    a @ x
    torch.cuda.synchronize()
    alone = torch.cuda.CUDAGraph()
    with torch.cuda.graph(alone):
        y = a @ x
    new = a.data.clone()
    step = torch.cuda.CUDAGraph()
    with torch.cuda.graph(step):
        a.data.copy_(new)
        z = a @ x
    print("replays", flush=True)
    for i in range(1, 4):
        new.mul_(2)
        want = 2 * want
        step.replay()
        torch.cuda.synchronize()
        assert torch.equal(z, want), i
        alone.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want), i
        assert torch.equal(a @ x, want), i
        a.data.mul_(-1)
        alone.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, -want) and torch.equal(a @ x, -want), i


@pytest.mark.parametrize("long_rows", [False, True])
def test_a_copy_that_cannot_be_allocated_leaves_row_blocks(buffers, long_rows):
    """Whichever allocation of a panel build fails (injected on the host), AUTO
    ends with row blocks that multiply and forced panels with MemoryError; the
    scratch block alone can be done without."""
    data, indices, indptr = buffers
    if long_rows:
        indptr = indptr.clone()
        indptr[1:1001] = indptr[1000].item()  # row 0 takes the values of the next 999
    want = _want(ms.csr_array((data, indices, indptr), shape=(N_ROWS, N_COLS)), _x())
    fail = _capi.lib().msx_test_panel_alloc_failure
    fatal = {1, 3, 4} if long_rows else {1, 2}
    try:
        for after in range(6 if long_rows else 4):
            print(f"allocation {after} fails long={long_rows}", flush=True)
            fail(after)
            plan = _capi.Plan(indptr, N_ROWS, VALUES, data=data, indices=indices, n_cols=N_COLS)
            assert (plan.info().n_panels == 0) == (after in fatal), after
            assert plan.info().n_panels or plan.info().panel_bytes == 0
            y = _capi.spmv(data, indices, indptr, _x(), N_ROWS, N_COLS, plan)
            assert torch.equal(y, want), after
            plan.close()
            if after in fatal:
                fail(after)
                with pytest.raises((MemoryError, RuntimeError), match="allocation"):
                    _capi.Plan(indptr, N_ROWS, VALUES, data=data, indices=indices, n_cols=N_COLS,
                               slice_mode=_capi.SLICE_PANELS)
    finally:
        fail(-1)


@pytest.mark.parametrize("long_rows", [False, True])
@pytest.mark.parametrize("stream_ordered", [True, False])
def test_products_without_room_for_the_copys_scratch(buffers, long_rows, stream_ordered):
    """torch may not allocate the scratch of a panel product or gradient: it
    comes from the stream-ordered allocator, and where that fails too
    (injected) the product runs over the plan's row blocks and the gradient
    without the panels."""
    data, indices, indptr = buffers
    if long_rows:
        indptr = indptr.clone()
        indptr[1:1001] = indptr[1000].item()
    a, x = _array((data, indices, indptr)), _x()
    a.plan()
    assert _panels(a) > 0
    a.data.requires_grad_(True)
    want, g = _want(a, x), torch.ones(N_ROWS, device=DEV)
    y = a @ x
    fail = _capi.lib().msx_test_panel_alloc_failure
    total = torch.cuda.mem_get_info()[1]
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    print(f"no room long={long_rows} stream ordered={stream_ordered}", flush=True)

    def leave(spare):
        """torch may allocate `spare` bytes more in one piece, and no second scratch."""
        room = torch.empty(spare, dtype=torch.uint8, device=DEV)
        torch.cuda.set_per_process_memory_fraction(torch.cuda.memory_reserved() / total)
        full = []
        with pytest.raises(torch.OutOfMemoryError):
            while True:
                full.append(torch.empty(VALUES, device=DEV))
        del room
        return full

    try:
        full = leave(8 << 20)  # the product's result
        fail(-1 if stream_ordered else 0)
        with torch.no_grad():
            got = a @ x
        torch.cuda.set_per_process_memory_fraction(1.0)
        del full
        assert torch.equal(got, want)
        full = leave(22 << 20)  # the gradient
        fail(-1 if stream_ordered else 0)
        d, = torch.autograd.grad(y, a.data, g)
        del full
    finally:
        fail(-1)
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.equal(d, x[a.indices])
