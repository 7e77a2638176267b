"""What a handle keeps from one call to the next, over streams and graphs: clear while queries are
under way and what comes after it on the same stream, another one, with new directions or by `add`;
a first query that is recorded and not run."""
import threading

import numpy as np
import pytest
import torch

from util import engine_index

pytestmark = pytest.mark.gpu

DIM, M, L, B, T, K, OUTER = 64, 2, 7, 40, 10, 10, 2000
PER_THREAD = 2          # hipStreamPerThread


def _rows(seed, n):
    return torch.randn(n, DIM, generator=torch.Generator().manual_seed(seed)).cuda()


def _query(dci, Q, stream, nn, dists):
    from dciknn_cuda_amd import _capi
    _capi.check(dci._lib.dcih_query(dci._dci_inst, DIM, Q.shape[0], Q.data_ptr(), K, 0, OUTER, 10 * K, B, T,
                                    nn.data_ptr(), dists.data_ptr(), None, stream))


def _append(dci, X, stream):
    from dciknn_cuda_amd import _capi
    _capi.check(dci._lib.dcih_append(dci._dci_inst, DIM, X.shape[0], X.data_ptr(), B, T, stream))
    dci.num_points += X.shape[0]


def _out(Q):
    return (torch.full((Q.shape[0], K), -7, dtype=torch.int32, device="cuda"),
            torch.full((Q.shape[0], K), -7.0, device="cuda"))


def _same(a, b):
    return all(torch.equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("then", ["same stream", "other stream", "per-thread stream", "new directions", "add", "reset", "after a graph"])
def test_clear_while_a_query_is_under_way(gpu, then):
    X1, X2, Q = _rows(1, 200_000), _rows(2, 200_000), _rows(3, 2000)
    one, two = gpu.DCI(DIM, M, L, B, T, seed=7), gpu.DCI(DIM, M, L, B, T, seed=7)
    other_dirs = gpu.DCI(DIM, M, L, B, T, seed=8).directions
    one.add(X1)
    if then == "new directions":
        two.directions = other_dirs
    want1, want2 = _out(Q), _out(Q)
    _query(one, Q, 0, *want1)
    torch.cuda.synchronize()
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    first = PER_THREAD if then == "per-thread stream" else a.cuda_stream
    second = {"other stream": b.cuda_stream, "per-thread stream": PER_THREAD}.get(then, a.cuda_stream)
    dci = gpu.DCI(DIM, M, L, B, T, seed=7)
    _append(dci, X1, first)
    _query(dci, Q, first, *_out(Q))           # (the workspace has its size now)
    got1, got2 = _out(Q), _out(Q)
    torch.cuda.synchronize()

    begun, over = threading.Event(), threading.Event()
    graph = torch.cuda.CUDAGraph() if then == "after a graph" else None
    if graph is not None:
        with torch.cuda.graph(graph, stream=a):
            _query(dci, Q, torch.cuda.current_stream().cuda_stream, *got1)

    def begin():
        for _ in range(8):                    # (milliseconds of work)
            if graph is not None:
                with torch.cuda.stream(a):
                    graph.replay()
            else:
                _query(dci, Q, first, *got1)
        begun.set()
        over.wait(60)                         # (a thread's own stream lives as long as the thread)

    def go_on():
        if then == "reset":
            dci.reset()
            two.directions = dci.directions
        else:
            dci.clear()
        if then == "new directions":
            dci.directions = other_dirs
        if then == "add":
            with torch.cuda.stream(a):
                dci.add(X2)
        else:
            _append(dci, X2, second)
        _query(dci, Q, second, *got2)

    t = threading.Thread(target=begin)        # (another thread: so is its per-thread stream)
    t.start()
    assert begun.wait(60)
    go_on()
    torch.cuda.synchronize()
    over.set()
    t.join()
    two.add(X2)
    _query(two, Q, 0, *want2)
    torch.cuda.synchronize()
    del graph
    assert _same(got1, want1)
    assert _same(got2, want2)
    keys, ids = engine_index(dci)
    keys2, ids2 = engine_index(two)
    np.testing.assert_array_equal(keys, keys2)
    np.testing.assert_array_equal(ids, ids2)
    for d in (one, two, dci):
        d.free()


def test_first_batch_traversal_recorded(gpu):
    """The table of positions that the batch kernel reads is filled by the first call that uses it: a call
    that is only recorded fills it when its graph runs, so an eager call before that fills it as well."""
    X, Q = _rows(5, 100_000), _rows(6, 64)
    step = gpu.DCI(DIM, M, L, B, T, seed=7, traversal="step")
    step.add(X)
    dci = gpu.DCI(DIM, M, L, B, T, seed=7, traversal="step")
    dci.add(X)
    want = _out(Q)
    _query(step, Q, 0, *want)
    _query(dci, Q, 0, *_out(Q))               # (the workspace has its size now)
    torch.cuda.synchronize()
    dci.set_traversal("batch")
    s, recorded, eager = torch.cuda.Stream(), _out(Q), _out(Q)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        _query(dci, Q, torch.cuda.current_stream().cuda_stream, *recorded)
    _query(dci, Q, 0, *eager)
    torch.cuda.synchronize()
    assert _same(eager, want)
    for _ in range(3):
        for out in recorded:
            out.fill_(-5)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert _same(recorded, want)
        _query(dci, Q, 0, *eager)
        torch.cuda.synchronize()
        assert _same(eager, want)
    del g
    dci.free()
    step.free()
