"""Calls in rounds whose bounds of tiles take more than their room come in parts of their queries: the same ids and distances, to the bit, whether
the last part is as large as the others, a single query, or every query is a part of its own, and where no room is enough for one.  (The
batch kernel's calls stay whole.)"""
import pytest
import torch

from test_gpu_rounds import ALWAYS, NEVER, _ask, _count_items, _rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("parts", [2, 3, 7, 50, 99, 10 ** 6])
@pytest.mark.parametrize("shape", [(20000, 64, 2, 7, 50, 10, 10, 5000, 99), (24001, 40, 2, 6, 48, 4, 4, 2000, 99), (36000, 48, 2, 15, 60, 128, 30, 10, 99)],
                         ids=["dense", "batch", "wide"])
def test_same_as_whole(gpu, shape, parts):
    from dciknn_cuda_amd import _capi
    n, dim, M, L, B, T, k, outer, nq = shape
    X, Q = _rows("clusters", n, nq, dim, 5)
    dci = gpu.DCI(dim, M, L, B, T, seed=3)
    dci.add(X)
    want = _ask(dci, dci._lib, NEVER, Q, k, outer)
    # (tiles of 64 or 128 rows, partitions padded to whole ones of up to 512 rows: between n / 128 and that of them)
    tiles = B * (((n + B - 1) // B + 511) // 512 * 512 // 64)
    _capi.check(dci._lib.dcih_debug_near_room(dci._dci_inst, max(1, tiles * nq * 4 // (2 * parts))))
    items = _count_items(dci)
    for again in range(2):
        got = _ask(dci, dci._lib, ALWAYS, Q, k, outer)
        assert torch.equal(got[0], want[0]), again
        assert torch.equal(got[1].view(torch.int32), want[1].view(torch.int32)), again
    if parts == 50 and T != 4:      # the last part is four queries at most; all of them take ten partitions and more each
        assert 0 < int(items[:4].sum()) <= 4 * B, items
    dci.free()


@pytest.mark.parametrize("float_ids", [False, True])
@pytest.mark.parametrize("parts", [2, 5, 250])
def test_chosen_by_itself(gpu, parts, float_ids):
    """Left to choose, a call comes in parts as long as these are calls in rounds with bounds of tiles themselves; else it goes in rounds as a whole,
    without those bounds."""
    from dciknn_cuda_amd import _capi
    from test_gpu_rounds import _route
    from test_gpu_steering import _plan
    n, dim, B, nq, k = 200_000, 64, 100, 2000, 10
    X, Q = _rows("clusters", n, nq, dim, 5)
    dci = gpu.DCI(dim, 2, 7, B, 10, seed=3)
    dci.add(X)
    want = _ask(dci, dci._lib, NEVER, Q, k, 5000)
    _capi.check(dci._lib.dcih_set_option(dci._dci_inst, _capi.OPT_ROUNDS, 0))
    dci.query(Q, k, 5000)
    assert _route(dci)[0] >= 2 and _route(dci)[1] == 1 and _plan(dci)[1] == 1
    # (partitions of 2000 rows, tiles of 128, whole ones of up to 512 rows)
    _capi.check(dci._lib.dcih_debug_near_room(dci._dci_inst, B * 16 * nq * 4 // parts))
    for again in range(2):
        ids, dists = dci.query(Q, k, 5000, return_int=not float_ids)
        assert _route(dci)[0] >= 2 and _route(dci)[1] == (parts < 250) and (_plan(dci)[1] > 1) == (parts < 250)
        assert torch.equal(ids.int(), want[0]) and torch.equal(dists, want[1]), again
    dci.free()


def test_in_a_graph(gpu):
    """Parts are recorded like any other call: after one that has taken the room, and replayed on other queries in the same buffer."""
    from dciknn_cuda_amd import _capi
    from test_gpu_rounds import _route
    from test_gpu_steering import _plan
    n, dim, B, T, nq, k, outer, parts = 30_000, 24, 12, 10, 400, 5, 500, 3
    X, Q = _rows("clusters", n, 2 * nq, dim, 9)
    dci = gpu.DCI(dim, 2, 7, B, T, seed=3)
    dci.add(X)
    want = [_ask(dci, dci._lib, NEVER, q, k, outer) for q in (Q[:nq], Q[nq:])]
    _capi.check(dci._lib.dcih_set_option(dci._dci_inst, _capi.OPT_ROUNDS, ALWAYS))
    _capi.check(dci._lib.dcih_debug_near_room(dci._dci_inst, B * 40 * nq * 4 // parts))      # (tiles of 64 rows)
    q = Q[:nq].clone()
    ids = torch.empty((nq, k), dtype=torch.int32, device="cuda")
    dists = torch.empty((nq, k), dtype=torch.float32, device="cuda")

    def call(stream):
        _capi.check(dci._lib.dcih_query(dci._dci_inst, dim, nq, q.data_ptr(), k, 0, outer, 10 * k, B, T, ids.data_ptr(), dists.data_ptr(), None, stream))
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    call(s.cuda_stream)
    s.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        call(torch.cuda.current_stream().cuda_stream)
    assert _route(dci)[0] >= 2 and _route(dci)[1] == 1 and _plan(dci)[1] >= 2
    for turn in (0, 1, 0, 1):
        q.copy_(Q[turn * nq:(turn + 1) * nq])
        ids.fill_(-5)
        dists.fill_(-5.0)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(ids, want[turn][0]) and torch.equal(dists, want[turn][1]), turn
        call(0)                                # eager work between the replays
        torch.cuda.synchronize()
        assert torch.equal(ids, want[turn][0]) and torch.equal(dists, want[turn][1]), turn
    del g
    dci.free()
