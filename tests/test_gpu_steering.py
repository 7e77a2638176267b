"""What a handle remembers of its calls to choose the way of the next ones.  (It never shows in results; other tests compare the ways.)"""
import pytest
import torch

from test_gpu_confirm import _confirmed
from test_gpu_rounds import _route, _rows

pytestmark = pytest.mark.gpu


def _plan(dci):
    """(near rows looked at alone first, parts, launches by windows' first lanes) of the last call."""
    from dciknn_cuda_amd import _capi
    plan = (_capi.ctypes.c_int64 * 3)()
    _capi.check(dci._lib.dcih_debug_plan(dci._dci_inst, plan))
    return tuple(plan)


# Rows of which half of the partitions are needed and too many of each are near: items have to be left to the traversals
N, DIM, M, L, B, T, K, OUTER, QUERIES = 123457, 67, 3, 5, 37, 3, 7, 1000, 1000


@pytest.fixture()
def of_no_use(gpu):
    """A handle on whose calls near rows alone have just been of no use, its rows and queries."""
    X, Q = _rows("normal", N, QUERIES, DIM, 5)
    dci = gpu.DCI(DIM, M, L, B, T, seed=3)
    dci.add(X)
    dci.query(Q, K, OUTER, return_int=True)
    assert _route(dci)[0] >= 2 and _plan(dci)[0] == 1
    torch.cuda.synchronize()
    dci.query(Q, K, OUTER, return_int=True)
    assert _route(dci)[0] >= 2 and _plan(dci)[0] == 0
    yield dci, X, Q
    dci.free()


def test_near_rows_are_tried_again_whatever_comes_between(of_no_use):
    dci, _, Q = of_no_use
    for call in range(300):
        dci.query(Q, K, OUTER, return_int=True)
        if _plan(dci)[0]:
            break
        dci.query(Q[:1], K, OUTER, return_int=True)      # traversed whole
        assert _route(dci)[0] == 0
    assert 200 < call < 256
    # (a few items ahead of the others, up to 64 a die, and no more of them: the others go to the traversals at once)
    torch.cuda.synchronize()
    answered, left = _confirmed(dci)
    assert answered == 0 and 17 < left <= 17 + 64 * 8


@pytest.mark.parametrize("other", ["results", "steps", "rows", "appended rows"])
def test_what_near_rows_were_no_use_for_says_nothing_of_other_calls(of_no_use, other):
    dci, X, Q = of_no_use
    if other in ("rows", "appended rows"):
        dci.clear()
        if other == "rows":
            dci.add(X)
        else:
            dci.append(X)
    k, outer = K + (other == "results"), OUTER - 100 * (other == "steps")
    dci.query(Q, k, outer, return_int=True)
    assert _route(dci)[0] >= 2 and _plan(dci)[0] == 1
    torch.cuda.synchronize()
    dci.query(Q, K, OUTER, return_int=True)      # (of its own record, which the other call has left as it was, or begun)
    assert _route(dci)[0] >= 2 and _plan(dci)[0] == 0


def test_many_shapes_of_queries_in_turn(of_no_use):
    """More of them than records are kept: each is tried again when its record was given to another."""
    dci, _, Q = of_no_use
    for turn in range(2):
        for k in range(K + 1, K + 6):
            dci.query(Q, k, OUTER, return_int=True)
            assert _plan(dci)[0] == 1, (turn, k)
            torch.cuda.synchronize()


def test_a_call_fits_the_room_of_the_one_before_it(gpu):
    """An index's first small call goes without near rows, the next one not: it finds its room all the same, also where nothing can grow, under
    capture (and where no build has left a workspace that holds it by chance)."""
    from dciknn_cuda_amd import _capi
    n, dim, nq, B, T, k = 200_000, 64, 32, 100, 10, 10
    X, Q = _rows("clusters", n, nq, dim, 6)
    dci = gpu.DCI(dim, 2, 7, B, T, seed=3)
    dci.append(X)
    ids = torch.empty((nq, k), dtype=torch.int32, device="cuda")
    dists = torch.empty((nq, k), dtype=torch.float32, device="cuda")

    def call(stream):
        _capi.check(dci._lib.dcih_query(dci._dci_inst, dim, nq, Q.data_ptr(), k, 0, 5000, 10 * k, B, T,
                                        ids.data_ptr(), dists.data_ptr(), None, stream))
    s = torch.cuda.Stream()
    call(s.cuda_stream)
    s.synchronize()
    assert _route(dci)[0] >= 2 and _plan(dci)[0] == 0
    want = ids.clone(), dists.clone()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        call(torch.cuda.current_stream().cuda_stream)
    assert _route(dci)[0] >= 2 and _plan(dci)[0] == 1
    for _ in range(3):
        ids.fill_(-5)
        dists.fill_(-5.0)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(ids, want[0]) and torch.equal(dists, want[1])
        call(0)                                # eager work between the replays
        torch.cuda.synchronize()
    del g
    dci.free()


def _held(make):
    """Device bytes that the handle made by `make` holds, and it."""
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    dci = make()
    torch.cuda.synchronize()
    return before - torch.cuda.mem_get_info()[0], dci


def test_no_room_is_held_for_positions_that_nothing_looks_up(gpu):
    """Wide windows, partitions too short for first lanes to be looked up: index and the build's workspace are all that is held."""
    n, M, L = 1_000_000, 2, 15
    X = torch.randn(n, 32, generator=torch.Generator(device="cuda").manual_seed(1), device="cuda")

    def make():
        dci = gpu.DCI(32, M, L, 900, 128, seed=3)
        dci.add(X)
        return dci
    gpu.DCI(32, M, L, 900, 128, seed=3).free()      # (what the library itself takes at its first use)
    held, dci = _held(make)
    dci.free()
    # keys, ids and two tables of positions, 12 bytes an entry, and the unsorted keys of the build: 4 more
    assert held < 16 * n * M * L + (16 << 20), held


@pytest.mark.parametrize("then", ["add", "add more", "append", "other stream"])
def test_positions_side_by_side_are_those_of_the_index(gpu, then):
    """The table of positions by points is formed anew for every index, whether its room holds it or not."""
    from dciknn_cuda_amd import _capi
    from test_gpu_rounds import ALWAYS, NEVER, _ask
    M, L, B, T, k, outer, dim = 2, 9, 4, 100, 8, 60, 24
    X, Q = _rows("normal", 30000, 80, dim, 7)
    dci = gpu.DCI(dim, M, L, B, T, seed=5)

    def check():
        want = _ask(dci, dci._lib, NEVER, Q, k, outer)
        for again in range(3):      # (formed once enough was asked for)
            got = _ask(dci, dci._lib, ALWAYS, Q, k, outer)
            assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1]), again
        assert _plan(dci)[2] > 0
    (dci.append if then == "append" else dci.add)(X[:24000])
    check()
    if then == "append":
        dci.append(X[24000:])
    else:
        dci.clear()
        X = X.flip(0).contiguous()
        dci.add(X[:24000] if then == "add" else X)
    if then == "other stream":
        torch.cuda.synchronize()
        with torch.cuda.stream(torch.cuda.Stream()):
            check()
    else:
        check()
    dci.free()


def test_positions_side_by_side_in_a_graph(gpu):
    """Recorded before they were formed, recorded when there is room for them but another index's, and recorded when they stand."""
    from dciknn_cuda_amd import _capi
    from test_gpu_rounds import ALWAYS, NEVER, _ask
    M, L, B, T, k, outer, dim, nq = 2, 9, 4, 100, 8, 60, 24, 80
    X, Q = _rows("normal", 24000, nq, dim, 7)
    ids = torch.empty((nq, k), dtype=torch.int32, device="cuda")
    dists = torch.empty((nq, k), dtype=torch.float32, device="cuda")
    dci = gpu.DCI(dim, M, L, B, T, seed=5)

    def call(stream, queries=Q):
        _capi.check(dci._lib.dcih_query(dci._dci_inst, dim, len(queries), queries.data_ptr(), k, 0, outer, 10 * k, B, T,
                                        ids.data_ptr(), dists.data_ptr(), None, stream))
    s = torch.cuda.Stream()
    for turn in ("none", "room", "formed"):
        if turn != "formed":
            dci.clear()
            X = X.flip(0).contiguous()
            dci.add(X)
        want = _ask(dci, dci._lib, NEVER, Q, k, outer)
        if turn == "none":      # (too few queries for the table, with room for all of them)
            _capi.check(dci._lib.dcih_set_option(dci._dci_inst, _capi.OPT_ROUNDS, ALWAYS))
            call(0, Q[:12])
        _capi.check(dci._lib.dcih_set_option(dci._dci_inst, _capi.OPT_ROUNDS, ALWAYS))
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            call(torch.cuda.current_stream().cuda_stream)
        assert _route(dci)[0] >= 2 and (_plan(dci)[2] > 0) == (turn != "none"), turn
        for _ in range(3):
            ids.fill_(-5)
            dists.fill_(-5.0)
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(ids, want[0]) and torch.equal(dists, want[1]), turn
            if turn != "room":
                call(0)                            # eager work between the replays
                torch.cuda.synchronize()
                assert torch.equal(ids, want[0]) and torch.equal(dists, want[1]), turn
        del g
    dci.free()


@pytest.mark.parametrize("dim", [64, 4096])
def test_steps_of_many_composites_do_not_fit_a_workgroup(gpu, dim):
    """64 composites of 64 simple indices: the steps of all their windows fit a workgroup's memory beside a short query, not beside a long one,
    whose calls look up all points as before."""
    from test_gpu_rounds import ALWAYS, NEVER, _ask
    X, Q = _rows("normal", 4000, 40, dim, 11)
    dci = gpu.DCI(dim, 64, 64, 4, 250, seed=5)
    dci.add(X)
    want = _ask(dci, dci._lib, NEVER, Q, 5, 20)
    for again in range(2):
        got = _ask(dci, dci._lib, ALWAYS, Q, 5, 20)
        assert _route(dci)[0] >= 2 and (_plan(dci)[2] > 0) == (dim == 64)
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1]), again
    dci.free()


@pytest.mark.parametrize("kind", ["normal", "sorted", "dup", "broken", "zero"])
@pytest.mark.parametrize("shape", [(20000, 96, 3, 8, 4, 128, 100, 100), (30000, 16, 2, 15, 4, 64, 9, 50), (24000, 64, 4, 5, 4, 48, 3, 150), (18000, 33, 3, 9, 3, 100, 10, 60),
                                   (24000, 40, 16, 2, 4, 48, 5, 150), (24001, 24, 8, 1, 4, 64, 9, 150)],
                         ids=["eight", "fifteen", "four composites", "three", "many composites", "one index each"])
def test_all_items_by_first_lanes(gpu, kind, shape):
    """Rounds whose items all go to the kernel that looks up first lanes of windows: several composites, and more promotions by first lanes (one a window and composite)
    than a workgroup lists, half as many as it ranks windows of a composite (the last two)."""
    from test_gpu_rounds import ALWAYS, NEVER, _ask
    n, dim, M, L, B, T, k, outer = shape
    X, Q = _rows(kind, n, 70, dim, n + dim)
    dci = gpu.DCI(dim, M, L, B, T, seed=5)
    dci.add(X)
    want = _ask(dci, dci._lib, NEVER, Q, k, outer)
    for again in range(3):
        got = _ask(dci, dci._lib, ALWAYS, Q, k, outer)
        assert torch.equal(got[0], want[0]), again
        assert torch.equal(got[1].view(torch.int32), want[1].view(torch.int32)), again
    assert _route(dci)[0] >= 2 and _plan(dci)[0] == 0 and _plan(dci)[2] > 0
    dci.free()
