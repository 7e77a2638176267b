"""Queries that first bound the partitions' nearest distances and then traverse, in rounds, only the partitions
that can hold a result (DCIH_OPT_ROUNDS), against the same queries traversed as a whole: ids and distances
must be equal to the bit, whatever the rows are, because a partition is left out only where none of its rows can
be as near as the k-th result.  Every traversal kernel that can run a round is covered."""
import math
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

NEVER, ALWAYS = 1, 2


def _ask(dci, lib, rounds, Q, k, outer, **kw):
    from dciknn_cuda_amd import _capi
    _capi.check(lib.dcih_set_option(dci._dci_inst, _capi.OPT_ROUNDS, rounds))
    ids, dists = dci.query(Q, k, outer, return_int=True, **kw)
    torch.cuda.synchronize()
    return ids.clone(), dists.clone()


def _route(dci):
    """(rounds, bounds of tiles kept, queries of the sample, queries selected by bounds of all rows) of the last call."""
    from dciknn_cuda_amd import _capi
    route = (_capi.ctypes.c_int64 * 4)()
    _capi.check(dci._lib.dcih_debug_route(dci._dci_inst, route))
    return tuple(route)


def _count_items(dci):
    """A tensor that later calls write the items of every round to, then what the sample decided."""
    from dciknn_cuda_amd import _capi
    items = torch.zeros(6, dtype=torch.int32, device="cuda")
    _capi.check(dci._lib.dcih_debug_round_items(dci._dci_inst, items.data_ptr()))
    return items


def _same(gpu, X, Q, M, L, B, T, k, outer, tag="", near=None):
    dci = gpu.DCI(X.shape[1], M, L, B, T, seed=3)
    dci.add(X)
    want = _ask(dci, dci._lib, NEVER, Q, k, outer)
    assert _route(dci) == (0, 0, 0, 0), tag
    got = _ask(dci, dci._lib, ALWAYS, Q, k, outer)
    route = _route(dci)
    dci.free()
    assert route[0] >= 2 or route[3] == len(Q), (tag, route)      # the call did go in rounds (or its results were selected)
    assert near is None or route[1] == near, (tag, route)
    assert torch.equal(got[0], want[0]), tag
    assert torch.equal(got[1].view(torch.int32), want[1].view(torch.int32)), tag
    return want


def _rows(kind, n, nq, dim, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    def randn(*s):
        return torch.randn(*s, generator=g, device="cuda")
    x = randn(n + nq, dim)
    if kind == "clusters":
        x = 30.0 * randn(20, dim)[torch.randint(0, 20, (n + nq,), generator=g, device="cuda")] + x
    elif kind == "sorted":          # a query's neighbours all lie in one or two partitions
        x = x[torch.argsort(x[:, 0])]
        x = x[torch.cat([torch.arange(0, n, device="cuda"), torch.randint(0, n, (nq,), generator=g, device="cuda")])]
        x[n:] += 0.01 * randn(nq, dim)
    elif kind == "dup":             # equal distances, by the id alone
        x = x[torch.randint(0, max(1, n // 8), (n + nq,), generator=g, device="cuda")]
    elif kind == "grid":
        x = torch.randint(0, 3, (n + nq, dim), generator=g, device="cuda").float()
    elif kind == "whole":           # whole numbers: many equal distances
        x = (40.0 * x).round()
    elif kind == "offset":          # squared lengths a million times the distances'
        x = x + 3000.0
    elif kind == "scales":          # rows from 1e-6 to 1e6: most of them outside what 16-bit floats of one scale hold
        x = x * 10.0 ** (12.0 * torch.rand(n + nq, 1, generator=g, device="cuda") - 6.0)
    elif kind == "tiny":            # squares below the smallest float: all distances are computed as zero
        x = x * 1e-25
    elif kind == "huge":            # squares that overflow
        x = x * 1e25
    elif kind == "broken":          # some rows and queries are not finite
        x[::97] = float("nan")
        x[5::101, 0] = float("inf")
        x[7::103, 0] = -float("inf")
    elif kind == "zero":
        x[: (n + nq) // 2] = 0.0
    return x[:n].contiguous(), x[n:].contiguous()


# one shape per kernel form: queries 1..32, 33..64, 65..128 and more, rows whole in LDS and staged by columns
# (past 256 elements), with and without whole octets, one element and one tile past each edge
@pytest.mark.parametrize("nq", [1, 32, 33, 65, 129, 300])
@pytest.mark.parametrize("dim", [8, 9, 16, 67, 256, 257, 520])
def test_forms_of_the_product(gpu, nq, dim):
    X, Q = _rows("clusters", 5000 + dim, nq, dim, nq * 1000 + dim)
    _same(gpu, X, Q, 2, 5, 11, 8, 5, 40, "dim %d nq %d" % (dim, nq))


@pytest.mark.parametrize("kind", ["normal", "clusters", "sorted", "dup", "grid", "offset", "scales", "tiny", "huge", "broken", "zero"])
@pytest.mark.parametrize("shape", [(2, 7, 20, 10, 10, 5000), (2, 10, 13, 2, 4, 100), (3, 5, 40, 64, 30, 20), (1, 3, 7, 130, 1, 5)],
                         ids=["defaults", "narrow", "wide", "one"])
@pytest.mark.parametrize("dim", [24, 33, 300])
def test_rows_of_every_kind(gpu, kind, shape, dim):
    M, L, B, T, k, outer = shape
    X, Q = _rows(kind, 9001, 150, dim, 17 + dim)
    ids, _ = _same(gpu, X, Q, M, L, B, T, k, outer, kind)
    assert ids.shape == (150, k)


# Wide windows: the first lanes of the windows and the rows of near tiles are looked up instead of all points, with positions side by side in
# eights (one, a whole eight, one more, two eights less one), windows of and not of a power of two, above 256; formed once enough was asked for.
@pytest.mark.parametrize("kind", ["normal", "sorted", "dup", "whole", "broken", "zero"])
@pytest.mark.parametrize("shape", [(9001, 24, 1, 1, 3, 64, 5, 400), (20000, 96, 3, 8, 4, 128, 100, 100), (9000, 33, 2, 9, 5, 100, 10, 60),
                                   (30000, 16, 2, 15, 4, 64, 9, 50), (24000, 200, 2, 4, 2, 300, 20, 40), (2400, 64, 4, 5, 6, 48, 3, 30)],
                         ids=["one", "eight", "nine", "fifteen", "four", "short"])
def test_wide_windows(gpu, kind, shape):
    n, dim, M, L, B, T, k, outer = shape
    X, Q = _rows(kind, n, 70, dim, n + dim)
    dci = gpu.DCI(dim, M, L, B, T, seed=5)
    dci.add(X)
    want = _ask(dci, dci._lib, NEVER, Q, k, outer)
    for again in range(3):
        got = _ask(dci, dci._lib, ALWAYS, Q, k, outer)
        assert _route(dci)[0] >= 2, again
        assert torch.equal(got[0], want[0]), again
        assert torch.equal(got[1].view(torch.int32), want[1].view(torch.int32)), again
    assert _route(dci)[1] == 1
    dci.free()


@pytest.mark.parametrize("n,B", [(130, 2), (257, 128), (1000, 999), (4096, 32), (4097, 32), (31 * 129, 31)])
def test_partitions_at_the_edges_of_tiles(gpu, n, B):
    """Partitions of 1, 2, 3, 65, 128, 129 rows, some of them empty, more results asked for than a partition holds."""
    for k in (1, 3, 40):
        X, Q = _rows("normal", n, 70, 40, n + k)
        _same(gpu, X, Q, 2, 4, B, 2, k, 3, "n %d B %d k %d" % (n, B, k))


def test_rows_off_their_boundaries(gpu):
    """Rows and queries that start four bytes past a 16-byte boundary."""
    X, Q = _rows("clusters", 6001, 90, 64, 5)
    pool_x = torch.empty(X.numel() + 1, device="cuda")
    pool_q = torch.empty(Q.numel() + 1, device="cuda")
    x, q = pool_x[1:].view(X.shape), pool_q[1:].view(Q.shape)
    x.copy_(X)
    q.copy_(Q)
    assert x.data_ptr() % 16 == 4 and q.data_ptr() % 16 == 4
    _same(gpu, x, q, 2, 7, 20, 10, 10, 500)


# Traversals of a small part of their partitions: a sample of the queries decides whether bounds are formed at all.  Rows that bounds tell
# apart and rows that they do not, more queries than the sample and as many, partitions by the dozen and a few.
@pytest.mark.parametrize("kind,dim,outcome", [("normal", 8, 0), ("grid", 64, 1), ("normal", 64, None), ("broken", 16, None)])
def test_a_sample_decides_about_rounds(gpu, kind, dim, outcome):
    n, nq, B, T, k, outer = 30000, 4000, 58, 2, 5, 100
    X, Q = _rows(kind, n, nq, dim, 8)
    dci = gpu.DCI(dim, 2, 10, B, T, seed=3)
    dci.add(X)
    want = _ask(dci, dci._lib, NEVER, Q, k, outer)
    items = _count_items(dci)
    got = _ask(dci, dci._lib, 0, Q, k, outer)
    assert _route(dci) == (3, 0, 16, 0)
    items = items.tolist()
    dci.free()
    assert torch.equal(got[0], want[0]) and torch.equal(got[1].view(torch.int32), want[1].view(torch.int32))
    assert outcome is None or items[4] == outcome, items
    if items[4]:
        assert items[:3] == [nq * B, 0, 0], items
    else:
        assert 0 < items[0] < nq * B // 2 and items[5] < 16 * 15, items


# Where many items are expected the dense kernel's launch holds a workgroup for each, and the last ones to start go on by tickets: as
# many items as expected, several times as many, and a few; partitions of 300 rows (64 threads a workgroup) and of 2500.
@pytest.mark.parametrize("kind,least,most", [("normal", 0.5, 2.0), ("far", 2.0, 20.0), ("apart", 0.0, 0.8)])
@pytest.mark.parametrize("B", [100, 12])
def test_a_workgroup_for_every_expected_item(gpu, kind, least, most, B):
    n, nq, dim, k = 30000, 10000 if B == 100 else 3000, 24, 5
    X, Q = _rows("normal", n, nq, dim, B)
    if kind != "normal":            # clusters in every partition, or each in one of them
        at = 5000.0 * torch.randn(100, dim, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
        rows = torch.arange(n, device="cuda")
        X += at[rows % 100 if kind == "far" else rows * 100 // n]
        Q += at[torch.arange(nq, device="cuda") % 100]
    dci = gpu.DCI(dim, 2, 7, B, 10, seed=3)
    dci.add(X)
    want = _ask(dci, dci._lib, NEVER, Q, k, 5000)
    items = _count_items(dci)
    got = _ask(dci, dci._lib, ALWAYS, Q, k, 5000)
    assert _route(dci)[0] == 4
    dci.free()
    assert torch.equal(got[0], want[0]) and torch.equal(got[1].view(torch.int32), want[1].view(torch.int32))
    expected = nq * (B * (1.0 - math.exp(-k / B)) + 0.5)
    assert expected >= 8 * 8 * 32 * (4 if B == 12 else 16)      # (dies, items a workgroup, CUs of a die, workgroups a CU)
    assert least * expected <= int(items[0]) <= most * expected, (items.tolist(), expected)


@pytest.mark.parametrize("dim", [40, 200])
def test_bounds_that_say_nothing(gpu, dim):
    """Clusters much further apart than they are wide, and a column that drowns the others: all partitions come in round 1, several times as
    many as the dense kernel's workgroups, by whole rows at first and by the rows' codes in later calls; other rows after that."""
    n, nq, B, T, k, outer = 60000, 500, 60, 10, 10, 5000
    dci = gpu.DCI(dim, 2, 7, B, T, seed=3)
    for kind in ("far", "column", "normal"):
        X, Q = _rows("normal", n, nq, dim, dim)
        if kind == "far":
            at = 5000.0 * torch.randn(20, dim, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
            X += at[torch.arange(n, device="cuda") % 20]
            Q += at[torch.arange(nq, device="cuda") % 20]
        elif kind == "column":
            X[:, 3] *= 1e5
            Q[:, 3] *= 1e5
        dci.clear()
        dci.add(X)
        want = _ask(dci, dci._lib, NEVER, Q, k, outer)
        items = _count_items(dci)
        for call in range(3):
            got = _ask(dci, dci._lib, 0, Q, k, outer)
            assert _route(dci)[0] >= 2 and _route(dci)[1] == 1, (kind, call)      # in rounds, with the tiles' bounds
            assert torch.equal(got[0], want[0]) and torch.equal(got[1].view(torch.int32), want[1].view(torch.int32)), (kind, call)
            assert kind == "normal" or int(items[0]) > 0.9 * nq * B, (kind, items.tolist())
    dci.free()


@pytest.mark.parametrize("nq", [1, 2, 15, 16, 17, 31, 100])
@pytest.mark.parametrize("B", [2, 11, 12, 13, 25, 300])
def test_samples_of_few_queries_and_partitions(gpu, nq, B):
    X, Q = _rows("clusters", 40 * B + 7, nq, 19, nq + B)
    _same(gpu, X, Q, 2, 6, B, 2, 2, 6, "nq %d B %d" % (nq, B))


@pytest.mark.parametrize("kind,dim,k,T,outer", [("normal", 64, 5, 2, 100), ("clusters", 64, 3, 2, 30)])
def test_more_items_in_a_later_round_than_its_launch_covers(gpu, kind, dim, k, T, outer):
    """A launch of the batch kernel in a later round covers three tenths of all items, 65536 at least."""
    n, nq, B = 30000, 4000, 58
    X, Q = _rows(kind, n, nq, dim, 8)
    dci = gpu.DCI(dim, 2, 10, B, T, seed=3)
    dci.add(X)
    want = _ask(dci, dci._lib, NEVER, Q, k, outer)
    items = _count_items(dci)
    got = _ask(dci, dci._lib, ALWAYS, Q, k, outer)
    items = items.tolist()
    dci.free()
    assert torch.equal(got[0], want[0]) and torch.equal(got[1].view(torch.int32), want[1].view(torch.int32))
    assert kind != "normal" or max(items[1:3]) > 0.3 * nq * B, items


def test_rounds_run_the_kernel_of_whole_calls(gpu):
    """The traversal kernel is chosen for all items: bounds that rule nothing out leave them all to it."""
    from dciknn_cuda_amd import _capi
    X, Q = _rows("normal", 100000, 300, 16, 2)
    dci = gpu.DCI(16, 2, 10, 58, 2, seed=1)
    dci.add(X)
    _capi.check(dci._lib.dcih_profile(dci._dci_inst, 1))
    ran = []
    for rounds in (NEVER, 0, ALWAYS):
        _ask(dci, dci._lib, rounds, Q, 30, 500)
        t = (_capi.ctypes.c_float * _capi.NUM_TIMERS)()
        _capi.check(dci._lib.dcih_last_timings(dci._dci_inst, t))
        ran.append(bool(t[_capi.T_BATCH] > 0))
    dci.free()
    assert ran[0] == ran[1] == ran[2], ran


# A query's elements leave the range of 16-bit floats at 2^16 times what puts the sampled queries' largest at 64 .. 128, and twice
# its elements, which the product takes, a factor of two before: single elements either side of both.  The rows' column holds values
# of one sign in every second partition, so that no other row of a partition makes up for an infinite product.
@pytest.mark.parametrize("T,outer", [(2, 1500), (10, 5000)], ids=["batch", "dense"])
@pytest.mark.parametrize("dim,nq", [(24, 30), (33, 61), (24, 100), (264, 200), (33, 400), (24, 1100)])
def test_one_element_far_from_the_others(gpu, dim, nq, T, outer):
    n, B = 40000, 16
    X, Q = _rows("normal", n, nq, dim, dim + nq)
    part = torch.arange(n, device="cuda") // (n // B)
    X[:, 0] = 1e-3 * (2.0 * (part % 2) - 1.0)
    Q[:, 0] = 0.0
    sampled = {nq * r // 16 for r in range(16)}
    others = [q for q in range(nq) if q not in sampled]
    for i, q in enumerate(others[:14]):
        Q[q, 0] = (1.5 if i % 2 else -1.5) * 2.0 ** (7 + i // 2)
    _same(gpu, X, Q, 2, 7, B, T, 10, outer, "dim %d nq %d" % (dim, nq))


@pytest.mark.parametrize("k,T,outer", [(3, 2, 100), (10, 10, 5000)], ids=["batch", "dense"])
def test_more_partitions_at_one_bound_than_expected(gpu, k, T, outer):
    """Queries that are not finite bound nothing: all their partitions come in round 1, far more items than its
    launch was sized for."""
    X, Q = _rows("normal", 60000, 700, 20, 8)
    Q[::2] = float("nan")
    _same(gpu, X, Q, 2, 8, 60, T, k, outer)


@pytest.mark.parametrize("k,T,outer", [(3, 2, 100), (10, 10, 5000)], ids=["batch", "dense"])
def test_rounds_in_a_graph(gpu, k, T, outer):
    from dciknn_cuda_amd import _capi
    n, dim, nq, B = 30000, 48, 96, 16
    X, Q = _rows("clusters", n, nq, dim, 21)
    dci = gpu.DCI(dim, 2, 7, B, T, seed=9)
    dci.add(X)
    want = _ask(dci, dci._lib, NEVER, Q, k, outer)
    _capi.check(dci._lib.dcih_set_option(dci._dci_inst, _capi.OPT_ROUNDS, ALWAYS))
    ids = torch.empty((nq, k), dtype=torch.int32, device="cuda")
    dists = torch.empty((nq, k), dtype=torch.float32, device="cuda")

    def call(stream):
        _capi.check(dci._lib.dcih_query(dci._dci_inst, dim, nq, Q.data_ptr(), k, 0, outer, 10 * k, B, T,
                                        ids.data_ptr(), dists.data_ptr(), None, stream))
    s = torch.cuda.Stream()
    call(s.cuda_stream)
    call(s.cuda_stream)
    s.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        call(torch.cuda.current_stream().cuda_stream)
    for _ in range(4):
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


def test_no_room_for_the_bounds(gpu):
    """A recorded call cannot enlarge the workspace: what fits the one that whole traversals left is answered by them."""
    from dciknn_cuda_amd import _capi
    n, dim, nq, B, k = 30000, 48, 10000, 16, 3      # (the build's own workspace is smaller than the queries')
    X, Q = _rows("clusters", n, nq, dim, 22)
    dci = gpu.DCI(dim, 2, 7, B, 2, seed=9)
    dci.add(X)
    want = _ask(dci, dci._lib, NEVER, Q, k, 100)
    ids = torch.empty((nq, k), dtype=torch.int32, device="cuda")
    dists = torch.empty((nq, k), dtype=torch.float32, device="cuda")

    def call(stream):
        _capi.check(dci._lib.dcih_query(dci._dci_inst, dim, nq, Q.data_ptr(), k, 0, 100, 10 * k, B, 2,
                                        ids.data_ptr(), dists.data_ptr(), None, stream))
    s = torch.cuda.Stream()
    call(s.cuda_stream)
    s.synchronize()
    _capi.check(dci._lib.dcih_set_option(dci._dci_inst, _capi.OPT_ROUNDS, ALWAYS))
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        call(torch.cuda.current_stream().cuda_stream)
    assert _route(dci) == (0, 0, 0, 0)
    for _ in range(3):
        ids.fill_(-5)
        dists.fill_(-5.0)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(ids, want[0]) and torch.equal(dists, want[1])
    del g
    got = _ask(dci, dci._lib, ALWAYS, Q, k, 100)      # (not recorded, the same call takes the room and goes in rounds)
    assert _route(dci)[0] >= 2
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    dci.free()


def test_what_asks_for_everything_gets_everything(gpu):
    """Counters and blind queries are of whole traversals, also where rounds are asked for."""
    from dciknn_cuda_amd import _capi
    X, Q = _rows("normal", 20000, 40, 32, 4)
    dci = gpu.DCI(32, 2, 7, 25, 10, seed=3)
    dci.add(X)
    res = []
    for rounds in (NEVER, ALWAYS):
        _capi.check(dci._lib.dcih_set_option(dci._dci_inst, _capi.OPT_ROUNDS, rounds))
        counted = dci.query(Q, 10, 500, return_int=True, return_counters=True)
        blind = dci.query(Q, 10, 500, blind=True, return_int=True)
        torch.cuda.synchronize()
        res.append([t.clone() for t in counted] + [t.clone() for t in (blind if isinstance(blind, tuple) else (blind,))])
    for a, b in zip(*res):
        assert torch.equal(a, b)
    dci.free()


# Where no partition stops early the k nearest of all rows are selected by bounds of their distances: columns in one part and in
# several, whole octets and quads or not, the most columns there can be, the fewest rows, k either side of 32 and the largest.
@pytest.mark.parametrize("kind", ["normal", "clusters", "dup", "grid", "offset", "scales", "tiny", "huge", "broken", "zero"])
@pytest.mark.parametrize("n,dim,nq,k", [(1500, 150, 300, 10), (3000, 67, 301, 4), (6001, 41, 250, 33), (6500, 640, 65, 100),
                                         (1024, 8, 1, 16), (1100, 4096, 3, 7), (8200, 9, 70, 128)])
def test_nearest_of_all_rows(gpu, kind, n, dim, nq, k):
    X, Q = _rows(kind, n, nq, dim, n + dim)
    dci = gpu.DCI(dim, 2, 7, n // 20, 10, seed=3)
    dci.add(X)
    want = _ask(dci, dci._lib, NEVER, Q, k, 5000)
    got = _ask(dci, dci._lib, ALWAYS, Q, k, 5000)
    dci.free()
    assert torch.equal(got[0], want[0])
    assert torch.equal(got[1].view(torch.int32), want[1].view(torch.int32))


# Queries whose bounds rule out too little: all rows of small tables by the query's own workgroup, of larger ones in pieces of 2048 rows by
# several.  Tables either side of where that changes and of a whole number of pieces, one such query, some, all of them, rows in ascending
# and in descending order of distance.
@pytest.mark.parametrize("n", [6401, 8191, 8192, 8193, 10239, 10240, 10241, 100003])
@pytest.mark.parametrize("kind,k", [("one", 1), ("some", 33), ("dup", 10), ("all", 100), ("ascending", 7), ("descending", 100)])
def test_nearest_where_bounds_say_little(gpu, n, kind, k):
    dim, nq = 21, 37
    X, Q = _rows("dup" if kind == "dup" else "normal", n, nq, dim, n + k)
    if kind == "one":
        Q[nq - 1, 3] = float("nan")
    elif kind == "some":
        Q[1::5, dim - 1] = float("inf")
        Q[2::7, 0] = -float("nan")
    elif kind == "dup":
        X[: n // 2] = X[0]
        Q[:] = X[0] + 1e-3
    elif kind == "all":
        X[:] = 1e6 * X[:1] + 1e-4 * X
    else:
        order = torch.arange(n, device="cuda", dtype=torch.float32) / n
        X[:] = 0.0
        X[:, 5] = 3000.0 + (order if kind == "ascending" else 1.0 - order)
        Q[:] = 0.0
        Q[:, 7] = 1e30 if kind == "descending" else 0.0
    dci = gpu.DCI(dim, 2, 7, max(2, n // (8 * k)), 10, seed=3)
    dci.add(X)
    want = _ask(dci, dci._lib, NEVER, Q, k, 5000)
    got = _ask(dci, dci._lib, ALWAYS, Q, k, 5000)
    assert _route(dci)[3] == nq
    dci.free()
    assert torch.equal(got[0], want[0])
    assert torch.equal(got[1].view(torch.int32), want[1].view(torch.int32))


def test_nearest_of_many_rows(gpu):      # more than 512 workgroups of the product
    X, Q = _rows("clusters", 40000, 500, 72, 12)
    Q[7] = float("nan")
    dci = gpu.DCI(72, 2, 7, 1000, 64, seed=3)
    dci.add(X)
    want = _ask(dci, dci._lib, NEVER, Q, 64, 100)
    got = _ask(dci, dci._lib, 0, Q, 64, 100)
    assert _route(dci)[3] == 500
    dci.free()
    assert torch.equal(got[0], want[0])
    assert torch.equal(got[1].view(torch.int32), want[1].view(torch.int32))


# Rows ranked by several workgroups (few rows) and by one (many): sizes at the edges of both, of the rows that are kept in registers
# and of the numbers of 16 bits; distances spread evenly, equal, in clusters too dense for a part, and not finite.
@pytest.mark.parametrize("kind", ["normal", "grid", "whole", "zero", "huge", "broken"])
@pytest.mark.parametrize("n", [8191, 8192, 10001, 16384, 16385, 20480, 20481, 32768, 32769, 65536, 65537])
def test_ranking_in_parts(gpu, kind, n):
    X, Q = _rows(kind, n, 300, 9, n)
    dci = gpu.DCI(9, 2, 3, 50, 10, seed=3)
    dci.add(X)
    want = dci.query(Q, return_int=True)
    for some in (Q[:1], Q[40:56], Q[40:104]):
        got = dci.query(some.contiguous(), return_int=True)
        first = 0 if len(some) == 1 else 40
        assert torch.equal(got[0], want[0][first:first + len(some)])
        assert torch.equal(got[1].view(torch.int32), want[1][first:first + len(some)].view(torch.int32))
    few = dci.query(Q[:3].contiguous(), 8200 if n > 8200 else 300, 5000, return_int=True)
    dci.free()
    assert torch.equal(few[0], want[0][:3, :few[0].shape[1]])
