"""What this engine's time is measured on.

A case is one call, or one short sequence of calls, that a program using `DCI` makes:

  query    an index stands, a batch of queries is answered
  blind    the same without distances: the candidates in the order they were promoted
  rebuild  `clear` + `add` of all rows on a handle that lives on, then a few lookups
  grow     `clear` + several `append`s, then a few lookups
  rank     a query with no number of neighbours given: every indexed point is ranked

The rows come from the five generators of dciknn_cuda_amd/workloads.py, made here on the
GPU: rows on a low-dimensional subspace ("example", the size of the reference's example), a
clipped and rounded Gaussian mixture ("mixture"), unit vectors ("sphere"), a noisy manifold
("manifold") and plain Gaussian rows ("normal").  (block_size, thread_size,
num_outer_iterations) are the settings bench.py runs and the constructor's and query's own
defaults (100, 10, 5000).
"""
import torch

import dciknn_cuda_amd as D

# (block_size, thread_size, num_outer_iterations)
DEFAULTS = (100, 10, 5000)
SETTINGS = [DEFAULTS, (100, 10, 500), (58, 2, 500), (100, 64, 126), (400, 128, 100), (900, 128, 10)]
# (num_comp_indices, num_simp_indices): the constructor's defaults and the benchmark's
INDICES = [(2, 7), (2, 10), (3, 8), (2, 12), (2, 15)]
ROWS = ["example", "mixture", "sphere", "manifold", "normal"]


def _case(name, op, rows, n, dim, indices, setting, k, nq, float_ids=False, parts=1):
    c = dict(op=op, rows=rows, n=n, dim=dim, m=indices[0], l=indices[1], bs=setting[0], ts=setting[1],
             outer=setting[2], k=k, nq=nq, float_ids=float_ids, parts=parts)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # The reference's example: a small table searched with the defaults, ids as the
        # reference returns them (float32).
        _case("example-query", "query", "example", 3000, 100, (2, 10), DEFAULTS, 10, 500, float_ids=True),
        # The same table indexed anew, as a program does whose rows change all the time.
        _case("example-rebuild", "rebuild", "example", 3000, 100, (2, 10), DEFAULTS, 10, 16),
        # One lookup in a million rows: an interactive user waits for it.
        _case("lookup-1", "query", "mixture", 1_000_000, 128, (2, 10), (58, 2, 500), 10, 1),
        # A server's small batch on a table of ordinary size with everything left at its default.
        _case("serve-32", "query", "mixture", 200_000, 64, (2, 7), DEFAULTS, 10, 32, float_ids=True),
        # Odd and ragged sizes: rows that start on no 16-byte boundary, partitions of unequal length.
        _case("ragged-query", "query", "normal", 123_457, 67, (3, 5), (37, 3, 1000), 7, 333),
        # The headline: 10k queries at recall@10 of 0.96.
        _case("batch-1m", "query", "mixture", 1_000_000, 128, (2, 10), (58, 2, 500), 10, 10_000),
        # A million rows with the constructor's and query's defaults.
        _case("defaults-1m", "query", "mixture", 1_000_000, 128, (2, 7), DEFAULTS, 10, 1000, float_ids=True),
        # The largest index: 10M unit vectors, 100 neighbours.
        _case("sphere-10m", "query", "sphere", 10_000_000, 96, (3, 8), (400, 128, 100), 100, 512),
        # Long rows.
        _case("manifold-1m", "query", "manifold", 1_000_000, 960, (2, 12), (100, 64, 126), 10, 500),
        # A million rows indexed anew.
        _case("rebuild-1m", "rebuild", "mixture", 1_000_000, 128, (2, 10), (58, 2, 500), 10, 16),
        # An index that grows by uneven batches.
        _case("grow-1m", "grow", "normal", 1_000_000, 64, (2, 15), (900, 128, 10), 50, 64, parts=4),
        # The default num_neighbours: all points in order of distance.
        _case("rank-20k", "rank", "manifold", 20_000, 100, (2, 7), DEFAULTS, 20_000, 64, float_ids=True),
    ]


def _spread(rng, lo, hi):
    """A whole number in [lo, hi], even over its logarithm."""
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    op = rng.choice(["query"] * 10 + ["blind"] + ["rebuild"] * 3 + ["grow"] * 2 + ["rank"] * 2)
    rows = rng.choice(ROWS)
    indices = rng.choice(INDICES)
    bs, ts, outer = rng.choice(SETTINGS)
    if op == "rank":
        n, dim = _spread(rng, 500, 50_000), _spread(rng, 16, 300)
    elif op == "grow":
        n, dim = _spread(rng, 2000, 1_000_000), _spread(rng, 16, 200)
    else:
        n, dim = _spread(rng, 1000, 1_500_000), _spread(rng, 16, 960)
        dim = min(dim, max(16, 250_000_000 // n))
    if rng.random() < 0.6:            # most tables have rows of whole 16-byte words
        dim = (dim + 3) // 4 * 4
    # block_size around the setting's, with at least 20 rows per partition
    bs = max(4, min(_spread(rng, int(0.7 * bs), int(1.4 * bs)), n // 20))
    k = n if op == "rank" else _spread(rng, 1, 100)
    if op in ("rebuild", "grow"):
        nq = _spread(rng, 1, 64)
    elif op == "rank":
        nq = _spread(rng, 1, 100)
    else:
        nq = _spread(rng, 1, 10_000)
    # no larger than the largest listed: (query, row, simple index) triples
    nq = max(1, min(nq, 8_000_000_000 // (n * indices[0] * indices[1])))
    float_ids = op == "rank" or rng.random() < 0.3
    parts = rng.randint(2, 6) if op == "grow" else 1
    return _case(None, op, rows, n, dim, indices, (bs, ts, outer), k, nq, float_ids, parts)


def _make_rows(kind, n, dim, gen):
    def randn(*shape):
        return torch.randn(*shape, generator=gen, device="cuda")

    def rand(*shape):
        return torch.rand(*shape, generator=gen, device="cuda")

    if kind == "example":
        latent = max(2, dim // 2)
        return rand(n, latent) @ randn(latent, dim)
    if kind == "mixture":
        centres = rand(min(1000, max(1, n // 50)), dim) * 255.0
        of = torch.randint(0, centres.shape[0], (n,), generator=gen, device="cuda")
        return centres[of].add_(randn(n, dim), alpha=20.0).clamp_(min=0.0).round_()
    if kind == "sphere":
        x = randn(n, dim)
        return x.div_(x.norm(dim=1, keepdim=True))
    if kind == "manifold":
        latent = min(32, dim)
        return ((rand(n, latent) * 2.0 - 1.0) @ randn(latent, dim)).add_(randn(n, dim), alpha=0.1)
    assert kind == "normal", kind
    return randn(n, dim)


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    # rows and queries are one draw, the queries its last rows
    both = _make_rows(case["rows"], case["n"] + case["nq"], case["dim"], gen)
    rows, queries = both[:case["n"]], both[case["n"]:].clone()
    dci = D.DCI(case["dim"], case["m"], case["l"], case["bs"], case["ts"], seed=seed)
    state = dict(case=case, dci=dci, rows=rows, queries=queries)
    if case["op"] == "grow":
        # batches of unequal size, none empty
        n, parts = case["n"], case["parts"]
        cuts = [0] + [int(n * ((i + 0.3 * (i % 2)) / parts)) for i in range(1, parts)] + [n]
        state["batches"] = [rows[a:b] for a, b in zip(cuts, cuts[1:])]
    elif case["op"] != "rebuild":
        dci.add(rows)
    return state


def run(state):
    case, dci = state["case"], state["dci"]
    ask = dict(return_int=not case["float_ids"])
    if case["op"] == "rank":
        return dci.query(state["queries"], **ask)
    if case["op"] == "rebuild":
        dci.clear()
        dci.add(state["rows"])
    elif case["op"] == "grow":
        dci.clear()
        for batch in state["batches"]:
            dci.append(batch)
    return dci.query(state["queries"], case["k"], case["outer"], blind=case["op"] == "blind", **ask)


def work(case):
    """Lower bounds.  A query: its row and its projections; in every partition at least k points
    have to be promoted (fewer where it holds fewer) before the traversal may stop, each found in
    the l simple indices of a composite (4 bytes) and its row read, no byte of rows or index more
    than once a pass; the results.  A build: rows read, keys and ids of every simple index
    written; appended rows are copied as well."""
    n, nq, dim, idx = case["n"], case["nq"], case["dim"], case["m"] * case["l"]
    per_part = -(-n // case["bs"])
    promoted = nq * case["bs"] * min(case["k"], per_part)
    width = min(10 * case["k"], case["outer"]) if case["op"] == "blind" else case["k"]
    nbytes = 4.0 * nq * dim + 8.0 * nq * width
    flops = 2.0 * nq * idx * dim
    nbytes += min(4.0 * idx * n, 4.0 * case["l"] * promoted)
    if case["op"] != "blind":
        nbytes += 4.0 * dim * min(n, promoted)
        flops += 3.0 * dim * promoted
    if case["op"] in ("rebuild", "grow"):
        nbytes += 4.0 * n * dim + 8.0 * n * idx
        flops += 2.0 * n * idx * dim
    if case["op"] == "grow":
        nbytes += 8.0 * n * dim
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # Distances are 32-bit sums over a row; ids (whole numbers, or float32 holding them) differ
    # only where two neighbours lie closer together than such a sum resolves.
    return {"rel": 1e-5, "max": 1e-4, "differ": 1e-3}
