"""Rows compared by their 8-bit codes: which items are, and that it never shows in the results."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

N, DIM, M, L, B, T, K, OUTER = 12_000, 256, 2, 7, 4, 16, 10, 400


def _rows(rng, n, spread=1.0):
    return (5.0 * (spread != 1.0) + spread * rng.standard_normal((n, DIM))).astype(np.float32)


class _Pair:
    """The same rows behind the dense kernel and behind the step-by-step kernel."""

    def __init__(self, gpu, X, parts=B):
        self.parts = parts
        self.dense, self.step = (gpu.DCI(DIM, M, L, parts, T, seed=3, traversal=t) for t in ("dense", "step"))
        xd = torch.from_numpy(X).cuda()
        self.dense.add(xd)
        self.step.add(xd)
        self.ticks = torch.zeros(16, dtype=torch.int64, device="cuda")

    def ask(self, Q):
        """Items the dense kernel took by codes, after comparing its answer with the other's."""
        from dciknn_cuda_amd import _capi
        lib, h = self.dense._lib, self.dense._dci_inst
        q = torch.from_numpy(Q).cuda()
        self.ticks.zero_()
        _capi.check(lib.dcih_phase_profile(h, self.ticks.data_ptr()))
        ids, dists = self.dense.query(q, K, OUTER, return_int=True)
        _capi.check(lib.dcih_phase_profile(h, None))
        want = self.step.query(q, K, OUTER, return_int=True)
        assert torch.equal(ids, want[0]) and torch.equal(dists, want[1])
        assert int(self.ticks[9]) == len(Q) * self.parts
        return int(self.ticks[15])

    def free(self):
        self.dense.free()
        self.step.free()


def test_an_outlying_query_costs_only_itself(gpu):
    rng = np.random.default_rng(1)
    p = _Pair(gpu, _rows(rng, N))
    Q = _rows(rng, 200)
    p.ask(Q)                                  # (the codes are formed by now)
    assert p.ask(Q) == 200 * B
    far = Q.copy()
    far[7] = 1e5 * Q[7]                       # distances that differ by less than the margin
    assert p.ask(far) == 199 * B
    assert p.ask(Q) == 200 * B
    p.free()


# (few long partitions, many short ones: different numbers of items are under way together)
@pytest.mark.parametrize("parts,every", [(4, 1), (4, 2), (24, 1), (24, 2), (24, 3)])
def test_many_outlying_queries_rest_the_codes_for_a_while(gpu, parts, every):
    rng = np.random.default_rng(2)
    p = _Pair(gpu, _rows(rng, N), parts)
    Q = _rows(rng, 600)
    p.ask(Q)
    far = Q.copy()
    far[::every] *= 1e5
    for _ in range(3):
        assert p.ask(far) <= (600 - len(far[::every])) * parts
    for _ in range(3):                        # rests are counted in items: ordinary batches end them
        took = p.ask(Q)
    assert took == 600 * parts
    p.free()


def test_rows_too_close_for_their_codes(gpu):
    rng = np.random.default_rng(3)
    p = _Pair(gpu, _rows(rng, N, spread=1e-4))
    Q = _rows(rng, 200, spread=1e-4)
    for _ in range(4):
        assert p.ask(Q) == 0
    p.free()


def _device_bytes():
    torch.cuda.synchronize()
    free, total = torch.cuda.mem_get_info()
    return total - free


def test_room_for_the_codes_is_taken_when_they_are_formed(gpu):
    n = 400_000                               # codes: 109 MB; index arrays: 5 MB per simple index
    X, Q = torch.randn(n, DIM, device="cuda"), torch.randn(400, DIM, device="cuda")
    codes = n * (16 + DIM)
    dci = gpu.DCI(DIM, 1, 2, 64, T, seed=3, traversal="dense")
    before = _device_bytes()
    dci.add(X)
    assert _device_bytes() - before < codes // 2
    for _ in range(3):
        first = dci.query(Q, K, OUTER, return_int=True)
    held = _device_bytes()
    assert held - before > codes
    dci.clear()                               # the same size again: the same room
    dci.add(X)
    for _ in range(3):
        again = dci.query(Q, K, OUTER, return_int=True)
    assert torch.equal(first[0], again[0]) and torch.equal(first[1], again[1])
    assert abs(_device_bytes() - held) < codes // 4
    dci.free()
    assert _device_bytes() - before < codes // 2


@pytest.mark.parametrize("then", ["on another stream", "in a graph"])
def test_codes_just_formed(gpu, then):
    from dciknn_cuda_amd import _capi
    rng = np.random.default_rng(4)
    Q = torch.from_numpy(_rows(rng, 300)).cuda()
    X = torch.from_numpy(_rows(rng, N)).cuda()
    step = gpu.DCI(DIM, M, L, B, T, seed=3, traversal="step")
    step.add(X)
    want = step.query(Q, K, OUTER, return_int=True)
    dci = gpu.DCI(DIM, M, L, B, T, seed=3, traversal="dense")
    dci.add(X)
    ticks = torch.zeros(16, dtype=torch.int64, device="cuda")
    _capi.check(dci._lib.dcih_phase_profile(dci._dci_inst, ticks.data_ptr()))
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    outs = [(torch.full((300, K), -7, dtype=torch.int32, device="cuda"), torch.full((300, K), -7.0, device="cuda"))
            for _ in range(3)]

    def call(stream, out):
        _capi.check(dci._lib.dcih_query(dci._dci_inst, DIM, 300, Q.data_ptr(), K, 0, OUTER, 10 * K, B, T,
                                        out[0].data_ptr(), out[1].data_ptr(), None, stream))

    torch.cuda.synchronize()
    call(a.cuda_stream, outs[0])              # forms the codes
    g = None
    if then == "in a graph":                  # (the very next call is recorded, on another stream)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=b):
            call(torch.cuda.current_stream().cuda_stream, outs[2])
    b.wait_stream(a)                          # (the workspace is the handle's: its calls are kept in order)
    call(b.cuda_stream, outs[1])
    torch.cuda.synchronize()
    assert int(ticks[15]) == int(ticks[9]) == 2 * 300 * B
    for _ in range(3):
        if g is not None:
            for out in outs[2]:
                out.fill_(-5)
            ticks.zero_()
            g.replay()
            torch.cuda.synchronize()
            assert int(ticks[15]) == 300 * B
        call(b.cuda_stream, outs[1])          # eager work between the replays
        torch.cuda.synchronize()
        for ids, dists in outs if g is not None else outs[:2]:
            assert torch.equal(ids, want[0]) and torch.equal(dists, want[1])
    _capi.check(dci._lib.dcih_phase_profile(dci._dci_inst, None))
    del g
    dci.free()
    step.free()
