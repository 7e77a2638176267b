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

    def __init__(self, gpu, X):
        self.dense, self.step = (gpu.DCI(DIM, M, L, B, T, seed=3, traversal=t) for t in ("dense", "step"))
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
        assert int(self.ticks[9]) == len(Q) * B
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


def test_many_outlying_queries_rest_the_codes_for_a_while(gpu):
    rng = np.random.default_rng(2)
    p = _Pair(gpu, _rows(rng, N))
    Q = _rows(rng, 300)
    p.ask(Q)
    assert p.ask(1e5 * Q) == 0
    for _ in range(3):                        # rests are counted in items: an ordinary batch ends them
        took = p.ask(Q)
    assert took == 300 * B
    p.free()


def test_rows_too_close_for_their_codes(gpu):
    rng = np.random.default_rng(3)
    p = _Pair(gpu, _rows(rng, N, spread=1e-4))
    Q = _rows(rng, 200, spread=1e-4)
    for _ in range(4):
        assert p.ask(Q) == 0
    p.free()
