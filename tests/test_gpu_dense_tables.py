"""The dense traversal at the edges of its tables: every workgroup size and number of windows per
thread, partitions of ties and of one cluster with a far point (the ranking by buckets gives up
there), rows compared by their 8-bit codes, and rows too close together for those."""
import numpy as np
import pytest
import torch

from util import engine_index, engine_project

pytestmark = pytest.mark.gpu

# (points per partition, partitions, L, T): windows per composite index at and just past the most a
# workgroup of 64, 256 or 512 threads holds at 5, 9, 13, 15, 33 and 21 windows per thread
TABLES = [(1, 3, 2, 1), (7, 2, 2, 3), (314, 2, 2, 2), (316, 2, 2, 2), (378, 1, 3, 2), (512, 1, 3, 1), (513, 1, 3, 1),
          (1225, 2, 10, 10), (2031, 2, 9, 8), (2045, 1, 5, 4), (4072, 1, 9, 8), (4080, 1, 9, 8), (5103, 1, 10, 8), (5300, 1, 10, 8), (5565, 2, 11, 8),
          (6127, 1, 11, 8), (6140, 2, 11, 8), (6127, 1, 14, 8), (9000, 1, 3, 300), (22223, 1, 15, 128)]


@pytest.mark.parametrize("ppb,B,L,T", TABLES)
@pytest.mark.parametrize("kind,dim", [("normal", 12), ("ties", 12), ("outlier", 12), ("normal", 100), ("close", 100),
                                      ("normal", 201), ("normal", 300), ("outlier", 520)])
def test_dense_tables(gpu, oracle, ppb, B, L, T, kind, dim):
    rng = np.random.default_rng(ppb + 7 * L + dim)
    n, M, nq, outer = ppb * B, 2, 24, 10_000
    X = rng.standard_normal((n, dim)).astype(np.float32)
    Q = rng.standard_normal((nq, dim)).astype(np.float32)
    if kind == "ties":
        X[: n // 2] = X[0]
        Q[0] = X[0]
    elif kind == "outlier":
        X[1:] *= 1e-3
        X[0] *= 1e4
        Q *= 1e-3
    elif kind == "close":
        X = (5.0 + 1e-4 * X).astype(np.float32)
        Q = (5.0 + 1e-4 * Q).astype(np.float32)
    got = {}
    for traversal in ("step", "dense"):
        dci = gpu.DCI(dim, M, L, B, T, seed=3, traversal=traversal)
        dci.add(torch.from_numpy(X).cuda())
        qd = torch.from_numpy(Q).cuda()
        # (the later calls find the codes of the rows formed)
        got[traversal] = [dci.query(qd, min(k, n), outer, return_int=True, return_counters=True) for k in (50, 50, 50, 8)]
        if traversal == "dense" and kind == "normal":
            skeys, sids = engine_index(dci)
            k = min(50, n)
            ref = oracle.query(skeys, sids, X, Q, engine_project(dci.directions.numpy(), Q).T.copy(), M, L, B, T, k, outer,
                               max_cand=10 * k)
            np.testing.assert_allclose(got["dense"][2][1].cpu().numpy(), ref["dists"], rtol=1e-5, atol=1e-6)
        dci.free()
    # (against the step kernel to the bit; against the oracle, whose sums run in another order, by distances)
    for (si, sd, sc), (di, dd, dc) in zip(got["step"], got["dense"]):
        assert torch.equal(si, di) and torch.equal(sd, dd)
        assert torch.equal(sc[:, 1], dc[:, 1])


# items from eight times what the device holds on: one workgroup each, in order (narrow workgroups, wide ones)
@pytest.mark.parametrize("ppb,B,nq", [(20, 37, 1100), (600, 13, 800), (3, 1, 40_000)])
def test_many_items(gpu, ppb, B, nq):
    rng = np.random.default_rng(ppb)
    dim, M, L, T, k, outer = 8, 2, 3, 4, 10, 60
    X = rng.standard_normal((ppb * B - 1, dim)).astype(np.float32)      # the last partition is one short
    Q = torch.from_numpy(rng.standard_normal((nq, dim)).astype(np.float32)).cuda()
    got = {}
    for traversal in ("step", "dense"):
        dci = gpu.DCI(dim, M, L, B, T, seed=3, traversal=traversal)
        dci.add(torch.from_numpy(X).cuda())
        got[traversal] = dci.query(Q, min(k, len(X)), outer, return_int=True, return_counters=True)
        dci.free()
    for j in (0, 1):
        assert torch.equal(got["step"][j], got["dense"][j])
    assert torch.equal(got["step"][2][:, [1, 3]], got["dense"][2][:, [1, 3]])


def test_one_window_too_many_is_refused(gpu):
    from dciknn_cuda_amd import _capi
    dci = gpu.DCI(8, 1, 14, 1, 8, seed=3, traversal="dense")
    X = torch.randn(6128, 8, device="cuda")            # 14 * (6128 / 8 + 3) = 10766 windows, 10752 fit
    dci.add(X)
    with pytest.raises(_capi.DCIError, match="dense"):
        dci.query(X[:4].contiguous(), 5, 50, return_int=True)
    dci.free()
