"""Rows of distances ranked in full: every number of items per thread at its edges, up to and
past the longest row one workgroup holds; ties, one far row (the ranking by buckets gives up
there), values that are not finite."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 257, 1025, 2048, 2049, 4096, 4097, 8191, 8193, 16384, 16385, 24575, 24576, 24577])
@pytest.mark.parametrize("kind", ["normal", "equal", "outlier", "infinite"])
def test_full_ranking(gpu, n, kind):
    rng = np.random.default_rng(n)
    dim, nq = 3, 3
    X = rng.standard_normal((n, dim)).astype(np.float32)
    if kind == "equal":
        X[: n // 2] = X[0]
        X[n - n // 3:] = X[n - 1]
    elif kind == "outlier":
        X *= 1e-3
        X[0] = 1e6
    elif kind == "infinite":
        X[::5] *= 1e30
    Q = rng.standard_normal((nq, dim)).astype(np.float32) * (1e-3 if kind == "outlier" else 1)
    dci = gpu.DCI(dim, 1, 2, max(1, n // 8), 2, seed=1)
    dci.add(torch.from_numpy(X).cuda())
    with np.errstate(over="ignore"):
        d = np.zeros((nq, n), np.float32)
        for c in range(dim):
            t = X[None, :, c] - Q[:, c, None]
            d += t * t
    d = np.sqrt(d)
    order = np.lexsort((np.broadcast_to(np.arange(n), d.shape), d))
    for k in {n, min(n, 300)}:
        ids, dists = dci.query(torch.from_numpy(Q).cuda(), -1 if k == n else k, 5000, return_int=True)
        fids, fdists = dci.query(torch.from_numpy(Q).cuda(), -1 if k == n else k, 5000)
        np.testing.assert_array_equal(ids.cpu().numpy(), order[:, :k])
        np.testing.assert_array_equal(dists.cpu().numpy(), np.take_along_axis(d, order[:, :k], 1))
        assert torch.equal(fids, ids.float()) and torch.equal(fdists, dists)
    dci.free()
