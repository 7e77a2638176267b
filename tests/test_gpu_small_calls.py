"""The kernels of small calls at the sizes where they can go wrong: the projection of few
rows and of rows on no 16-byte boundary, the merge of the partitions' lists, the selection
of few results from a row of distances."""
import numpy as np
import pytest
import torch

from util import engine_index, engine_project

pytestmark = pytest.mark.gpu


# (rows, dim, directions): around the workgroup's 8 rows, 32 directions and 128 columns, and
# on the streaming kernel's side of the limit with every remainder of the row length
@pytest.mark.parametrize("n,dim,I", [(1, 1, 1), (7, 3, 33), (8, 127, 32), (9, 128, 31), (17, 129, 64), (64, 257, 5),
                                     (32767, 5, 20), (32768, 4, 3), (32769, 5, 20), (32800, 30, 33), (33000, 67, 15),
                                     (32832, 31, 24), (40000, 1, 2), (33333, 36, 14), (32999, 98, 20)])
def test_projection(gpu, oracle, n, dim, I):
    rng = np.random.default_rng(n + 31 * dim + I)
    P = rng.standard_normal((I, dim)).astype(np.float32)
    X = rng.standard_normal((n, dim)).astype(np.float32)
    np.testing.assert_array_equal(engine_project(P, X), oracle.project(P, X))


# (partitions, k): one and several wavefronts, fewer and more list heads than threads, lists
# shorter than asked for, more entries below the bound than the buffer holds
@pytest.mark.parametrize("B,k", [(1, 1), (1, 64), (3, 32), (3, 33), (64, 32), (65, 32), (100, 1), (128, 16), (200, 10),
                                 (40, 100), (300, 128), (300, 256), (9, 256), (9, 257), (500, 40)])
@pytest.mark.parametrize("layout", ["mixed", "ordered"])
def test_merge_of_partition_lists(gpu, oracle, B, k, layout):
    rng = np.random.default_rng(B * 1000 + k)
    n, dim, nq, M, L, T, outer = 6000, 5, 6, 2, 3, 4, 30
    X = rng.standard_normal((n, dim)).astype(np.float32)
    Q = rng.standard_normal((nq, dim)).astype(np.float32)
    if layout == "ordered":      # a few partitions hold nearly all of a query's best
        X = X[np.argsort(X[:, 0], kind="stable")]
    dci = gpu.DCI(dim, M, L, B, T, seed=3, traversal="dense" if k <= 512 else "auto")
    dci.add(torch.from_numpy(X).cuda())
    qd = torch.from_numpy(Q).cuda()
    ids, dists = dci.query(qd, k, outer, return_int=True)
    fids, fdists = dci.query(qd, k, outer)
    skeys, sids = engine_index(dci)
    ref = oracle.query(skeys, sids, X, Q, engine_project(dci.directions.numpy(), Q).T.copy(), M, L, B, T, k, outer,
                       max_cand=10 * k)
    np.testing.assert_array_equal(ids.cpu().numpy(), ref["ids"])
    np.testing.assert_allclose(dists.cpu().numpy(), ref["dists"], rtol=1e-5, atol=1e-6)
    assert torch.equal(fids, ids.float()) and torch.equal(fdists, dists)
    dci.free()


# (points, dim, k, queries): pieces of a row, remainders, k up to and past the selection's limit
@pytest.mark.parametrize("n,dim,k,nq", [(1, 1, 1, 1), (2, 3, 2, 3), (63, 5, 63, 2), (300, 2, 256, 4), (300, 4, 257, 4),
                                        (4096, 33, 10, 5), (4097, 35, 10, 5), (4095, 7, 256, 2), (9001, 64, 100, 9),
                                        (12289, 130, 1, 3), (3000, 100, 200, 70)])
@pytest.mark.parametrize("kind", ["normal", "equal"])
def test_ranking_where_nothing_stops_early(gpu, oracle, n, dim, k, nq, kind):
    rng = np.random.default_rng(n + dim + k)
    X = rng.standard_normal((n, dim)).astype(np.float32)
    if kind == "equal":          # distances tie: ascending ids
        X[: n // 2] = X[0]
    Q = rng.standard_normal((nq, dim)).astype(np.float32)
    B = max(1, n // 8)
    dci = gpu.DCI(dim, 1, 2, B, 2, seed=1)
    dci.add(torch.from_numpy(X).cuda())
    ids, dists = dci.query(torch.from_numpy(Q).cuda(), k, 5000, return_int=True)
    d = np.zeros((nq, n), np.float32)
    for c in range(dim):
        t = X[None, :, c] - Q[:, c, None]
        d += t * t
    d = np.sqrt(d)
    order = np.lexsort((np.broadcast_to(np.arange(n), d.shape), d))[:, :k]
    np.testing.assert_array_equal(ids.cpu().numpy(), order)
    np.testing.assert_array_equal(dists.cpu().numpy(), np.take_along_axis(d, order, 1))
    dci.free()


# Items fewer than the device holds have workgroups of more wavefronts and larger tables: one item to a CU, up to four, and more.
@pytest.mark.parametrize("nq", [1, 4, 5, 17, 18, 29])
@pytest.mark.parametrize("M,L,T,k,outer", [(2, 10, 2, 10, 500), (2, 15, 3, 40, 50), (1, 30, 10, 1, 5000), (4, 16, 1, 5, 300)])
def test_items_of_more_wavefronts(gpu, nq, M, L, T, k, outer):
    from dciknn_cuda_amd import _capi
    gen = torch.Generator().manual_seed(nq)
    X = torch.randn(400011, 24, generator=gen).cuda()
    Q = torch.randn(150, 24, generator=gen).cuda()
    dci = gpu.DCI(24, M, L, 58, T, seed=3)
    dci.add(X)
    _capi.check(dci._lib.dcih_set_option(dci._dci_inst, _capi.OPT_ROUNDS, 1))      # every partition is traversed
    want = [t.clone() for t in dci.query(Q, k, outer, return_int=True)]
    for start in (0, 60):
        got = dci.query(Q[start:start + nq].contiguous(), k, outer, return_int=True)
        assert torch.equal(got[0], want[0][start:start + nq])
        assert torch.equal(got[1].view(torch.int32), want[1][start:start + nq].view(torch.int32))
    dci.free()
