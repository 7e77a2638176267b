"""Rows that hold NaN: their distances sort behind every finite one, and they take no finite
neighbour's place, whichever kernel answers."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


# (row length): rows read by 16 and by 32 lanes, one element at a time, and by their 8-bit codes
@pytest.mark.parametrize("dim", [64, 128, 67, 100, 300])
@pytest.mark.parametrize("ppb,B", [(1100, 1), (1100, 5), (4000, 3)])
@pytest.mark.parametrize("where", ["few", "scattered", "run"])
def test_kernels_agree(gpu, dim, ppb, B, where):
    rng = np.random.default_rng(ppb + B + dim)
    n, M, L, T, nq, outer = ppb * B, 2, 7, 10, 48, 5000
    X = rng.standard_normal((n, dim)).astype(np.float32)
    Q = rng.standard_normal((nq, dim)).astype(np.float32)
    bad = {"few": rng.choice(ppb, 2, replace=False), "scattered": rng.choice(n, n // 50, replace=False),
           "run": np.arange(ppb // 3, ppb // 3 + 200)}[where]
    X[bad, rng.integers(0, dim, len(bad))] = np.nan
    got = {}
    for traversal in ("step", "dense"):
        dci = gpu.DCI(dim, M, L, B, T, seed=3, traversal=traversal)
        dci.add(torch.from_numpy(X).cuda())
        qd = torch.from_numpy(Q).cuda()
        # (the later calls find the codes of the rows formed)
        got[traversal] = [dci.query(qd, k, outer, return_int=True) for k in (100, 100, 10)]
        dci.free()
    for (si, sd), (di, dd) in zip(got["step"], got["dense"]):
        finite = torch.isfinite(sd)
        wrong = (torch.isfinite(dd) != finite) | (finite & ((si != di) | (sd != dd)))
        assert not bool(wrong.any()), "queries %s" % wrong.any(1).nonzero().flatten().tolist()
