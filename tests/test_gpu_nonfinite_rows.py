"""Rows that hold NaN or infinite values: their distances sort behind every finite one, they take no
finite neighbour's place, and a window whose priority is not finite is never reached, whichever
kernel answers."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# (row length): rows read by 16 and by 32 lanes, one element at a time, and by their 8-bit codes
@pytest.mark.parametrize("dim", [64, 128, 67, 100, 300])
@pytest.mark.parametrize("ppb,B", [(1100, 1), (1100, 5), (4000, 3)])
@pytest.mark.parametrize("value", [np.nan, np.inf], ids=["nan", "inf"])
@pytest.mark.parametrize("where", ["few", "scattered", "run"])
# (windows of 10: ranked by radix passes where some priority is not finite; of 128: sorted as words)
@pytest.mark.parametrize("T", [10, 128])
def test_kernels_agree(gpu, dim, ppb, B, value, where, T):
    rng = np.random.default_rng(ppb + B + dim)
    n, M, L, nq, outer = ppb * B, 2, 7, 48, 5000
    X = rng.standard_normal((n, dim)).astype(np.float32)
    Q = rng.standard_normal((nq, dim)).astype(np.float32)
    bad = {"few": rng.choice(ppb, 2, replace=False), "scattered": rng.choice(n, n // 50, replace=False),
           "run": np.arange(ppb // 3, ppb // 3 + 200)}[where]
    X[bad, rng.integers(0, dim, len(bad))] = value
    got = {}
    for traversal in ("step", "dense", "batch"):
        dci = gpu.DCI(dim, M, L, B, T, seed=3, traversal=traversal)
        dci.add(torch.from_numpy(X).cuda())
        qd = torch.from_numpy(Q).cuda()
        # (the later calls find the codes of the rows formed)
        got[traversal] = [dci.query(qd, k, outer, return_int=True, return_counters=True) for k in (100, 100, 10)]
        dci.free()
    for other in ("dense", "batch"):
        for (si, sd, sc), (di, dd, dc) in zip(got["step"], got[other]):
            finite = torch.isfinite(sd)
            wrong = (torch.isfinite(dd) != finite) | (finite & ((si != di) | (sd != dd)))
            assert not bool(wrong.any()), "%s: queries %s" % (other, wrong.any(1).nonzero().flatten().tolist())
            # candidates and steps
            assert torch.equal(sc[:, [1, 3]], dc[:, [1, 3]]), other
