"""Items of a call in rounds that are answered by their near rows alone (confirm.hip), against the same queries traversed as a whole: ids and
distances must be equal to the bit, whatever is answered and whatever is left.  Shapes at the edges of its tables and of the variants: one
wavefront to an item and the rest by eight, four wavefronts, windows alone; slices that start on no 16-byte boundary, rows of less than 32 elements,
past 128, not of whole 16-byte words; one, two and eight composites; windows of one point; near rows that repeat, that no composite promotes,
that come before and after the stop."""
import pytest
import torch

from test_gpu_rounds import ALWAYS, NEVER, _ask, _rows

pytestmark = pytest.mark.gpu


def _confirmed(dci):
    from dciknn_cuda_amd import _capi
    counts = (_capi.ctypes.c_uint32 * 2)()
    _capi.check(dci._lib.dcih_debug_confirmed(dci._dci_inst, counts))
    return tuple(counts)


# n, dim, M, L, B, T, k, outer, queries
SHAPES = {
    "defaults": (20000, 64, 2, 7, 50, 10, 10, 5000, 300),
    "narrow": (30000, 128, 2, 10, 20, 2, 10, 500, 1500),
    "many": (24001, 40, 2, 6, 48, 4, 4, 2000, 3000),
    "odd": (12347, 67, 3, 5, 37, 3, 7, 1000, 200),
    "long": (6000, 300, 2, 7, 30, 5, 6, 5000, 120),
    "short": (9000, 20, 1, 2, 30, 1, 5, 60, 150),
    "eight": (16000, 33, 8, 4, 16, 7, 12, 300, 90),
    "wide": (36000, 48, 2, 15, 60, 128, 30, 10, 100),
    "results": (24000, 30, 2, 5, 16, 6, 90, 5000, 100),
}


@pytest.mark.parametrize("kind", ["clusters", "normal", "sorted", "dup", "grid", "broken", "offset", "tiny"])
@pytest.mark.parametrize("shape", list(SHAPES), ids=list(SHAPES))
def test_same_as_whole(gpu, shape, kind):
    n, dim, M, L, B, T, k, outer, nq = SHAPES[shape]
    X, Q = _rows(kind, n, nq, dim, n + dim)
    dci = gpu.DCI(dim, M, L, B, T, seed=9)
    dci.add(X)
    want = _ask(dci, dci._lib, NEVER, Q, k, outer)
    assert _confirmed(dci) == (0, 0)
    for again in range(3):      # with nothing on record, and with what the calls before left there
        got = _ask(dci, dci._lib, ALWAYS, Q, k, outer)
        assert torch.equal(got[0], want[0]), again
        assert torch.equal(got[1].view(torch.int32), want[1].view(torch.int32)), again
    answered, left = _confirmed(dci)
    dci.free()
    assert answered + left > 0
    if kind == "clusters" and shape != "results":      # rows whose nearest are promoted first
        assert answered > left, (answered, left)


@pytest.mark.parametrize("dim", [40, 64, 128, 132])
@pytest.mark.parametrize("per,nq", [(600, 3), (900, 3), (600, 20)])
def test_a_distance_that_is_not_a_number_limits_nothing(gpu, dim, per, nq):
    """A query whose k-th result so far has the distance NaN takes rows at any distance in the rounds that follow.  Two clusters 200 times as far
    apart as they are wide, so that round 1's limit, a bound, lies below the distances of all but a few finite rows; rows that are not finite,
    which are promoted with windows that begin with a finite projection, stand at the k-th place until then."""
    B, k = 24, 8
    X, Q = _rows("normal", B * per, nq, dim, per + dim)
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    for rows in (X, Q):
        rows += 200.0 * torch.randint(0, 2, (len(rows), 1), generator=g, device="cuda") - 100.0
    X[7:31, 3] = float("nan")
    dci = gpu.DCI(dim, 1, 2, B, 64, seed=4)
    dci.add(X)
    want = _ask(dci, dci._lib, NEVER, Q, k, 5000)
    assert torch.isfinite(want[1]).all()
    for again in range(2):
        got = _ask(dci, dci._lib, ALWAYS, Q, k, 5000)
        assert _confirmed(dci)[0] > 0
        assert torch.equal(got[0], want[0]), again
        assert torch.equal(got[1].view(torch.int32), want[1].view(torch.int32)), again
    dci.free()
