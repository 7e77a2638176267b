"""The build's sort of slices of 65 to 25600 projections (csrc/bucketsort.hip) and what it leaves to the sort by digits: exactly the
order by (key, id), whatever the keys."""
import numpy as np
import pytest
import torch

from util import engine_index, engine_segsort

pytestmark = pytest.mark.gpu

KINDS = ["normal", "clusters", "far", "heavy", "ties", "few", "zeros", "descending", "nonfinite"]


def _keys(kind, rng, rows, n):
    x = rng.standard_normal((rows, n)).astype(np.float32)
    if kind == "clusters":
        x = x + 1000.0 * rng.integers(-3, 4, (rows, n))
    elif kind == "far":
        x[:, ::97] *= 1e7
    elif kind == "heavy":
        x = x / rng.standard_normal((rows, n))
    elif kind == "ties":
        x = np.round(x * n / 8)
    elif kind == "few":
        x = rng.integers(0, 3, (rows, n))
    elif kind == "zeros":
        x = np.where(rng.random((rows, n)) < 0.3, rng.choice([0.0, -0.0], (rows, n)), x)
    elif kind == "descending":
        x = -np.sort(x, axis=1)
    elif kind == "nonfinite":
        x[:, ::61] = np.inf
        x[:, 5::83] = -np.inf
    return np.ascontiguousarray(x, dtype=np.float32)


def _sorted(keys, block_size):
    rows, n = keys.shape
    per = -(-n // block_size)
    out_k, out_i = np.empty_like(keys), np.empty(keys.shape, np.int32)
    for a in range(0, n, per):
        b = min(n, a + per)
        order = np.argsort(keys[:, a:b] + np.float32(0), axis=1, kind="stable")
        out_k[:, a:b] = np.take_along_axis(keys[:, a:b] + np.float32(0), order, axis=1)
        out_i[:, a:b] = order + a
    return out_k, out_i


# the most points of every workgroup shape and one more, and the ends of the range
@pytest.mark.parametrize("per", [64, 65, 320, 321, 576, 577, 832, 1088, 1344, 1345, 2304, 3329, 4352, 4353, 8704, 8961, 10753, 12800, 12801,
                                 13313, 17408, 21505, 25600, 25601])
def test_slices_come_out_in_order(gpu, per):
    rng = np.random.default_rng(per)
    for kind in KINDS:
        block_size = 3
        keys = _keys(kind, rng, 3, block_size * per - 2)             # the last slice is shorter, the rows start on any 4-byte boundary
        got_k, got_i = engine_segsort(keys, block_size)
        want_k, want_i = _sorted(keys, block_size)
        np.testing.assert_array_equal(got_i, want_i, err_msg=kind)
        np.testing.assert_array_equal(got_k.view(np.uint32), want_k.view(np.uint32), err_msg=kind)


@pytest.mark.parametrize("n,block_size", [(1000, 7), (4001, 3), (30000, 2), (17000, 1), (60001, 3)])
def test_positions_are_the_inverse(gpu, n, block_size):
    from dciknn_cuda_amd import _capi
    rng = np.random.default_rng(n)
    x = rng.standard_normal((n, 12)).astype(np.float32)
    x[: n // 3] = x[0]                                               # a third of the rows are one row
    dci = gpu.DCI(12, 2, 3, block_size, 2, seed=3)
    rows = torch.from_numpy(x).cuda()
    for again in range(2):                                           # (a handle that lives on)
        dci.add(rows)
        inv = torch.zeros((6, n), dtype=torch.int16, device="cuda")
        _capi.check(dci._lib.dcih_debug_positions(dci._dci_inst, inv.data_ptr(), None, None))
        keys, ids = engine_index(dci)
        per = -(-n // block_size)
        pos = inv.cpu().numpy().view(np.uint16).astype(np.int64)
        place = np.arange(n) % per
        for i in range(6):
            np.testing.assert_array_equal(pos[i][ids[i]], place)
            for a in range(0, n, per):
                assert (np.diff(keys[i, a:a + per]) >= 0).all()
        dci.clear()
    dci.free()
