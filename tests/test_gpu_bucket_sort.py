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


def _copies(rng, rows, n, of):
    """Each key `of` times, one after the other: more than a bucket may hold."""
    return np.ascontiguousarray(np.repeat(rng.standard_normal((rows, -(-n // of))), of, axis=1)[:, :n], dtype=np.float32)


# the ends of every shape that sorts what is left
@pytest.mark.parametrize("per", [65, 100, 128, 129, 1345, 1600, 1601, 2112, 2113, 2688, 2689, 3456, 3457, 4224, 4225, 5376, 5377, 6912, 6913, 8960])
def test_copies_of_rows(gpu, per):
    """Slices of which none, some and all are left."""
    rng = np.random.default_rng(per)
    keys = _copies(rng, 3, 4 * per - 1, 32)
    keys[1] = rng.standard_normal(keys.shape[1])
    keys[2, per:2 * per] = rng.standard_normal(per)
    got_k, got_i = engine_segsort(keys, 4)
    want_k, want_i = _sorted(keys, 4)
    np.testing.assert_array_equal(got_i, want_i)
    np.testing.assert_array_equal(got_k.view(np.uint32), want_k.view(np.uint32))


@pytest.mark.parametrize("per,block_size", [(80, 12000), (300, 5000), (2200, 1500)])
def test_copies_of_rows_in_many_slices(gpu, per, block_size):
    """More of them than workgroups start."""
    rng = np.random.default_rng(per)
    n = per * block_size
    keys = _copies(rng, 2, n, 32)
    keys[1, n // 2:] = rng.standard_normal(n - n // 2)
    got_k, got_i = engine_segsort(keys, block_size)
    want = keys.reshape(2, block_size, per)
    order = np.argsort(want, axis=2, kind="stable")
    np.testing.assert_array_equal(got_i.reshape(2, block_size, per), order + per * np.arange(block_size)[None, :, None])
    np.testing.assert_array_equal(got_k.reshape(2, block_size, per), np.take_along_axis(want, order, axis=2))


def test_copies_of_rows_cost_no_multiple(gpu):
    """All slices left: the attempt and the sort by digits, about three times as long here as where none is left (twelve times when few workgroups
    shared them, each with room for slices six times as long)."""
    from dciknn_cuda_amd import _capi
    rows, n, block_size = 20, 500_000, 5000
    gen = torch.Generator(device="cuda").manual_seed(1)
    plain = torch.randn(rows, n, generator=gen, device="cuda")
    copies = plain[:, :n // 32 + 1].repeat_interleave(32, 1)[:, :n].contiguous()
    out = torch.empty_like(plain), torch.empty(plain.shape, dtype=torch.int32, device="cuda")

    def best(keys):
        times = []
        for _ in range(8):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            _capi.check(_capi.lib().dcih_segsort(keys.data_ptr(), rows, n, block_size, out[0].data_ptr(), out[1].data_ptr(),
                                                 torch.cuda.current_stream().cuda_stream))
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)
    a, b = best(plain), best(copies)
    assert b < 7 * a, (a, b)
