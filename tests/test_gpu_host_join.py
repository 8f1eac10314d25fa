"""GPU parity of the host-to-host join's way up: rows that need padding or none, odd dimensionalities, rows that go up in
several pieces, and the buffer kept from call to call, for larger and smaller joins than the one that left it."""
import ctypes

import numpy as np
import pytest

import oracle
from tests import datasets

pytestmark = pytest.mark.gpu


def _self_join(bits, eps, cap):
    import fasted_amd as fasted

    lib = fasted.load_findpairs()
    found, stored = ctypes.c_ulonglong(), ctypes.c_ulonglong()
    out = np.full((cap, 2), -1, dtype=np.int32)
    rc = lib.fasted_self_join(bits.ctypes.data, bits.shape[0], bits.shape[1], eps, out.ctypes.data, cap, ctypes.byref(found),
                              ctypes.byref(stored))
    return rc, out[: stored.value], found.value


def _case(n, d):
    """Integer coordinates and an epsilon with about eight neighbours a point whose square lies half-way between two integers."""
    bits = datasets.small_integers(n, d, high=3, seed=n + d)
    eps = datasets.epsilon_for_neighbours(bits, min(8, n - 1) or 1, sample=128) if n > 1 else 1.0
    return bits, float(np.sqrt(np.floor(eps * eps) + 0.5))


# one row; odd, even and multiple-of-8 padding; no padding; more than 32 MB of packed rows and fewer of pairs (two pieces)
@pytest.mark.parametrize("n,d", [(1, 1), (300, 3), (2000, 63), (2000, 64), (2001, 66), (1500, 72), (1000, 129), (70001, 250)])
def test_host_join_equals_device_join(n, d):
    import torch

    import fasted_amd as fasted
    from fasted_amd.find_pairs import FASTED_FULL_MATRIX, FASTED_SORT_PAIRS

    bits, eps = _case(n, d)
    ld = (d + 63) // 64 * 64
    pts = torch.zeros((n, ld), dtype=torch.int16, device="cuda")
    pts[:, :d] = torch.from_numpy(bits.view(np.int16)).cuda()
    count = int(fasted.self_join_device(pts.data_ptr(), n, d, ld, eps, None, 0, flags=0).pairsFound)
    assert n == 1 or count > 2 * n  # what is checked is not the diagonal alone
    pairs = torch.zeros((count + 1, 2), dtype=torch.int32, device="cuda")
    st = fasted.self_join_device(pts.data_ptr(), n, d, ld, eps, pairs.data_ptr(), count + 1,
                                 flags=FASTED_SORT_PAIRS | FASTED_FULL_MATRIX)
    assert st.pairsFound == st.pairsStored == count
    want = pairs[:-1].cpu().numpy()
    if n <= 2001:
        assert np.array_equal(want, oracle.self_join_f64(bits, eps))
    small, small_eps = _case(200, 65)
    small_want = oracle.self_join_f64(small, small_eps)
    for release in (False, False, True):
        if release:
            fasted.load_findpairs().releaseResources()
        rc, got, found = _self_join(bits, eps, count + 1)
        assert rc == 0 and found == count and np.array_equal(got, want)
        rc, got, found = _self_join(bits, eps, count // 2 or 1)  # room for some of them only
        assert rc == 0 and found == count and len(got) == (count // 2 or 1)
        rc, got, _ = _self_join(small, small_eps, len(small_want))
        assert rc == 0 and np.array_equal(got, small_want)


def test_host_join_after_one_that_was_refused():
    bits, eps = _case(500, 70)
    want = oracle.self_join_f64(bits, eps)
    for _ in range(2):
        rc, _, _ = _self_join(bits, float("nan"), len(want))
        assert rc != 0
        rc, got, found = _self_join(bits, eps, len(want))
        assert rc == 0 and found == len(want) and np.array_equal(got, want)


# lists that come down in one copy and in pinned pieces of 2 MB: a record short of 4 MB and as much, whole pieces, a piece and a
# record, many; in one go and in blocks of rows
@pytest.mark.parametrize("n,cap", [(725, 524287), (725, 524288), (725, 525625), (900, 786432), (900, 786433), (2900, 2900 * 2900)])
@pytest.mark.parametrize("block", [0, 512])
def test_long_lists_come_down_whole(n, cap, block):
    import fasted_amd as fasted

    bits = datasets.small_integers(n, 5, high=3, seed=n)
    lib = fasted.load_findpairs()
    found, stored = ctypes.c_ulonglong(), ctypes.c_ulonglong()
    want = np.stack(np.divmod(np.arange(cap, dtype=np.int32), np.int32(n)), 1)
    for _ in range(2):
        out = np.full((cap + 1, 2), -1, dtype=np.int32)
        args = (out.ctypes.data, cap, ctypes.byref(found), ctypes.byref(stored))
        if block:
            rc = lib.fasted_self_join_blocked(bits.ctypes.data, n, 5, float("inf"), block, *args)
        else:
            rc = lib.fasted_self_join(bits.ctypes.data, n, 5, float("inf"), *args)
        assert rc == 0
        if not block:
            assert found.value == n * n and stored.value == cap
            assert np.array_equal(out[:cap], want) and (out[cap] == -1).all()
        else:
            # (a block of rows keeps 256 pairs per point: as many of its pairs as that, in order)
            got = out[: stored.value]
            assert found.value == n * n and stored.value == min(cap, 256 * 512 * -(-n // 512))
            keys = got[:, 0].astype(np.int64) * n + got[:, 1]
            assert (np.diff(keys) > 0).all() and got.min() >= 0 and got.max() < n and (out[stored.value :] == -1).all()
