"""GPU parity of the host-to-host join's way up: rows that need padding or none, odd dimensionalities, rows that go up in
several pieces, the buffer kept from call to call, and a call that fails in between."""
import ctypes

import numpy as np
import pytest

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


# one row; odd, even and multiple-of-8 padding; no padding; more than 32 MB of packed rows (two pieces, as no pair list is longer)
@pytest.mark.parametrize("n,d", [(1, 1), (300, 3), (2000, 63), (2000, 64), (2001, 66), (1500, 72), (1000, 129), (70001, 250)])
def test_host_join_equals_device_join(n, d):
    import torch

    import fasted_amd as fasted
    from fasted_amd.find_pairs import FASTED_SORT_PAIRS

    bits = datasets.small_integers(n, d, high=3, seed=n + d)
    ld = (d + 63) // 64 * 64
    pts = torch.zeros((n, ld), dtype=torch.int16, device="cuda")
    pts[:, :d] = torch.from_numpy(bits.view(np.int16)).cuda()
    eps = float(np.sqrt(max(1.0, d * 0.6) + 0.5))  # below the typical squared distance, half-way between two integers
    cap = 2 * n + 1000
    pairs = torch.zeros((cap, 2), dtype=torch.int32, device="cuda")
    st = fasted.self_join_device(pts.data_ptr(), n, d, ld, eps, pairs.data_ptr(), cap, flags=FASTED_SORT_PAIRS)
    for _ in range(2):
        rc, got, found = _self_join(bits, eps, cap)
        assert rc == 0 and found == st.pairsFound and len(got) == st.pairsStored
        if st.pairsFound <= cap:
            assert np.array_equal(got, pairs[: st.pairsStored].cpu().numpy())
        rc, _, _ = _self_join(bits, float("nan"), cap)
        assert rc != 0
    fasted.load_findpairs().releaseResources()
    rc, got, found = _self_join(bits, eps, cap)
    assert rc == 0 and found == st.pairsFound
