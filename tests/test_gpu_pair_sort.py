"""GPU parity of the row-major order of the stored pairs, at the counts and distributions where the sort takes another path:
one workgroup, one and two levels of buckets, buckets too full for the LDS, keys of more than 32 bits, the radix sort."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _coded(values):
    """Points of two coordinates below 2000 that stand for the integers `values`: equal points, and only those, are pairs."""
    import torch

    pts = torch.zeros((len(values), 64), dtype=torch.float16, device="cuda")
    v = torch.from_numpy(np.ascontiguousarray(values)).cuda()
    pts[:, 0] = (v // 2000).to(torch.float16)
    pts[:, 1] = (v % 2000).to(torch.float16)
    return pts, v


def _hub(n, row, share):
    q = np.arange(n) + 1
    q[row] = 0
    c = np.arange(n) + 1
    c[: int(n * share)] = 0
    return q, c


def _rand(nq, nc, distinct):
    rng = np.random.default_rng(nq + nc)
    return rng.integers(0, distinct, nq), rng.integers(0, distinct, nc)


CASES = {
    "two records": lambda: (np.array([7]), np.array([7, 7])),
    "the last count of one workgroup": lambda: (np.zeros(64, int), np.zeros(128, int)),
    "the first of one level": lambda: (np.zeros(1, int), np.zeros(8193, int)),
    "the last of one level": lambda: (np.zeros(1024, int), np.zeros(1024, int)),
    "the first of two levels": lambda: (np.zeros(1025, int), np.zeros(1024, int)),
    "a small join of runs": lambda: (np.arange(1000) // 8, np.arange(1000) // 8),
    "one level of runs": lambda: (np.arange(9000) // 90, np.arange(9000) // 90),
    "two levels of runs": lambda: (np.arange(40000) // 70, np.arange(40000) // 70),
    "one level, a crowded row": lambda: _hub(20011, 4321, 0.7),
    "two levels, a crowded row": lambda: tuple(np.concatenate(x) for x in zip(_hub(30011, 20000, 0.9), _rand(5000, 30000, 100))),
    "a row too crowded for one workgroup": lambda: tuple(np.concatenate(x) for x in zip(_hub(300, 7, 1.0), ([], np.zeros(1000000, int)))),
    "few records, long keys": lambda: _rand(40000, 70001, 500000),
    "many records, long keys": lambda: _rand(40000, 70001, 1501),
}


@pytest.mark.parametrize("name", list(CASES))
def test_sorted_pairs_are_row_major(name):
    import torch

    import fasted_amd as fasted
    from fasted_amd.find_pairs import FASTED_SORT_PAIRS

    qv, cv = (np.asarray(x).astype(np.int64) for x in CASES[name]())
    (q, vq), (c, vc) = _coded(qv), _coded(cv)
    rows = max(1, (1 << 28) // len(cv))
    want = torch.cat([torch.nonzero(vq[r : r + rows, None] == vc[None, :]) + torch.tensor([r, 0], device="cuda")
                      for r in range(0, len(qv), rows)]).to(torch.int32)
    pairs = torch.zeros((len(want) + 1, 2), dtype=torch.int32, device="cuda")
    for _ in range(2):  # the second call finds the tables as the first one left them
        st = fasted.join_device(q.data_ptr(), len(qv), 64, c.data_ptr(), len(cv), 64, 2, 0.5, pairs.data_ptr(), len(want) + 1,
                                flags=FASTED_SORT_PAIRS)
        assert st.pairsFound == st.pairsStored == len(want)
        assert torch.equal(pairs[:-1], want)
        assert int(pairs[-1].abs().sum()) == 0
