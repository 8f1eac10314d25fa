"""GPU parity of the row-major order of the stored pairs, at the counts and distributions where the sort takes another path:
one workgroup, one and two levels of buckets, buckets too full for the LDS, crowded cells, keys of more than 32 bits, lists
that a level breaks off, the radix sort behind them.  tests/test_sort_routes.py holds the lists to these paths, and to more
points than a join may have whose list is made in order without a sort."""
import ctypes

import numpy as np
import pytest

from tests import sort_routes

pytestmark = pytest.mark.gpu


def _coded(values):
    """Points of two coordinates below 2000 that stand for the integers `values`: equal points, and only those, are pairs."""
    import torch

    pts = torch.zeros((len(values), 64), dtype=torch.float16, device="cuda")
    v = torch.from_numpy(np.ascontiguousarray(values)).cuda()
    pts[:, 0] = (v // 2000).to(torch.float16)
    pts[:, 1] = (v % 2000).to(torch.float16)
    return pts, v


MAX_BIT_ROWS = 20224  # points of either side up to which no sort follows the join


def _to_be_sorted(q, c):
    """The same pairs, in a join of enough candidates that they are sorted."""
    return q, np.concatenate([c, 3000000 + np.arange(MAX_BIT_ROWS + 1 - len(c))])


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
    "two records": lambda: _to_be_sorted(np.array([7]), np.array([7, 7])),
    "the last count of one workgroup": lambda: _to_be_sorted(np.zeros(64, int), np.zeros(128, int)),
    "the first of one level": lambda: _to_be_sorted(np.zeros(1, int), np.zeros(8193, int)),
    "the last of one level": lambda: _to_be_sorted(np.zeros(1024, int), np.zeros(1024, int)),
    "the first of two levels": lambda: _to_be_sorted(np.zeros(1025, int), np.zeros(1024, int)),
    "a small join of runs": lambda: _to_be_sorted(np.arange(1000) // 8, np.arange(1000) // 8),
    "one level of runs": lambda: _to_be_sorted(np.arange(9000) // 90, np.arange(9000) // 90),
    "two levels of runs": lambda: (np.arange(40000) // 70, np.arange(40000) // 70),
    "one level, a crowded row": lambda: _to_be_sorted(*_hub(20011, 4321, 0.7)),
    "two levels, a crowded row": lambda: tuple(np.concatenate(x) for x in zip(_hub(30011, 20000, 0.9), _rand(5000, 30000, 100))),
    "a row too crowded for one workgroup": lambda: tuple(np.concatenate(x) for x in zip(_hub(300, 7, 1.0), ([], np.zeros(1000000, int)))),
    "few records, long keys": lambda: _rand(40000, 70001, 500000),
    "many records, long keys": lambda: _rand(40000, 70001, 1501),
}


def _check(qv, cv, calls=2):
    """The sorted join of the coded sets against the pairs computed here; the shortest of its sorts, in milliseconds."""
    import torch

    import fasted_amd as fasted
    from fasted_amd.find_pairs import FASTED_SORT_PAIRS

    qv, cv = np.asarray(qv).astype(np.int64), np.asarray(cv).astype(np.int64)
    (q, vq), (c, vc) = _coded(qv), _coded(cv)
    rows = max(1, (1 << 28) // len(cv))
    want = torch.cat([torch.nonzero(vq[r : r + rows, None] == vc[None, :]) + torch.tensor([r, 0], device="cuda")
                      for r in range(0, len(qv), rows)]).to(torch.int32)
    pairs = torch.zeros((len(want) + 1, 2), dtype=torch.int32, device="cuda")
    sort_ms = []
    for _ in range(calls):  # a second call finds the tables as the first one left them
        st = fasted.join_device(q.data_ptr(), len(qv), 64, c.data_ptr(), len(cv), 64, 2, 0.5, pairs.data_ptr(), len(want) + 1,
                                flags=FASTED_SORT_PAIRS)
        assert st.pairsFound == st.pairsStored == len(want)
        assert torch.equal(pairs[:-1], want)
        assert int(pairs[-1].abs().sum()) == 0
        assert st.sortMs > 0  # the list was sorted, not made in order
        sort_ms.append(st.sortMs)
    return min(sort_ms)


@pytest.mark.parametrize("name", list(CASES))
def test_sorted_pairs_are_row_major(name):
    _check(*CASES[name]())


def _groups(n, per):
    """Two sets of n points in which every query has `per` candidates on average, anywhere."""
    rng = np.random.default_rng(n)
    small, large = int(per), int(per) + 1
    split = int(n * (large - per))
    v = np.concatenate([np.arange(split) // small, n + np.arange(n - split) // large])
    return rng.permutation(v), rng.permutation(v)


def _core():
    """100 000 queries with two candidates each, but 2000 neighbouring ones with 200."""
    rng = np.random.default_rng(1)
    q = rng.permutation(np.arange(98000) // 2)
    core = 100000 + np.arange(2000) % 10
    return np.concatenate([q[:50000], core, q[50000:]]), rng.permutation(np.concatenate([q, core]))


# lists on both sides of the line between one level and two, and one that crowds into a few rows
SPARSE = {
    "0.97 million in 130 000 rows": lambda: _groups(130000, 7.46),
    "1.04 million in 130 000 rows": lambda: _groups(130000, 8.04),
    "1.0 million in 200 000 rows": lambda: _groups(200000, 5.0),
    "1.04 million in 250 000 rows": lambda: _groups(250000, 4.18),
    "1.1 million in 250 000 rows": lambda: _groups(250000, 4.4),
    "a crowded core": _core,
}


@pytest.mark.parametrize("name", list(SPARSE))
def test_sparse_lists_are_sorted_at_the_rate_of_others(name):
    # buckets that outgrow the LDS cost 30 to 100 times this; the lists here take 1.0 to 1.8 times as long
    even = _check(*_groups(100000, 6.0), calls=6)
    assert _check(*SPARSE[name](), calls=6) < 5 * even


@pytest.mark.parametrize("name", list(sort_routes.CASES))
def test_crowded_lists_are_row_major_and_leave_the_sort_as_it_was(name):
    import torch

    import fasted_amd as fasted
    from fasted_amd.find_pairs import FASTED_SORT_PAIRS

    ordinary = _groups(30000, 10.0)
    for qv, cv in (sort_routes.CASES[name][0](), ordinary, sort_routes.CASES[name][0]()):
        want = torch.from_numpy(sort_routes.pairs_of(qv, cv)).cuda()
        (q, _), (c, _) = _coded(qv), _coded(cv)
        pairs = torch.zeros((len(want) + 1, 2), dtype=torch.int32, device="cuda")
        st = fasted.join_device(q.data_ptr(), len(qv), 64, c.data_ptr(), len(cv), 64, 2, 0.5, pairs.data_ptr(), len(want) + 1,
                                flags=FASTED_SORT_PAIRS)
        assert st.pairsFound == st.pairsStored == len(want)
        assert torch.equal(pairs[:-1], want)
        assert int(pairs[-1].abs().sum()) == 0
        assert st.sortMs > 0


def test_crowded_rows_of_a_later_query_block_are_row_major():
    # 24 blocks of query points; 4500 equal points, some in every block, whose rows are too full for the LDS
    import fasted_amd as fasted

    n, block = 24 * 4096, 4096
    v = np.arange(n) + 1
    v[np.random.default_rng(3).permutation(n)[:4500]] = 0
    want = sort_routes.pairs_of(v, v)
    bits = np.zeros((n, 64), dtype=np.float16)
    bits[:, 0], bits[:, 1] = v // 2000, v % 2000
    for r in range(0, n, block):
        mine = want[(want[:, 0] >= r) & (want[:, 0] < r + block)] - np.array([r, 0])
        assert {"one level", "windows"} <= sort_routes.route(mine, block, n)
    lib = fasted.load_findpairs()
    found, stored = ctypes.c_ulonglong(), ctypes.c_ulonglong()
    out = np.full((len(want) + 1, 2), -1, dtype=np.int32)
    rc = lib.fasted_self_join_blocked(bits.ctypes.data, n, 64, 0.5, block, out.ctypes.data, len(out), ctypes.byref(found),
                                      ctypes.byref(stored))
    assert rc == 0, lib.fasted_last_error()
    assert found.value == stored.value == len(want)
    assert np.array_equal(out[:-1], want) and (out[-1] == -1).all()
