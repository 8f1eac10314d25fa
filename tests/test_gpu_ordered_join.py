"""GPU parity of sorted joins of few points, whose list is made from hit bits: where the number of bands, words and tiles
changes, few and all elements a hit, lists longer than their buffer, and the first size that is sorted instead."""
import pytest

pytestmark = pytest.mark.gpu


def _points(n, d, high, seed):
    import torch

    gen = torch.Generator(device="cuda").manual_seed(seed)
    ld = (d + 63) // 64 * 64
    pts = torch.zeros((n, ld), dtype=torch.float16, device="cuda")
    pts[:, :d] = torch.randint(0, high, (n, d), generator=gen, device="cuda").to(torch.float16)
    return pts, ld


def _want(q, c, eps2):
    """Row-major list of the pairs of integer points within a squared distance: every sum is exact in FP32."""
    import torch

    x, y = q.float(), c.float()
    sx, sy = (x * x).sum(1), (y * y).sum(1)
    rows = [torch.nonzero(sx[r : r + 2048, None] + sy[None, :] - 2.0 * (x[r : r + 2048] @ y.T) <= eps2) + torch.tensor([r, 0], device="cuda")
            for r in range(0, len(x), 2048)]
    return torch.cat(rows).to(torch.int32)


# share of the elements that are hits: hardly any, some, nearly all, all
@pytest.mark.parametrize("share", [0.0, 0.01, 0.9, 1.0])
@pytest.mark.parametrize("n,d", [(1, 5), (2, 64), (31, 64), (32, 65), (33, 1100), (255, 64), (257, 130), (1000, 64), (2049, 1100), (2817, 40),
                                 (4096, 64), (4097, 1030)])
def test_lists_of_every_density(n, d, share):
    import torch

    import fasted_amd as fasted
    from fasted_amd import find_pairs as fp

    pts, ld = _points(n, d, 9 if d < 300 else 3, n + d)
    x = pts[: min(n, 64)].double()
    d2 = torch.cdist(x, pts.double()).square().round().flatten().sort().values
    eps2 = float(d2[min(len(d2) - 1, int(share * len(d2)))]) + 0.5
    want = _want(pts, pts, eps2)
    cap = len(want) + 3
    for flags in (0, fp.FASTED_FULL_MATRIX, fp.FASTED_SYMMETRIC, fp.FASTED_EVENT_TIMING):
        pairs = torch.full((cap, 2), -1, dtype=torch.int32, device="cuda")
        st = fasted.self_join_device(pts.data_ptr(), n, d, ld, eps2**0.5, pairs.data_ptr(), cap, flags=flags | fp.FASTED_SORT_PAIRS)
        assert st.pairsFound == st.pairsStored == len(want), flags
        assert torch.equal(pairs[: len(want)], want) and bool((pairs[len(want) :] == -1).all()), flags
        # the list is part of the join, and 8 bytes a pair take their time at 8 TB/s
        assert st.joinMs > len(want) * 8 / 8e9 and st.sumSquaredMs > 0 and st.sortMs == 0
    # a buffer that is too small holds the beginning of the list; what lies behind it is left alone
    small = max(1, len(want) // 3)
    pairs = torch.full((cap, 2), -1, dtype=torch.int32, device="cuda")
    st = fasted.self_join_device(pts.data_ptr(), n, d, ld, eps2**0.5, pairs.data_ptr(), small, flags=fp.FASTED_SORT_PAIRS)
    assert st.pairsFound == len(want) and st.pairsStored == small
    assert torch.equal(pairs[:small], want[:small]) and bool((pairs[small:] == -1).all())


@pytest.mark.parametrize("rows", [None, "256", "128"])
@pytest.mark.parametrize("nq,nc,d", [(1, 20224, 64), (20224, 1, 40), (33, 9000, 100), (9000, 33, 1100), (3000, 5000, 64), (20224, 700, 65),
                                     (20225, 700, 65), (700, 20225, 65)])
def test_two_sets(nq, nc, d, rows, monkeypatch):
    """Both sides up to the last size that leaves hit bits, and one past it on either side; both tile heights."""
    import torch

    import fasted_amd as fasted
    from fasted_amd import find_pairs as fp

    if rows:
        monkeypatch.setenv("FASTED_TILE_ROWS", rows)
    (q, ld), (c, _) = _points(nq, d, 4, 1), _points(nc, d, 4, 2)
    d2 = torch.cdist(q[:64].double(), c[:64].double()).square().round().flatten()
    eps2 = float(d2.quantile(0.05).round()) + 0.5
    want = _want(q, c, eps2)
    cap = len(want) + 3
    pairs = torch.full((cap, 2), -1, dtype=torch.int32, device="cuda")
    for _ in range(2):
        st = fasted.join_device(q.data_ptr(), nq, ld, c.data_ptr(), nc, ld, d, eps2**0.5, pairs.data_ptr(), cap, flags=fp.FASTED_SORT_PAIRS)
        assert st.pairsFound == st.pairsStored == len(want)
        assert torch.equal(pairs[: len(want)], want)


@pytest.mark.parametrize("n", [20224, 20225])
@pytest.mark.parametrize("rows", [None, "128"])
def test_the_last_size_in_bits_and_the_next(n, rows, monkeypatch):
    import torch

    import fasted_amd as fasted
    from fasted_amd import find_pairs as fp

    if rows:
        monkeypatch.setenv("FASTED_TILE_ROWS", rows)
    d = 72
    pts, ld = _points(n, d, 4, 3)
    eps2 = float(torch.cdist(pts[:64].double(), pts.double()).square().round().flatten().kthvalue(64 * 20).values) + 0.5
    want = _want(pts, pts, eps2)
    pairs = torch.full((len(want) + 3, 2), -1, dtype=torch.int32, device="cuda")
    # an unsorted join in between: the counters of the bands are cleared by every join
    for flags in (fp.FASTED_SORT_PAIRS, 0, fp.FASTED_SORT_PAIRS, fp.FASTED_SORT_PAIRS | fp.FASTED_FULL_MATRIX):
        st = fasted.self_join_device(pts.data_ptr(), n, d, ld, eps2**0.5, pairs.data_ptr(), len(pairs), flags=flags)
        assert st.pairsFound == st.pairsStored == len(want), flags
        if flags & fp.FASTED_SORT_PAIRS:
            assert torch.equal(pairs[: len(want)], want), flags


def test_points_that_are_not_finite():
    """A point with an infinite or NaN coordinate pairs with nothing but itself."""
    import torch

    import fasted_amd as fasted

    n, d = 2900, 100
    pts, ld = _points(n, d, 3, 4)
    eps2 = float(torch.cdist(pts[:64].double(), pts.double()).square().round().flatten().kthvalue(64 * 20).values) + 0.5
    want = _want(pts, pts, eps2).long()
    bad = torch.tensor([0, 31, 256, 2899], device="cuda")
    pts[bad, torch.tensor([0, 50, 99, 7], device="cuda")] = torch.tensor([float("inf"), float("nan"), float("-inf"), float("nan")],
                                                                        dtype=torch.float16, device="cuda")
    keep = ~(torch.isin(want, bad).any(1)) | (want[:, 0] == want[:, 1])
    want = want[keep].to(torch.int32)
    pairs = torch.full((len(want) + 3, 2), -1, dtype=torch.int32, device="cuda")
    st = fasted.self_join_device(pts.data_ptr(), n, d, ld, eps2**0.5, pairs.data_ptr(), len(pairs))
    assert st.pairsFound == len(want) and torch.equal(pairs[: len(want)], want)
