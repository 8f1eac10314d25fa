"""GPU parity tests of mid-size matrices: more tiles than two rounds of the workgroups (so the tiles come from the
per-XCD work queues, not one workgroup per tile), in strips and in super-squares, several slabs per tile.  A sorted join of
up to 20 224 points leaves hit bits, an unsorted one stages its pairs: other kernels, so both are asked for.  The size band of the reference's own sweep rows of 10 000 and 21 544 points
(results/speed_results/ExpoDataSpeedVsSize_OnDemandRasterizer.json); kernel counterpart
source/findPairs.cuh:360-546 with source/rasterizer/onDemandRasterizer.cuh:78-108."""
import numpy as np
import pytest

import oracle
from tests import datasets

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fasted():
    import fasted_amd

    fasted_amd.load_findpairs()
    return fasted_amd


def integer_case(n, d, seed, rank=10):
    """Integer coordinates (every product and sum exact in FP32) and an epsilon whose square lies half-way between
    two integers: the pair list must equal the FP64 checker's record for record."""
    bits = datasets.small_integers(n, d, high=3, seed=seed)
    x = bits[:64].view(np.float16).astype(np.float64)
    d2 = ((x[:, None, :] - x[None, :, :]) ** 2).sum(-1)
    eps = float(np.sqrt(np.sort(d2[np.triu_indices(64, 1)])[rank] + 0.5))
    return bits, eps


@pytest.mark.parametrize("n,d", [(7000, 128), (7000, 320), (12000, 128), (12000, 320), (6000, 1088)])
def test_queue_mode_exact_pair_lists(fasted, n, d, monkeypatch):
    """784 and 2209 tiles of 256 rows (1540 and 4418 of 128 rows), in strips, and 17 slabs (hit bits behind the k-loop):
    the library's choice, the full matrix and the triangle, both tile heights, with and without squared norms brought by
    the caller, sorted and not."""
    import torch
    from fasted_amd import find_pairs as fp

    bits, eps = integer_case(n, d, seed=n + d)
    truth = oracle.self_join_f64(bits, eps)
    assert len(truth) > 2 * n  # off-diagonal pairs are what is being checked
    pts = torch.from_numpy(bits.view(np.int16).copy()).cuda()
    cap = len(truth) + 1024
    pairs = torch.empty((cap, 2), dtype=torch.int32, device="cuda")
    sums = torch.empty(n, dtype=torch.float32, device="cuda")
    fasted.sum_squared_device(pts.data_ptr(), n, d, d, sums.data_ptr())
    for rows in ("256", "128"):
        monkeypatch.setenv("FASTED_TILE_ROWS", rows)
        for flags in (0, fp.FASTED_FULL_MATRIX, fp.FASTED_SYMMETRIC, fp.FASTED_SKIP_SUMS, fp.FASTED_FULL_MATRIX | fp.FASTED_SKIP_SUMS):
            for order in (fp.FASTED_SORT_PAIRS, 0):
                pairs.fill_(-1)
                st = fasted.self_join_device(pts.data_ptr(), n, d, d, eps, pairs.data_ptr(), cap, sums_ptr=sums.data_ptr(),
                                             flags=flags | order)
                assert st.pairsFound == st.pairsStored == len(truth), (rows, flags, order)
                got = pairs[: st.pairsStored] if order else datasets.row_major(pairs[: st.pairsStored])
                assert np.array_equal(got.cpu().numpy(), truth), (rows, flags, order)
                assert bool((pairs[st.pairsStored :] == -1).all())


def test_queue_mode_two_set_exact_pair_list(fasted, monkeypatch):
    """6000 queries x 9000 candidates: 24 x 36 = 864 tiles (47 x 36 of 128 rows), none forced."""
    import torch
    from fasted_amd import find_pairs as fp

    nq, nc, d = 6000, 9000, 192
    bits, eps = integer_case(nq + nc, d, seed=77)
    stacked = oracle.self_join_f64(bits, eps)
    want = stacked[(stacked[:, 0] < nq) & (stacked[:, 1] >= nq)].copy()
    want[:, 1] -= nq
    assert len(want) > nq
    q = torch.from_numpy(bits[:nq].view(np.int16).copy()).cuda()
    c = torch.from_numpy(bits[nq:].view(np.int16).copy()).cuda()
    cap = len(want) + 1024
    pairs = torch.empty((cap, 2), dtype=torch.int32, device="cuda")
    sq = torch.empty(nq, dtype=torch.float32, device="cuda")
    sc = torch.empty(nc, dtype=torch.float32, device="cuda")
    fasted.sum_squared_device(q.data_ptr(), nq, d, d, sq.data_ptr())
    fasted.sum_squared_device(c.data_ptr(), nc, d, d, sc.data_ptr())
    for rows in ("256", "128"):
        monkeypatch.setenv("FASTED_TILE_ROWS", rows)
        for flags in (fp.FASTED_SORT_PAIRS, fp.FASTED_SORT_PAIRS | fp.FASTED_SKIP_SUMS, 0, fp.FASTED_SKIP_SUMS):
            pairs.fill_(-1)
            st = fasted.join_device(q.data_ptr(), nq, d, c.data_ptr(), nc, d, d, eps, pairs.data_ptr(), cap, flags=flags,
                                    sums_queries_ptr=sq.data_ptr(), sums_candidates_ptr=sc.data_ptr())
            assert st.pairsFound == st.pairsStored == len(want), (rows, flags)
            got = pairs[: st.pairsStored] if flags & fp.FASTED_SORT_PAIRS else datasets.row_major(pairs[: st.pairsStored])
            assert np.array_equal(got.cpu().numpy(), want), (rows, flags)


def test_queue_mode_band_check_exponential_10000x1024(fasted):
    """Exp(40) data of the headline kind at 10 000 x 1024 (1600 tiles, 16 slabs): the whole pair set against the
    FP64 checker under the relative 1e-3 band rule, the full matrix and its triangle."""
    import torch
    from fasted_amd import find_pairs as fp

    n, d = 10000, 1024
    bits = datasets.exponential(n, d, seed=31)
    eps = datasets.epsilon_for_neighbours(bits, 16)
    truth = oracle.self_join_f64(bits, eps)
    pts = torch.from_numpy(bits.view(np.int16).copy()).cuda()
    cap = 4 * len(truth)
    pairs = torch.empty((cap, 2), dtype=torch.int32, device="cuda")
    lists = []
    for flags in (fp.FASTED_SORT_PAIRS | fp.FASTED_FULL_MATRIX, fp.FASTED_SORT_PAIRS | fp.FASTED_SYMMETRIC):
        st = fasted.self_join_device(pts.data_ptr(), n, d, d, eps, pairs.data_ptr(), cap, flags=flags)
        got = pairs[: st.pairsStored].cpu().numpy()
        rep = oracle.epsilon_band_report(bits, got, eps, truth_pairs=truth)
        assert rep["outside_band"] == 0, rep
        assert 8 < (st.pairsFound - n) / n < 32
        lists.append(got)
        print("10000 x 1024:", rep)
    assert np.array_equal(lists[0], lists[1])


def test_skip_sums_needs_the_buffers_and_gives_the_same_list(fasted):
    """FASTED_SKIP_SUMS: the caller's squared norms (from fasted_sum_squared_device) are read instead of computed;
    same pair list as the default on ordinary data; refused without a buffer."""
    import torch
    from fasted_amd import find_pairs as fp

    n, d = 3000, 192
    bits = datasets.uniform_bytes(n, d, seed=8)
    eps = datasets.epsilon_for_neighbours(bits, 12)
    pts = torch.from_numpy(bits.view(np.int16).copy()).cuda()
    cap = 300 * n
    pairs = torch.empty((cap, 2), dtype=torch.int32, device="cuda")
    sums = torch.empty(n, dtype=torch.float32, device="cuda")
    st = fasted.self_join_device(pts.data_ptr(), n, d, d, eps, pairs.data_ptr(), cap, sums_ptr=sums.data_ptr())
    want = pairs[: st.pairsStored].cpu().numpy().copy()
    assert np.allclose(sums.cpu().numpy(), oracle.sum_squared(bits, "f64"), rtol=d * 2.0 ** -24)
    fasted.sum_squared_device(pts.data_ptr(), n, d, d, sums.data_ptr())
    pairs.fill_(-1)
    st2 = fasted.self_join_device(pts.data_ptr(), n, d, d, eps, pairs.data_ptr(), cap, sums_ptr=sums.data_ptr(),
                                  flags=fp.FASTED_SORT_PAIRS | fp.FASTED_SKIP_SUMS)
    assert st2.pairsFound == st.pairsFound
    assert np.array_equal(pairs[: st2.pairsStored].cpu().numpy(), want)
    # an infinite squared norm handed in by the caller: that point pairs with nothing but itself
    spoiled = sums.clone()
    spoiled[17] = float("inf")
    st3 = fasted.self_join_device(pts.data_ptr(), n, d, d, eps, pairs.data_ptr(), cap, sums_ptr=spoiled.data_ptr(),
                                  flags=fp.FASTED_SORT_PAIRS | fp.FASTED_SKIP_SUMS)
    got3 = pairs[: st3.pairsStored].cpu().numpy()
    keep = want[(want[:, 0] != 17) & (want[:, 1] != 17)]
    expect = oracle.sort_pairs(np.vstack([keep, [[17, 17]]]).astype(np.int32))
    assert np.array_equal(got3, expect)
    with pytest.raises(fp.FastedError):
        fasted.self_join_device(pts.data_ptr(), n, d, d, eps, pairs.data_ptr(), cap, sums_ptr=None,
                                flags=fp.FASTED_SKIP_SUMS)


# 2900: one workgroup per tile; 7001: the queues, in strips; 24500 (96 rows of tiles): the full matrix and all points against
# some in super-squares, the triangle in strips; 33100 (130 rows): the triangle in super-squares, the full matrix in strips
@pytest.mark.parametrize("n,d", [(n, d) for n in (2900, 7001) for d in (1, 32, 33, 65, 96, 97, 160, 992, 993)] +
                         [(n, d) for n in (24500, 33100) for d in (24, 33, 65, 150)])
def test_last_slab_with_one_and_two_steps(fasted, n, d):
    """Dimensions that reach 32 columns or more into a tile's last slab, and fewer: the triangle, the full matrix and two sets,
    with hit bits (sorted joins of up to 20 224 points) and with staged pairs.  Integer coordinates: every sum is exact, the
    lists are equal."""
    import torch
    from fasted_amd import find_pairs as fp

    gen = torch.Generator(device="cuda").manual_seed(n + d)
    ld, high = (d + 63) // 64 * 64, 2000 if d == 1 else 8 if d < 64 else 3
    pts = torch.zeros((n, ld), dtype=torch.float16, device="cuda")
    pts[:, :d] = torch.randint(0, high, (n, d), generator=gen, device="cuda").to(torch.float16)
    x = pts.float()
    sq = (x * x).sum(1)
    blocks = [(r, sq[r : r + 2048, None] + sq[None, :] - 2.0 * (x[r : r + 2048] @ x.T)) for r in range(0, n, 2048)]
    eps2 = float(torch.kthvalue(blocks[0][1][:256].flatten(), 256 * 12).values) + 0.5
    want = torch.cat([torch.nonzero(d2 <= eps2) + torch.tensor([r, 0], device="cuda") for r, d2 in blocks]).to(torch.int32)
    del blocks
    assert len(want) > 2 * n
    cap = len(want) + 64
    pairs = torch.empty((cap, 2), dtype=torch.int32, device="cuda")

    def check(st, expected, what):
        assert st.pairsFound == st.pairsStored == len(expected), what
        got = pairs[: st.pairsStored]
        assert torch.equal(got if what[-1] else datasets.row_major(got), expected), what
        assert bool((pairs[st.pairsStored :] == -1).all()), what

    m, some = n // 3, 1000
    lo = torch.tensor([0, m], dtype=torch.int32, device="cuda")
    two = want[(want[:, 0] < m) & (want[:, 1] >= m)] - lo
    against_some = want[want[:, 1] < some]
    for order in (fp.FASTED_SORT_PAIRS, 0):
        for flags in (0, fp.FASTED_FULL_MATRIX, fp.FASTED_SYMMETRIC):
            pairs.fill_(-1)
            st = fasted.self_join_device(pts.data_ptr(), n, d, ld, eps2**0.5, pairs.data_ptr(), cap, flags=flags | order)
            check(st, want, (flags, order))
        pairs.fill_(-1)
        st = fasted.join_device(pts.data_ptr(), m, ld, pts[m:].data_ptr(), n - m, ld, d, eps2**0.5, pairs.data_ptr(), cap, flags=order)
        check(st, two, ("two sets", order))
        pairs.fill_(-1)
        st = fasted.join_device(pts.data_ptr(), n, ld, pts.data_ptr(), some, ld, d, eps2**0.5, pairs.data_ptr(), cap, flags=order)
        check(st, against_some, ("all against some", order))


# one workgroup per tile, strips and super-squares; one slab and more; the full matrix, the triangle and the smaller tiles
@pytest.mark.parametrize("n,d", [(1000, 64), (3000, 100), (7001, 64), (7001, 200), (24500, 64), (17000, 1088)])
def test_contraction_alone_ends_and_finds_nothing(fasted, n, d, monkeypatch):
    import torch
    from fasted_amd import find_pairs as fp

    ld = (d + 63) // 64 * 64
    pts = torch.zeros((n, ld), dtype=torch.float16, device="cuda")
    pairs = torch.full((64, 2), -1, dtype=torch.int32, device="cuda")
    for rows in ("256", "128"):
        monkeypatch.setenv("FASTED_TILE_ROWS", rows)
        for flags in (0, fp.FASTED_SYMMETRIC, fp.FASTED_SORT_PAIRS, fp.FASTED_EVENT_TIMING):
            st = fasted.self_join_device(pts.data_ptr(), n, d, ld, 1.0, pairs.data_ptr(), len(pairs), flags=flags | fp.FASTED_NO_EPILOGUE)
            assert st.pairsFound == st.pairsStored == 0 and st.joinMs > 0
    assert bool((pairs == -1).all())
