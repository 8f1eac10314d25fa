"""GPU tests at the benchmark configurations' full sizes.  A full FP64 join is out of reach there,
so these check size-independent properties of the pair list (sorted, duplicate free, symmetric, every
self pair present, nothing lost) and compare a seeded sample of query rows against FP64 distances
with the epsilon-band rule: a pair may disagree with FP64 only if |d - eps| / eps <= 1e-3.  The checks are made on the
list of the full matrix, as the benchmark computes it; the library's own choice, the triangle, must give the same list."""
import numpy as np
import pytest

import oracle
from fasted_amd import find_pairs as fp

pytestmark = pytest.mark.gpu

BAND = 1e-3


@pytest.fixture(scope="module")
def env():
    import torch

    import bench
    import fasted_amd

    fasted_amd.load_findpairs()
    return torch, bench, fasted_amd


def run_config(env, name, n=None, sample_rows=256, oracle_rows=0):
    torch, bench, fasted = env
    n0, d, kind, neighbours, _ = bench.CONFIGS[name]
    n = n or n0
    pts = bench.generate_points(torch, kind, n, d, seed=777 + d)
    eps = bench.calibrate_epsilon(torch, pts, neighbours, sample=512)
    cap = int(max(n * 64, 2.0 * n * (neighbours + 1)))
    pairs = torch.empty((cap, 2), dtype=torch.int32, device="cuda")
    full = fp.FASTED_SORT_PAIRS | fp.FASTED_FULL_MATRIX
    st = fasted.self_join_device(pts.data_ptr(), n, d, d, eps, pairs.data_ptr(), cap, flags=full)
    print(f"{name}: N={n} D={d} eps={eps:.6g} found={st.pairsFound} neighbours/point={(st.pairsFound - n) / n:.1f} "
          f"join={st.joinMs:.1f} ms ({2.0 * n * n * d / st.joinMs / 1e9:.0f} TFLOPS) sort={st.sortMs:.1f} ms")
    assert st.pairsFound == st.pairsStored <= cap, "pair buffer overflowed: nothing may be lost here"
    got = pairs[: st.pairsStored]
    again = torch.empty_like(pairs)
    chosen = fasted.self_join_device(pts.data_ptr(), n, d, d, eps, again.data_ptr(), cap)
    assert chosen.pairsFound == chosen.pairsStored == st.pairsFound and torch.equal(again[: st.pairsStored], got)
    del again
    q, c = got[:, 0].to(torch.int64), got[:, 1].to(torch.int64)

    # sorted row-major, hence duplicate free
    keys = q * n + c
    assert bool((keys[1:] > keys[:-1]).all())
    del keys
    assert int(q.min()) >= 0 and int(q.max()) < n and int(c.min()) >= 0 and int(c.max()) < n
    # every self pair is there
    assert int((q == c).sum()) == n
    # symmetric: the multiset of (c, q) equals the multiset of (q, c)
    swapped = torch.sort(c * n + q).values
    assert bool((swapped == q * n + c).all())
    del swapped
    # neighbours per point in the right ballpark of the calibration target
    mean_nb = (st.pairsFound - n) / n
    assert 0.25 * neighbours < mean_nb < 4.0 * neighbours, mean_nb

    # seeded sample of query rows against FP64 distances to all points (computed in chunks)
    g = torch.Generator(device="cuda")
    g.manual_seed(5)
    rows = torch.sort(torch.randperm(n, generator=g, device="cuda")[:sample_rows]).values
    xs = pts[rows].to(torch.float64)
    xs2 = (xs * xs).sum(1)
    start = torch.searchsorted(q.contiguous(), rows)
    stop = torch.searchsorted(q.contiguous(), rows + 1)
    got_mask = torch.zeros((len(rows), n), dtype=torch.bool, device="cuda")
    for i in range(len(rows)):
        got_mask[i, c[start[i]:stop[i]]] = True
    band_pairs, worst, outside = 0, 0.0, 0
    chunk = max(1, (1 << 26) // d)
    for c0 in range(0, n, chunk):
        y = pts[c0:c0 + chunk].to(torch.float64)
        d2 = (xs2[:, None] + (y * y).sum(1)[None, :] - 2.0 * (xs @ y.T)).clamp_min(0.0)
        truth = d2 <= eps * eps
        diff = truth != got_mask[:, c0:c0 + chunk]
        if bool(diff.any()):
            rel = (d2[diff].sqrt() - eps).abs() / eps
            band_pairs += int(diff.sum())
            worst = max(worst, float(rel.max()))
            outside += int((rel > BAND).sum())
    print(f"{name}: {sample_rows} sampled rows vs FP64: {band_pairs} pairs inside the band, "
          f"max relative distance error {worst:.2e}, outside the band {outside}")
    assert outside == 0

    # a few rows against the CPU checker as well (needs the points on the host)
    if oracle_rows:
        host = pts.cpu().numpy().view(np.uint16)
        r0 = int(rows[0])
        ref = oracle.self_join_f64(host, eps, n=n, rows=(r0, r0 + oracle_rows))
        lo = int(torch.searchsorted(q.contiguous(), torch.tensor([r0], device="cuda"))[0])
        hi = int(torch.searchsorted(q.contiguous(), torch.tensor([r0 + oracle_rows], device="cuda"))[0])
        mine = got[lo:hi].cpu().numpy()
        rep = oracle.epsilon_band_report(host, mine, eps, truth_pairs=ref, band=BAND)
        print(f"{name}: rows [{r0}, {r0 + oracle_rows}) vs CPU checker: {rep}")
        assert rep["outside_band"] == 0
    return st


def test_config2_low_dim_100k_x_128(env):
    run_config(env, "c2", sample_rows=1024, oracle_rows=64)


def test_config4_clustered_500k_x_960(env):
    run_config(env, "c4", sample_rows=1024, oracle_rows=4)


def test_config5_output_heavy_2m_x_384(env):
    st = run_config(env, "c5", sample_rows=1024, oracle_rows=4)
    assert st.pairsFound > 2e8  # the output-heavy case really is output heavy


def test_config3_headline_1m_x_4096(env):
    run_config(env, "c3", sample_rows=1024, oracle_rows=4)


def test_two_sets_whose_norms_do_not_fit_one_launch(env):
    """One query and 67 108 860 candidates of 512 dimensions: as many workgroups of the norm kernel as a launch can hold for
    the candidates alone, and one more for the query."""
    torch, _, fasted = env
    n, d = 67_108_860, 512
    if torch.cuda.mem_get_info()[0] < 80 << 30:
        pytest.skip("needs 70 GB of device memory")
    points = torch.zeros((n, d), dtype=torch.float16, device="cuda")
    query = torch.ones((1, d), dtype=torch.float16, device="cuda")
    near = torch.tensor([0, 255, 256, n // 2, n - 1], device="cuda")
    points[near] = 1.0
    sq, sc = torch.empty(1, device="cuda"), torch.full((n,), -1.0, device="cuda")
    pairs = torch.full((16, 2), -1, dtype=torch.int32, device="cuda")
    st = fasted.join_device(query.data_ptr(), 1, d, points.data_ptr(), n, d, d, 0.5, pairs.data_ptr(), 16, flags=fp.FASTED_SORT_PAIRS,
                            sums_queries_ptr=sq.data_ptr(), sums_candidates_ptr=sc.data_ptr())
    assert st.pairsFound == st.pairsStored == len(near)
    assert torch.equal(pairs[: len(near), 1].long(), near) and bool((pairs[: len(near), 0] == 0).all())
    assert float(sq[0]) == d and bool((sc[near] == d).all()) and float(sc.double().sum()) == d * len(near)
    del points, sc
    torch.cuda.empty_cache()
