"""Performance cases of the epsilon self-join: what a program that uses this library has it do.

Sizes, data and neighbour counts follow the repository's own workloads (``bench.py``'s five configurations, scaled to
passes of at most a fraction of a second, and the size x dimensionality sweep of the speed experiment) and the odd
sizes of its tests.  Every case goes through the public entry points of ``fasted_amd``.  Whether a pair belongs to the
result depends on the FP16 inputs and the FP32 accumulation only, so pair lists, which come back sorted row-major, are
compared exactly; buffers come back whole, with the zeros the program put there behind the last pair.
"""
import ctypes
import math

import numpy as np
import torch

import fasted_amd as fa
from fasted_amd.find_pairs import FASTED_SORT_PAIRS, FASTED_SYMMETRIC

MAX_FLOPS = 2.0 * 100_000**2 * 4096  # no drawn case costs more than the largest listed one
MAX_PAIRS = 200_000 * 1001


def _case(kind, n, d, data, neighbours, queries=0, symmetric=False, name=None):
    case = {"kind": kind, "n": n, "d": d, "data": data, "neighbours": neighbours, "queries": queries, "symmetric": symmetric}
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # smallest cell of the size x dimensionality sweep: launches and latency are all of it
        _case("self", 1000, 64, "exponential", 4, name="sweep_1000x64"),
        # the plumbing workload: a join of microseconds whose pair list still has to come back in order
        _case("self", 4096, 128, "exponential", 32, name="plumbing_4096x128"),
        # sizes that are a multiple of nothing, clustered as feature vectors are: a mid-size dataset
        _case("self", 9733, 257, "mixture", 100, name="ragged_9733x257"),
        # the opt-in symmetric join on a sweep size
        _case("self", 46416, 512, "exponential", 64, symmetric=True, name="symmetric_46416x512"),
        # the low-dimensional workload (byte-valued descriptors)
        _case("self", 100_000, 128, "bytes", 64, name="lowdim_100000x128"),
        # the headline workload's data and dimensionality at a tenth of its points
        _case("self", 100_000, 4096, "exponential", 16, name="highdim_100000x4096"),
        # the clustered workload at two fifths of its points
        _case("self", 200_003, 960, "mixture", 100, name="clustered_200003x960"),
        # the output-heavy workload at a tenth of its points: 200 million pairs
        _case("self", 200_000, 384, "unit", 1000, name="outputheavy_200000x384"),
        # a batch of new points against a standing collection
        _case("two", 250_000, 200, "bytes", 16, queries=10_007, name="twosets_10007x250000x200"),
        # how many neighbours has a point at this epsilon: the first count-only probe of an epsilon calibration on
        # sampled rows, which also leaves the squared norms for the probes that follow
        _case("count", 200_000, 384, "unit", 100, queries=16_384, name="probe_16384of200000x384"),
        # points in host memory in, pairs in host memory out
        _case("host", 30_000, 200, "exponential", 32, name="host_30000x200"),
        # the distance column of a neighbour table: one distance per pair of a join's result
        _case("distances", 50_021, 384, "unit", 100, name="distances_50021x384"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["self", "self", "self", "self", "two", "count", "host", "distances"])
    data = rng.choice(["exponential", "bytes", "mixture", "unit"])
    d = _log_int(rng, 17, 4096)
    if rng.random() < 0.4:  # dimensionalities of real descriptors are often multiples of 64
        d = max(64, 64 * (d // 64))
    lo, hi = {"self": (1000, 250_000), "two": (4000, 250_000), "count": (20_000, 250_000), "host": (1000, 50_000),
              "distances": (4000, 60_000)}[kind]
    hi = min(hi, int(math.sqrt(MAX_FLOPS / (2.0 * d))))
    n = _log_int(rng, lo, hi)
    if kind in ("host", "distances"):
        neighbours = _log_int(rng, 4, 128)
    else:
        neighbours = min(_log_int(rng, 4, 1000), n // 8, MAX_PAIRS // n)
    queries = _log_int(rng, 1000, max(2000, n // 4)) if kind in ("two", "count") else 0
    symmetric = kind == "self" and rng.random() < 0.2
    return _case(kind, n, d, data, neighbours, queries, symmetric)


def _points(gen, data, n, d, centers):
    """n x ld FP16 points on the device, zeros in the padding columns d .. ld-1 (ld: d rounded up to 64)."""
    ld = (d + 63) // 64 * 64
    out = torch.zeros((n, ld), dtype=torch.float16, device="cuda")
    rows = max(1, (1 << 27) // d)
    for r0 in range(0, n, rows):
        m = min(n, r0 + rows) - r0
        if data == "exponential":
            x = torch.empty((m, d), device="cuda").exponential_(40.0, generator=gen).clamp_(0.0, 1.0)
        elif data == "bytes":
            x = torch.randint(0, 256, (m, d), generator=gen, device="cuda").to(torch.float32) / 255.0
        elif data == "mixture":
            which = torch.randint(0, centers.shape[0], (m,), generator=gen, device="cuda")
            x = centers[which] + 0.05 * torch.randn((m, d), generator=gen, device="cuda")
        else:
            x = torch.randn((m, d), generator=gen, device="cuda")
            x = x / x.norm(dim=1, keepdim=True)
        out[r0:r0 + m, :d] = x.to(torch.float16)
    return out


def _epsilon(gen, queries, points, neighbours, self_pairs):
    """The distance that gives sampled query rows the wanted mean number of neighbours among all points."""
    m = min(512, queries.shape[0])
    rows = torch.randperm(queries.shape[0], generator=gen, device="cuda")[:m]
    q = queries[rows].to(torch.float32)
    qs = (q * q).sum(1)
    d2 = torch.empty((m, points.shape[0]), device="cuda")
    for c0 in range(0, points.shape[0], 32768):
        c = points[c0:c0 + 32768].to(torch.float32)
        d2[:, c0:c0 + c.shape[0]] = qs[:, None] + (c * c).sum(1)[None, :] - 2.0 * (q @ c.T)
    want = m * (neighbours + (1 if self_pairs else 0))
    lo, hi = 0.0, float(d2.max())
    for _ in range(40):
        mid = 0.5 * (lo + hi)
        if int((d2 <= mid).sum()) < want:
            lo = mid
        else:
            hi = mid
    return math.sqrt(hi)


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    kind, n, d, data = case["kind"], case["n"], case["d"], case["data"]
    centers = torch.rand((min(1000, max(2, n // 500)), d), generator=gen, device="cuda") if data == "mixture" else None
    points = _points(gen, data, n, d, centers)
    state = {"kind": kind, "n": n, "d": d, "ld": points.shape[1], "points": points}
    if kind in ("two", "count"):
        if kind == "two":
            queries = _points(gen, data, case["queries"], d, centers)
        else:
            queries = points[torch.randperm(n, generator=gen, device="cuda")[:case["queries"]]].contiguous()
        state["queries"] = queries
        state["epsilon"] = _epsilon(gen, queries, points, case["neighbours"], kind == "count")
        rows = case["queries"]
    else:
        state["epsilon"] = _epsilon(gen, points, points, case["neighbours"], True)
        rows = n
    if kind == "count":
        state["sums"] = [torch.empty((m,), dtype=torch.float32, device="cuda") for m in (rows, n)]
    else:
        # room for half as many pairs again as the sample promises
        cap = rows * (case["neighbours"] + 1) * 3 // 2 + 4096
        state["cap"] = cap
        state["flags"] = FASTED_SORT_PAIRS | (FASTED_SYMMETRIC if case["symmetric"] else 0)
        if kind == "host":
            state["points"] = points[:, :d].contiguous().cpu().numpy()
            state["pairs"] = np.zeros((cap, 2), dtype=np.int32)
        else:
            state["pairs"] = torch.zeros((cap, 2), dtype=torch.int32, device="cuda")
    if kind == "distances":
        st = fa.self_join_device(points.data_ptr(), n, d, state["ld"], state["epsilon"], state["pairs"].data_ptr(), cap)
        state["count"] = int(st.pairsStored)
        state["distances"] = torch.zeros((cap,), dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    return state


def run(state):
    kind, p, n, d, ld, eps = (state[k] for k in ("kind", "points", "n", "d", "ld", "epsilon"))
    if kind == "self":
        st = fa.self_join_device(p.data_ptr(), n, d, ld, eps, state["pairs"].data_ptr(), state["cap"], flags=state["flags"])
        return {"found": int(st.pairsFound), "stored": int(st.pairsStored), "pairs": state["pairs"]}
    if kind == "two":
        q = state["queries"]
        st = fa.join_device(q.data_ptr(), q.shape[0], ld, p.data_ptr(), n, ld, d, eps, state["pairs"].data_ptr(),
                            state["cap"], flags=state["flags"])
        return {"found": int(st.pairsFound), "stored": int(st.pairsStored), "pairs": state["pairs"]}
    if kind == "count":
        q, (sums_q, sums_p) = state["queries"], state["sums"]
        st = fa.join_device(q.data_ptr(), q.shape[0], ld, p.data_ptr(), n, ld, d, eps, None, 0, flags=0,
                            sums_queries_ptr=sums_q.data_ptr(), sums_candidates_ptr=sums_p.data_ptr())
        return {"found": int(st.pairsFound), "sums_queries": sums_q, "sums_candidates": sums_p}
    if kind == "host":
        lib = fa.load_findpairs()
        found, stored = ctypes.c_ulonglong(), ctypes.c_ulonglong()
        rc = lib.fasted_self_join(p.ctypes.data, n, d, eps, state["pairs"].ctypes.data, state["cap"], ctypes.byref(found),
                                  ctypes.byref(stored))
        if rc != 0:
            raise RuntimeError(lib.fasted_last_error().decode())
        return {"found": found.value, "stored": stored.value, "pairs": state["pairs"]}
    fa.pair_distances_device(p.data_ptr(), n, ld, p.data_ptr(), n, ld, d, state["pairs"].data_ptr(), state["count"],
                             state["distances"].data_ptr())
    return state["distances"]


def work(case):
    n, d, kind = case["n"], case["d"], case["kind"]
    per_point = case["neighbours"] + (0 if kind == "two" else 1)
    if kind in ("two", "count"):
        q = case["queries"]
        return {"bytes": 2.0 * (q + n) * d + (8.0 * q * per_point if kind == "two" else 4.0 * (q + n)), "flops": 2.0 * q * n * d}
    if kind == "distances":
        return {"bytes": 2.0 * n * d + 12.0 * n * per_point, "flops": 3.0 * n * per_point * d}
    # a self-join needs every unordered pair's product once: dist(q, c) = dist(c, q)
    return {"bytes": 2.0 * n * d + 8.0 * n * per_point, "flops": float(n) * (n + 1) * d}


def tolerance(case):
    if case["kind"] in ("distances", "count"):
        # FP32 sums of D terms: measured against FP64 at D = 17 ... 4000 at most 9.4e-8 (2-norm) and 2.8e-7 (largest)
        return {"rel": 4e-7, "max": 1.2e-6}
    return "exact"
