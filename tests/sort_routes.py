"""The way of a list through the row-major sort, restated from its rules (csrc/pair_sort.hip: make_plan, plan_buckets_kernel,
sort_bucket_kernel) on sorted keys, so that a test can say which branches its lists reach."""
import numpy as np

ALONE, BUCKET, TARGET = 8192, 4096, 4096 // 3
BINS1, BINS2_BITS, MAX_IDS = 4096, 10, 2048
WINDOW_BITS, WINDOWS_ONE_LEVEL, READS_ONE_LEVEL = 18, 1024, 1 << 24
TWO_LEVELS_FROM, TWO_LEVELS_AFTER_ONE_FROM, DISTRIBUTE_UP_TO = 1 << 20, 1 << 18, 1 << 29
CELL_MAX = 48


def pairs_of(qv, cv):
    """Every (q, c) with qv[q] == cv[c], row-major."""
    order = np.argsort(cv, kind="stable")
    left, right = (np.searchsorted(cv[order], qv, side=s) for s in ("left", "right"))
    n = right - left
    rows = np.repeat(np.arange(len(qv)), n)
    at = np.arange(n.sum()) - np.repeat(np.cumsum(n) - n, n)
    return np.stack([rows, order[np.repeat(left, n) + at]], axis=1).astype(np.int32)


def _bits(n):
    return max(1, int(n - 1).bit_length())


def _bucket_features(keys, lo, last, cap):
    """How sort_bucket_kernel orders keys that lie in [lo, last] of one 2^32 range."""
    m = len(keys)
    cells = cap // 2 if m <= cap // 2 else cap
    scale = min(int(cells * 4294967296.0 / (last - lo + 1.0)), 0xFFFFFFFF)
    cell = ((keys - lo).astype(np.uint64) * np.uint64(scale) >> np.uint64(32)).astype(np.int64)
    n = np.bincount(cell, minlength=cells)
    if n.max() <= CELL_MAX:
        return set()
    begin = np.cumsum(n) - n
    first, final = keys[np.minimum(begin, m - 1)], keys[np.minimum(begin + n - 1, m - 1)]
    per_key = n.astype(np.float32) / ((final - first).astype(np.float32) + np.float32(1))
    inside = ((keys - first[cell]).astype(np.float32) * per_key[cell]).astype(np.int64)
    again = np.bincount(begin[cell] + np.minimum(n[cell] - 1, inside))
    return {"second cut"} | ({"bitonic"} if again.max() > CELL_MAX else set())


def _buckets(keys, base, shift, bins, target, first_level):
    """(records, lowest key, highest key) of the buckets; consecutive bins with one number."""
    n = np.bincount((keys - base) >> shift, minlength=bins)
    before = np.cumsum(n) - n
    ids = before // target + (n >= 2 * target)
    if first_level:
        ids = ids + ((np.arange(bins) << shift) >> 32)
    starts = np.flatnonzero(np.diff(ids, prepend=-1))
    ends = np.append(starts[1:], bins)
    for s, e in zip(starts, ends):
        a, b = before[s], before[e - 1] + n[e - 1]
        if b > a:
            yield keys[a:b], base + (int(s) << shift), base + (int(e) << shift) - 1


def _distribute(keys, last, two_levels):
    """The features on the way, or None where the distribution is broken off."""
    count, shift = len(keys), max(0, int(last).bit_length() - 12)
    target = TARGET if two_levels else min(TARGET, max(512, (count + 255) // 256))
    target1 = int(np.sqrt(float(count) * target)) if two_levels else target
    leaves, features, windows = [], set(), 0
    for part, lo, hi in _buckets(keys, 0, shift, BINS1, target1, True):
        hi = min(hi, last)
        if not two_levels:
            leaves.append((part, lo, hi))
        elif len(part) // target + 2 > MAX_IDS:
            return None
        else:
            shift2 = max(0, int(hi - lo).bit_length() - BINS2_BITS)
            leaves += [(p, a, min(b, hi)) for p, a, b in _buckets(part, lo, shift2, 1 << BINS2_BITS, target, False)]
    for part, lo, hi in leaves:
        if len(part) > BUCKET:
            w = ((hi - lo) >> WINDOW_BITS) + 1
            if not two_levels and (w > WINDOWS_ONE_LEVEL or len(part) * w > READS_ONE_LEVEL):
                return None
            windows += w
            features.add("windows")
        else:
            features |= _bucket_features(part, lo, hi, BUCKET)
    return None if windows > (count >> 8 if two_levels else WINDOWS_ONE_LEVEL) else features


def route(pairs, nq, nc):
    """The set of branches that a list of sorted distinct pairs takes."""
    bits = _bits(nc)
    keys = pairs[:, 0].astype(np.int64) << bits | pairs[:, 1]
    count, last = len(keys), (nq - 1) << bits | (nc - 1)
    if count <= ALONE and last >> 32 == 0:
        return {"one workgroup"} | _bucket_features(keys, 0, last, ALONE)
    taken = set()
    two_levels = count > TWO_LEVELS_FROM
    while count <= DISTRIBUTE_UP_TO and last >> 42 == 0:
        level = "two levels" if two_levels else "one level"
        features = _distribute(keys, last, two_levels)
        if features is not None:
            return taken | features | {level}
        taken.add(level + " broken off")
        if two_levels or count < TWO_LEVELS_AFTER_ONE_FROM:
            break
        two_levels = True
    return taken | {"radix"}


def _with_row(nq, nc, row, candidates, others=1.0):
    """`others` pairs per query on average, anywhere, and one query that has the given candidates."""
    rng = np.random.default_rng(nq + nc + row)
    q = np.arange(nq) + 1
    c = nq + 1 + np.arange(nc)
    place = rng.permutation(nc)[: int(nq * others)]
    c[place] = q[np.arange(len(place)) % nq]
    q[row], c[candidates] = 0, 0
    return q, c


def _scattered(nc, n):
    return np.random.default_rng(nc + n).permutation(nc)[:n]


def _full_rows():
    q, c = _with_row(1 << 14, 1 << 20, 4, _scattered(1 << 20, 1000000), 0.5)
    q[5:7] = 0
    return q, c


def _run(start, length, far):
    return np.append(start + np.arange(length), far)


# lists that crowd: coded query and candidate points, and branches they have to reach
CASES = {
    "one level breaks off, the radix sort takes over": (
        lambda: _with_row(300000, 300000, 77, _scattered(300000, 100000), 0.3), {"one level broken off", "radix"}),
    "one level breaks off, two take over": (
        lambda: _with_row(300000, 300000, 77, _scattered(300000, 270000), 0.3), {"one level broken off", "two levels"}),
    "two levels break off": (_full_rows, {"two levels broken off", "radix"}),
    "two levels, thin windows": (
        lambda: _with_row(1100000, 1100000, 500001, _scattered(1100000, 5000), 1.0), {"two levels", "windows"}),
    "one level, thin windows": (
        lambda: _with_row(300000, 300000, 299999, _scattered(300000, 10000), 0.1), {"one level", "windows"}),
    "one level, half-full windows": (
        lambda: _with_row(1000, 1000000, 517, _scattered(1000000, 500000), 1.0), {"one level", "windows"}),
    "one level, full windows": (
        lambda: _with_row(1000, 1000000, 517, np.arange(3, 999999), 0.0), {"one level", "windows"}),
    "one workgroup, runs in runs": (
        lambda: _with_row(1000, 1000000, 5, _run(0, 300, 100000), 2.0), {"one workgroup", "bitonic"}),
    "a bucket, runs in runs": (
        lambda: _with_row(20000, 1 << 20, 4321, _run(70000, 300, 90000), 0.5), {"one level", "bitonic"}),
}
