// pair_sort.hip -- row-major order of the stored pairs on the device after the join.
//
// The reference sorts its pair buffer with thrust::sort and Pair::operator< (query index,
// then candidate index; source/pair.cuh:39-45,151-158).  A pair is 8 bytes with the query
// index in the low word; packed as (query << bits of a candidate index) | candidate that order is plain
// unsigned order.  Two ways to it: distribution into buckets that fit a workgroup's LDS (see below), and, for what
// that does not take (more than 2^29 records, keys of more than 42 bits, lists it breaks off because they crowd into
// a few rows), rocPRIM's radix sort over the bits the indices can occupy: pack, sort, unpack.
#include <cstring>
#include <type_traits>

#include <rocprim/device/device_radix_sort.hpp>

#include "join_kernels.h"

namespace fasted {
namespace {

// record (candidate << 32 | query) -> key (query << candidateBits | candidate), and back
__global__ void pack_pairs_kernel(const unsigned long long* __restrict__ in, unsigned long long* __restrict__ out,
                                  unsigned long long count, int candidateBits) {
    const unsigned long long stride = (unsigned long long)gridDim.x * blockDim.x;
    for (unsigned long long i = (unsigned long long)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += stride) {
        const unsigned long long v = in[i];
        out[i] = ((v & 0xffffffffull) << candidateBits) | (v >> 32);
    }
}
__global__ void unpack_pairs_kernel(const unsigned long long* __restrict__ in, unsigned long long* __restrict__ out,
                                    unsigned long long count, int candidateBits) {
    const unsigned long long stride = (unsigned long long)gridDim.x * blockDim.x;
    for (unsigned long long i = (unsigned long long)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += stride) {
        const unsigned long long k = in[i];
        out[i] = ((k & ((1ull << candidateBits) - 1ull)) << 32) | (k >> candidateBits);
    }
}

int index_bits(long long n) {  // bits of the largest index of n items; 32 when n is not known
    if (n <= 0 || n > (1ll << 32)) return 32;
    int b = 1;
    while ((1ll << b) < n) ++b;
    return b;
}

// ------------------------------------------------------------------------------------------
// Row-major order by distribution.  The key of a record is (query << form) | candidate; the keys of a join
// are distinct and, apart from clustering, spread evenly, so a record's place is found by counting instead of by
// passes over all key bits:
//   count_keys_kernel     how many records fall into each of at most 4096 equal key ranges (bins)
//   plan_buckets_kernel   prefix sums over the bins; runs of bins become buckets of about `target` records, 512 to 1365
//                         (a bucket never crosses a multiple of 2^32, so the low word of the key is enough from here on)
//   scatter_keys_kernel   every record's low key word goes to its bucket, in any order inside the bucket
//   sort_bucket_kernel    one workgroup orders a bucket of up to 4096 keys in LDS and writes the records out
// From 2^20 records on the first three run twice, the second time on every bucket of the first by itself (1024 bins
// each).  A bucket of more than 4096 keys is a bin that is crowded by itself; the last kernel orders it in windows
// (order_windows).  Too many windows: one level breaks off after its plan and starts again with two, where a bin covers at
// most 16 windows; lists of less than 2^18 records, and bins that two levels cannot cut small enough (millions of records
// in 1/4096 of the key range), go to the radix sort.  A few times 4096 records are ordered by one workgroup alone (sort_bucket_kernel on the records themselves).
// Bound by memory traffic: 32 bytes per record in one level, 44 in two, of which a key on its way is 4 (the radix sort
// with its pack and unpack moves 120 at 36 key bits); below a million records by the launches.  Measured, join records,
// radix sort -> this: 4 849 records 45 -> 18 us, 135 thousand 75 -> 34, 974 thousand 195 -> 43, 6.5 million 330 -> 160,
// 200 million 7.5 -> 2.6 ms; 1.04 million in 200 000 rows 200 -> 52, 0.6 million of which 0.4 in 2000 of 100 000 rows 165
// -> 76.  Slower where a list that breaks off is short, or one row holds most of a long one: 100 thousand records, half of
// them in one row of a million, 71 -> 102 us, 3 million, half of them in one row of two million, 262 -> 323.
// Where the lines between one workgroup, one level and two lie: one workgroup takes 8192 records in 22 us, two launches
// less than the 32 us of one level; one level takes 1.04 million records in 53 us, two take 1.1 million in 65.  Where a list
// breaks off, two levels took 500 thousand records in 150 us and the radix sort 180, 100 thousand in 140 and 100.
typedef unsigned int u32;
typedef unsigned long long u64;
typedef u32 u32x4 __attribute__((ext_vector_type(4)));
constexpr int kSortThreads = 1024;
constexpr int kAloneCap = 8192;                       // records that one workgroup orders by itself
constexpr int kBucketThreads = 512, kBucketCap = 4096; // a workgroup that orders a bucket in LDS, and the bucket's keys
constexpr u32 kTargetMax = kBucketCap / 3;              // up to one target plus a bin of less than two share a bucket
constexpr int kBins1 = 4096, kBins2Bits = 10, kBins2 = 1 << kBins2Bits;
constexpr int kMaxIds = 2048;                         // buckets one workgroup of scatter_keys_kernel can tell apart
constexpr int kWindowBits = 18;                       // key range that a workgroup marks in a bit map in LDS
static_assert(1 << kWindowBits == 2 * kBucketCap * 32, "the bit map is the two key arrays of sort_bucket_kernel");
constexpr int kWindowWorkers = 256;                   // workgroups of sort_bucket_kernel that work on windows
constexpr u32 kWindowsOneLevel = 1024;                // one level breaks off where there are more windows than this, or a
constexpr u64 kReadsOneLevel = 1ull << 24;            // bucket's keys would be read more often than this
constexpr int kWindowNumberBits = 12;                 // a window is stored as bucket << kWindowNumberBits | number
constexpr u32 kCellMax = 48;                          // cells fuller than this: the bucket goes through the bitonic network

// What the kernels of a sort tell each other, in front of the tables.
struct SortState {
    u64 brokenOff[2];  // number of the last sort that the plan of the first, of the second level has broken off
    u32 windows;       // windows of the buckets that are too large for the LDS
};
__device__ __forceinline__ bool broken_off(const SortState* s, u64 epoch) {
    return s->brokenOff[0] == epoch || s->brokenOff[1] == epoch;
}

struct Bucket {
    u32 start, end;   // records [start, end) of the key array
    u32 window;       // key >> 32
    u32 lo, last;     // smallest and largest low key word that can occur
    u32 shift;        // (next level) bin = (low word - lo) >> shift
    u32 pad[2];
};

// How a record and its key correspond: key = (query - firstQuery) << candidateBits | candidate.
struct KeyForm {
    int candidateBits;
    u32 firstQuery;
};
__device__ __forceinline__ u64 key_of(u64 record, KeyForm f) {
    return ((u64)((u32)record - f.firstQuery) << f.candidateBits) | (record >> 32);
}

// Which bucket workgroup `unit` works on when bucket b gets one workgroup per `chunk` records: the workgroups of b
// start at b.start / chunk + b, which leaves every bucket as many numbers as it needs.  ~0: none.
__device__ __forceinline__ u32 find_bucket(const Bucket* __restrict__ buckets, u32 count, u32 unit, u32 chunk, u32* found) {
    if (threadIdx.x == 0) *found = ~0u;
    __syncthreads();
    for (u32 b = threadIdx.x; b < count; b += kSortThreads) {
        const u32 first = buckets[b].start / chunk + b, size = buckets[b].end - buckets[b].start;
        if (unit >= first && unit - first < (size + chunk - 1) / chunk) *found = b;
    }
    __syncthreads();
    return *found;
}

template <bool kRecords>
__global__ void __launch_bounds__(kSortThreads) count_keys_kernel(const void* __restrict__ in, u32 count, KeyForm form,
                                                                  int shift, const Bucket* __restrict__ parents,
                                                                  u32 parentCount, u32 chunk, u32* __restrict__ bins,
                                                                  SortState* __restrict__ state) {
    constexpr int kBins = kRecords ? kBins1 : kBins2;
    typedef std::conditional_t<kRecords, u64, u32> Key;
    __shared__ u32 local[kBins];
    __shared__ u32 which;
    u32 begin = blockIdx.x * chunk, end = min(count - begin, chunk) + begin, lo = 0;
    if (kRecords) {
        if (blockIdx.x == 0 && threadIdx.x == 0) state->windows = 0;
    } else {
        const u32 b = find_bucket(parents, parentCount, blockIdx.x, chunk, &which);
        if (b == ~0u) return;
        const Bucket p = parents[b];
        begin = p.start + (blockIdx.x - (p.start / chunk + b)) * chunk;
        end = min(p.end - begin, chunk) + begin;
        lo = p.lo;
        shift = (int)p.shift;
        bins += (size_t)b * kBins2;
    }
    for (int i = threadIdx.x; i < kBins; i += kSortThreads) local[i] = 0;
    __syncthreads();
    constexpr int kUnroll = 4;
    for (u32 base = begin; base < end; base += kUnroll * kSortThreads) {
        // (all loads are issued before the first is used: no branch between them)
        Key v[kUnroll];
        u32 bin[kUnroll];
#pragma unroll
        for (int e = 0; e < kUnroll; ++e) v[e] = static_cast<const Key*>(in)[min(base + e * kSortThreads + threadIdx.x, end - 1)];
#pragma unroll
        for (int e = 0; e < kUnroll; ++e) {
            bin[e] = kRecords ? (u32)(key_of(v[e], form) >> shift) : ((u32)v[e] - lo) >> shift;
            if (base + e * kSortThreads + threadIdx.x >= end) bin[e] = ~0u;
        }
#pragma unroll
        for (int e = 0; e < kUnroll; ++e)
            if (bin[e] < (u32)kBins) atomicAdd(&local[bin[e]], 1u);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < kBins; i += kSortThreads)
        if (local[i]) atomicAdd(&bins[i], local[i]);
}

// Exclusive prefix sum over the workgroup's values, one per thread.
template <int kThreads>
__device__ __forceinline__ u32 block_exclusive_scan(u32 v, u32* waveSums) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    u32 x = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const u32 y = __shfl_up(x, off, 64);
        if (lane >= off) x += y;
    }
    if (lane == 63) waveSums[wave] = x;
    __syncthreads();
    u32 before = 0;
#pragma unroll
    for (int w = 0; w < kThreads / 64; ++w)
        if (w < wave) before += waveSums[w];
    __syncthreads();
    return before + x - v;
}

// One workgroup per parent bucket (first level: one, for everything).  Bin i belongs to bucket (records before the
// bin) / target, moved on by one at every multiple of 2^32 of the key: consecutive bins, less than three targets of
// records in all.  A bin of two targets or more is a bucket of its own (it ends at least two numbers further on, so the
// number after the one in front of it is free).  The children of parent b are numbered from b.start / target + b on.  Bins are left zeroed.
template <bool kFirst>
__global__ void __launch_bounds__(kSortThreads) plan_buckets_kernel(u32* __restrict__ bins, u32 count, int shift, u32 lastHigh,
                                                                    u32 lastLow, const Bucket* __restrict__ parents, u32 target,
                                                                    u32 childCount, u32 nextTarget, Bucket* __restrict__ children,
                                                                    unsigned short* __restrict__ childOfBin,
                                                                    u32* __restrict__ cursors, u32* __restrict__ windowList,
                                                                    u32 maxWindows, SortState* __restrict__ state, u64 epoch,
                                                                    u64* brokenOffHost) {
    constexpr int kBins = kFirst ? kBins1 : kBins2;
    constexpr int kPer = kBins / kSortThreads;
    __shared__ u32 waveSums[kSortThreads / 64];
    __shared__ u32 idOf[kBins + 1], startOf[kBins + 1], firstOf[kMaxIds];
    Bucket p{0u, count, 0u, 0u, lastLow, 0u, {0u, 0u}};
    u32 firstChild = 0, ids = childCount;
    if (!kFirst) {
        p = parents[blockIdx.x];
        if (state->brokenOff[0] == epoch) return;  // (the other one may turn while this kernel runs)
        shift = (int)p.shift;
        firstChild = p.start / target + blockIdx.x;
        ids = (blockIdx.x + 1 < gridDim.x ? parents[blockIdx.x + 1].start / target + blockIdx.x + 1 : childCount) - firstChild;
        bins += (size_t)blockIdx.x * kBins2;
        childOfBin += (size_t)blockIdx.x * kBins2;
        children += firstChild;
        cursors += firstChild;
    }
    for (u32 i = threadIdx.x; i < (u32)kMaxIds; i += kSortThreads) firstOf[i] = ~0u;
    u32 n[kPer], sum = 0;
#pragma unroll
    for (int e = 0; e < kPer; ++e) {
        n[e] = bins[threadIdx.x * kPer + e];
        bins[threadIdx.x * kPer + e] = 0;
        sum += n[e];
    }
    u32 before = block_exclusive_scan<kSortThreads>(sum, waveSums);
#pragma unroll
    for (int e = 0; e < kPer; ++e) {
        const u32 i = threadIdx.x * kPer + e;
        const u32 id = before / target + (n[e] >= 2 * target ? 1u : 0u) + (kFirst ? (u32)(((u64)i << shift) >> 32) : 0u);
        idOf[i] = min(id, ids - 1);  // (bins past the last key only)
        startOf[i] = before;
        atomicMin(&firstOf[id < ids ? id : ids - 1], i);
        childOfBin[i] = (unsigned short)idOf[i];
        before += n[e];
    }
    if (threadIdx.x == kSortThreads - 1) {
        idOf[kBins] = ids;
        startOf[kBins] = p.end - p.start;
    }
    __syncthreads();
    bool breakOff = false;
#pragma unroll
    for (int e = 0; e < kPer; ++e) {
        const u32 i = threadIdx.x * kPer + e;
        const u32 id = idOf[i], previous = i ? idOf[i - 1] : ~0u;
        if (id != previous) {
            // the first bin of a bucket; the numbers skipped in front of it are empty buckets
            const u32 at = p.start + startOf[i];
            for (u32 s = previous + 1; s < id; ++s) children[s] = Bucket{at, at, 0u, 0u, 0u, 0u, {0u, 0u}};
            const u64 low = kFirst ? ((u64)i << shift) : (u64)p.lo + ((u64)i << shift);
            children[id].start = at;
            children[id].window = kFirst ? (u32)(low >> 32) : p.window;
            children[id].lo = (u32)low;
            cursors[id] = at;
        }
    }
#pragma unroll
    for (int e = 0; e < kPer; ++e) {
        const u32 i = threadIdx.x * kPer + e;
        const u32 id = idOf[i];
        if (idOf[i + 1] != id) {
            // its last bin: where it ends, and the key range it covers
            const u32 first = firstOf[id];
            const u64 base = kFirst ? 0ull : (u64)p.lo;
            const u64 lowest = base + ((u64)first << shift);
            u64 highest = base + ((u64)(i + 1) << shift) - 1;
            const u64 bound = kFirst ? (((u64)lastHigh << 32) | lastLow) : (u64)p.last;
            if (highest > bound) highest = bound;
            if (highest < lowest) highest = lowest;
            children[id].end = p.start + startOf[i + 1];
            children[id].last = (u32)highest;
            const u64 range = highest - lowest;
            const int bits = 64 - __clzll((long long)range);
            children[id].shift = (u32)(bits > kBins2Bits ? bits - kBins2Bits : 0);
            const u32 size = startOf[i + 1] - startOf[first];
            if (nextTarget) {
                // cut into at most size / nextTarget + 2 at the next level: as many as scatter_keys_kernel can tell apart?
                breakOff |= size / nextTarget + 2 > (u32)kMaxIds;
            } else if (size > (u32)kBucketCap) {
                const u64 windows = (range >> kWindowBits) + 1;
                const bool few = windows <= min(maxWindows, 1u << kWindowNumberBits) && (!kFirst || size * windows <= kReadsOneLevel);
                const u32 at = few ? atomicAdd(&state->windows, (u32)windows) : 0u;
                breakOff |= !few || at + (u32)windows > maxWindows;
                if (!breakOff)
                    for (u32 w = 0; w < (u32)windows; ++w) windowList[at + w] = (firstChild + id) << kWindowNumberBits | w;
            }
        }
    }
    if (threadIdx.x == kSortThreads - 1)
        for (u32 s = idOf[kBins - 1] + 1; s < ids; ++s) children[s] = Bucket{p.end, p.end, 0u, 0u, 0u, 0u, {0u, 0u}};
    if (breakOff) {
        state->brokenOff[kFirst ? 0 : 1] = epoch;
        __hip_atomic_store(brokenOffHost, epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// Every key to its bucket: a workgroup counts its records per bucket in LDS, reserves a run in every bucket it has
// records for with one atomic, puts the records of a bucket next to each other in LDS and stores the runs.  The order
// inside a bucket does not matter: sort_bucket_kernel makes it.  60 million shuffled records: 316 us from records
// (2.3 TB/s), 149 us from keys (3.2 TB/s); stored straight from registers, one line per lane, 416 and 283 us.
template <bool kRecords, int kPerThread>
__global__ void __launch_bounds__(kSortThreads) scatter_keys_kernel(const void* __restrict__ in, u32 count, KeyForm form,
                                                                    int shift, const Bucket* __restrict__ parents,
                                                                    u32 parentCount, u32 target,
                                                                    const unsigned short* __restrict__ childOfBin,
                                                                    u32* __restrict__ cursors, u32* __restrict__ out, u64 epoch,
                                                                    const SortState* __restrict__ state) {
    constexpr u32 kChunk = kPerThread * kSortThreads;
    constexpr int kBins = kRecords ? kBins1 : kBins2;
    typedef std::conditional_t<kRecords, u64, u32> Key;
    __shared__ u32 local[kMaxIds];
    __shared__ u32 keys[kChunk];
    __shared__ unsigned short child[kBins], keyChild[kChunk];
    __shared__ u32 waveSums[kSortThreads / 64];
    __shared__ u32 which;
    if (broken_off(state, epoch)) return;
    u32 begin = blockIdx.x * kChunk, end = min(count - begin, kChunk) + begin, lo = 0;
    if (!kRecords) {
        const u32 b = find_bucket(parents, parentCount, blockIdx.x, kChunk, &which);
        if (b == ~0u) return;
        const Bucket p = parents[b];
        begin = p.start + (blockIdx.x - (p.start / kChunk + b)) * kChunk;
        end = min(p.end - begin, kChunk) + begin;
        lo = p.lo;
        shift = (int)p.shift;
        const u32 firstChild = p.start / target + b;
        cursors += firstChild;
        childOfBin += (size_t)b * kBins2;
    }
    for (u32 i = threadIdx.x; i < (u32)kMaxIds; i += kSortThreads) local[i] = 0;
    for (int i = threadIdx.x; i < kBins; i += kSortThreads) child[i] = childOfBin[i];
    Key v[kPerThread];
    u32 low[kPerThread], bin[kPerThread];
#pragma unroll
    for (int e = 0; e < kPerThread; ++e) v[e] = static_cast<const Key*>(in)[min(begin + e * kSortThreads + threadIdx.x, end - 1)];
#pragma unroll
    for (int e = 0; e < kPerThread; ++e) {
        const u64 k = kRecords ? key_of(v[e], form) : (u64)v[e];
        low[e] = (u32)k;
        bin[e] = kRecords ? (u32)(k >> shift) : (low[e] - lo) >> shift;
        if (begin + e * kSortThreads + threadIdx.x >= end) bin[e] = ~0u;
    }
    __syncthreads();
    u32 rank[kPerThread];
#pragma unroll
    for (int e = 0; e < kPerThread; ++e)
        if (bin[e] < (u32)kBins) {
            bin[e] = child[bin[e]];
            rank[e] = atomicAdd(&local[bin[e]], 1u);
        }
    __syncthreads();
    // in LDS, the records of a bucket next to each other: they leave as runs of consecutive addresses
    constexpr int kIdsPerThread = kMaxIds / kSortThreads;
    u32 n[kIdsPerThread], sum = 0;
#pragma unroll
    for (int j = 0; j < kIdsPerThread; ++j) sum += n[j] = local[threadIdx.x * kIdsPerThread + j];
    u32 at = block_exclusive_scan<kSortThreads>(sum, waveSums);
    const u32 mine = at;
#pragma unroll
    for (int j = 0; j < kIdsPerThread; ++j) {
        local[threadIdx.x * kIdsPerThread + j] = at;
        at += n[j];
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < kPerThread; ++e)
        if (bin[e] < (u32)kMaxIds) {
            const u32 place = local[bin[e]] + rank[e];
            keys[place] = low[e];
            keyChild[place] = (unsigned short)bin[e];
        }
    __syncthreads();
    at = mine;
#pragma unroll
    for (int j = 0; j < kIdsPerThread; ++j) {
        const u32 id = threadIdx.x * kIdsPerThread + j;
        if (n[j]) local[id] = atomicAdd(&cursors[id], n[j]) - at;
        at += n[j];
    }
    __syncthreads();
    for (u32 i = threadIdx.x; i < end - begin; i += kSortThreads) out[local[keyChild[i]] + i] = keys[i];
}

// Windows of the buckets that are too large for the LDS: a workgroup reads all keys of the bucket, marks those of its
// window of 2^18 in a bit map and counts those below it, which is where the window's records begin; the windows of a
// bucket know nothing of each other.  Bound by the instructions per key (read, compare, mark), about 10 keys a nanosecond
// and workgroup.  Full chunks of a window leave in runs of up to 64 records (a lane's next records lie 256 bytes from its
// neighbour's otherwise: 64 lines a store), thin ones record by record.
// Measured, whole sorts, one workgroup that goes through all windows of a bucket -> this: a row of a million records, four
// windows, 355 -> 167 us; 20 thousand records, half of them in one row of 300 000, 256 windows, 1450 -> 50; three million,
// half of them in one row of two million, 2598 -> 324.
template <int kThreads, int kWords>
__device__ __forceinline__ void order_windows(const u32* __restrict__ in, const Bucket* __restrict__ buckets,
                                              const u32* __restrict__ windowList, u32 windows, KeyForm form,
                                              u64* __restrict__ records, u32* bits, u32* waveSums, u32* below) {
    typedef u32 LooseU32x4 __attribute__((ext_vector_type(4), aligned(4)));
    constexpr int kChunks = kWords / 64, kUnroll = 2;  // a wave writes out 64 words, a chunk, at a time
    constexpr u32 kThin = 768;                         // records of a chunk that leave one by one
    static_assert(kWords * 32 == 1 << kWindowBits && kWords % (4 * kThreads) == 0 && kChunks * 4 == kThreads, "window");
    __shared__ u32 chunkAt[kChunks];
    const u32 t = threadIdx.x, lane = t & 63;
    for (u32 u = blockIdx.x; u < windows; u += kWindowWorkers) {
        const u32 number = windowList[u] & ((1u << kWindowNumberBits) - 1u);
        const Bucket b = buckets[windowList[u] >> kWindowNumberBits];
        const u32* const keys = in + b.start;
        const u32 m = b.end - b.start, fours = m / 4;
        for (int i = 0; i < kWords / 4 / kThreads; ++i) reinterpret_cast<u32x4*>(bits)[i * kThreads + t] = u32x4{0u, 0u, 0u, 0u};
        __syncthreads();
        u32 less = 0;
        auto mark = [&](u32 key) {
            const u32 at = key - b.lo, w = at >> kWindowBits;
            if (w == number) atomicOr(&bits[(at & ((1u << kWindowBits) - 1u)) >> 5], 1u << (at & 31u));
            less += w < number ? 1u : 0u;
        };
        for (u32 base = 0; base < fours; base += kUnroll * kThreads) {
            u32x4 four[kUnroll];
#pragma unroll
            for (int e = 0; e < kUnroll; ++e) four[e] = reinterpret_cast<const LooseU32x4*>(keys)[min(base + e * kThreads + t, fours - 1)];
#pragma unroll
            for (int e = 0; e < kUnroll; ++e)
                if (base + e * kThreads + t < fours) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) mark(four[e][i]);
                }
        }
        if (t < m % 4) mark(keys[fours * 4 + t]);
        const u32 lessBefore = block_exclusive_scan<kThreads>(less, waveSums);  // (its barrier: the bits are set)
        if (t == kThreads - 1) *below = lessBefore + less;
        // where the records of every chunk go: four threads count one, each 16 words (not all from the same bank)
        u32 n = 0;
#pragma unroll
        for (u32 i = 0; i < 16; ++i) n += __popc(bits[t * 16 + ((i + t) & 15)]);
        n += __shfl_xor(n, 1, 64);
        n += __shfl_xor(n, 2, 64);
        const u32 before = block_exclusive_scan<kThreads>(t % 4 == 0 ? n : 0u, waveSums);
        if (t % 4 == 0) chunkAt[t / 4] = b.start + *below + before;
        __syncthreads();
        const u32 lowest = b.lo + (number << kWindowBits), candidates = (1u << form.candidateBits) - 1u;
        auto put = [&](u64* record, u32 bit) {
            const u32 low = lowest + bit;
            *record = (u64)(low & candidates) << 32 | (__builtin_amdgcn_alignbit(b.window, low, form.candidateBits) + form.firstQuery);
        };
        for (u32 c = t / 64; c < (u32)kChunks; c += kThreads / 64) {
            u32 word = bits[c * 64 + lane];
            if (__builtin_amdgcn_ballot_w64(word != 0u) == 0ull) continue;
            u64* out = records + __builtin_amdgcn_readfirstlane(chunkAt[c]);
            u32 x = __popc(word);
            const u32 mine = x;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const u32 y = __shfl_up(x, off, 64);
                if (lane >= (u32)off) x += y;
            }
            if (__builtin_amdgcn_readlane(x, 63) <= kThin) {
                for (out += x - mine; word; word &= word - 1) put(out++, (c * 64 + lane) * 32 + (__ffs(word) - 1));
            } else {
                for (int j = 0; j < 64; j += 2) {
                    const u32 even = __builtin_amdgcn_readlane(word, j), odd = __builtin_amdgcn_readlane(word, j + 1);
                    if ((lane < 32 ? even : odd) >> (lane & 31) & 1)
                        put(out + __builtin_amdgcn_mbcnt_hi(odd, __builtin_amdgcn_mbcnt_lo(even, 0u)), (c * 64 + j) * 32 + lane);
                    out += __popc(even) + __popc(odd);
                }
            }
        }
        __syncthreads();  // the bits and where they go are read
    }
}

// One bucket.  The key range is cut into at least as many cells as there are keys (half or all of the capacity): a key's cell gives its rank
// up to the few keys that share the cell, which are then counted one by one.  Where keys crowd into few cells (runs of
// consecutive candidates, say), a cell's own key range, from its smallest to its largest key, is cut once more, into as
// many cells as it has keys; what is still crowded then goes through a bitonic network.  The first kWindowWorkers
// workgroups see to the buckets of more keys than the LDS holds.
// Bound by LDS latency between barriers, so four workgroups of 512 share a CU (64 registers; the spills lie on the
// crowded path): 60 million keys 231 us, 380 us with 1024 threads and 8192 keys, two to a CU.
template <bool kRecords, int kThreads, int kCap>
__global__ void __launch_bounds__(kThreads, kRecords ? 4 : 8) sort_bucket_kernel(const void* in, const Bucket* __restrict__ buckets,
                                                                   Bucket whole, KeyForm form, u64* records,
                                                                   const u32* __restrict__ windowList, u64 epoch,
                                                                   const SortState* __restrict__ state) {
    __shared__ __align__(16) u32 lds[2 * kCap];
    __shared__ u32 waveSums[kThreads / 64];
    __shared__ u32 fullest, half;
    constexpr int kPer = kCap / kThreads;
    static_assert(kCap == 8 * kThreads, "two vectors of four cells per thread");
    u32* const cells = lds;
    u32* const keys = lds + kCap;
    Bucket b = whole;
    if constexpr (!kRecords) {
        if (broken_off(state, epoch)) return;
        if (blockIdx.x < (u32)kWindowWorkers) {
            order_windows<kThreads, 2 * kCap>(static_cast<const u32*>(in), buckets, windowList, state->windows, form, records,
                                              lds, waveSums, &half);
            return;
        }
        b = buckets[blockIdx.x - kWindowWorkers];
        if (b.end - b.start > (u32)kCap) return;
    }
    const u32 m = b.end - b.start;
    if (m == 0) return;
    const u32 t = threadIdx.x;
    const u64 high = (u64)b.window << 32, mask = (1ull << form.candidateBits) - 1ull;
    auto put_record = [&](u32 at, u32 low) {
        const u64 k = high | low;
        records[b.start + at] = ((k & mask) << 32) | (u32)((u32)(k >> form.candidateBits) + form.firstQuery);
    };
    const u32 nCells = m <= kCap / 2 ? kCap / 2 : kCap;
    const bool two = nCells == kCap;  // cells 4t .. 4t + 3 belong to thread t, and with all cells those half the capacity further on
    u32 key[kPer], cell[kPer];
    {
        typedef std::conditional_t<kRecords, u64, u32> Key;
        Key v[kPer];
        // (the second half only where it is needed; no branch between the loads of a half)
#pragma unroll
        for (int e = 0; e < kPer / 2; ++e) v[e] = static_cast<const Key*>(in)[b.start + min(e * kThreads + t, m - 1)];
        if (two) {
#pragma unroll
            for (int e = kPer / 2; e < kPer; ++e) v[e] = static_cast<const Key*>(in)[b.start + min(e * kThreads + t, m - 1)];
        }
#pragma unroll
        for (int e = 0; e < kPer; ++e)
            if (e < kPer / 2 || two) key[e] = kRecords ? (u32)key_of(v[e], form) : (u32)v[e];
    }
    // f(e) for every key this thread holds
    auto each = [&](auto&& f) {
#pragma unroll
        for (int e = 0; e < kPer; ++e)
            if (e * kThreads + t < m) f(e);
    };
    auto fill = [&](u32* a, u32 v) {
        const u32x4 v4 = {v, v, v, v};
        reinterpret_cast<u32x4*>(a)[t] = v4;
        if (two) reinterpret_cast<u32x4*>(a)[kThreads + t] = v4;
        __syncthreads();
    };
    // Ranks by cell: counts in `first`, turned into where each cell starts; false if some cell is too full.  Otherwise the
    // sorted keys are in `first` at the end; `other` is overwritten.
    auto order = [&](u32* first, u32* other) {
        u32 place[kPer];
        if (t == 0) fullest = 0;
        fill(first, 0u);
        each([&](int e) { place[e] = atomicAdd(&first[cell[e]], 1u); });
        __syncthreads();
        u32 before = 0;
        for (int h = 0; h < (two ? 2 : 1); ++h) {
            u32x4* const mine = reinterpret_cast<u32x4*>(first) + h * kThreads + t;
            const u32x4 n = *mine;
            if (max(max(n[0], n[1]), max(n[2], n[3])) > kCellMax) fullest = kCellMax + 1;
            const u32 at = before + block_exclusive_scan<kThreads>(n[0] + n[1] + n[2] + n[3], waveSums);
            *mine = u32x4{at, at + n[0], at + n[0] + n[1], at + n[0] + n[1] + n[2]};
            if (two && h == 0) {
                if (t == kThreads - 1) half = at + n[0] + n[1] + n[2] + n[3];
                __syncthreads();
                before = half;
            }
        }
        __syncthreads();
        if (fullest > kCellMax) return false;
        each([&](int e) { other[first[cell[e]] + place[e]] = key[e]; });
        __syncthreads();
        each([&](int e) {
            const u32 begin = first[cell[e]], end = cell[e] + 1 < nCells ? first[cell[e] + 1] : m, own = begin + place[e];
            u32 less = 0;
            for (u32 j = begin; j < end; ++j) {
                const u32 o = other[j];
                less += (o < key[e] || (o == key[e] && j < own)) ? 1u : 0u;
            }
            place[e] = begin + less;
        });
        __syncthreads();
        each([&](int e) { first[place[e]] = key[e]; });
        __syncthreads();
        return true;
    };
    // mulhi(key - lo, scale) < nCells and monotonic for any scale up to nCells / (range + 1) * 2^32
    const double exact = (double)nCells * 4294967296.0 / ((double)(b.last - b.lo) + 1.0);
    const u32 scale = exact >= 4294967295.0 ? 0xffffffffu : (u32)exact;
    each([&](int e) { cell[e] = __umulhi(key[e] - b.lo, scale); });
    const u32* result = cells;
    if (!order(cells, keys)) {
        u32 least[kPer];
        fill(keys, ~0u);
        each([&](int e) { atomicMin(&keys[cell[e]], key[e]); });
        __syncthreads();
        each([&](int e) { least[e] = keys[cell[e]]; });
        __syncthreads();
        fill(keys, 0u);
        each([&](int e) { atomicMax(&keys[cell[e]], key[e]); });
        __syncthreads();
        each([&](int e) {
            const u32 begin = cells[cell[e]], n = (cell[e] + 1 < nCells ? cells[cell[e] + 1] : m) - begin;
            const float perKey = (float)n / ((float)(keys[cell[e]] - least[e]) + 1.0f);
            cell[e] = begin + min(n - 1, (u32)((float)(key[e] - least[e]) * perKey));  // monotonic in the key
        });
        __syncthreads();
        result = keys;
        if (!order(keys, cells)) {
            u32 size = kThreads;
            while (size < m) size <<= 1;
#pragma unroll
            for (int e = 0; e < kPer; ++e) {
                const u32 i = e * kThreads + t;
                if (i < size) keys[i] = i < m ? key[e] : 0xffffffffu;
            }
            __syncthreads();
            for (u32 k = 2; k <= size; k <<= 1)
                for (u32 j = k >> 1; j > 0; j >>= 1) {
                    for (u32 i = t; i < size / 2; i += kThreads) {
                        const u32 a = ((i & ~(j - 1)) << 1) | (i & (j - 1)), c = a | j;
                        const u32 x = keys[a], y = keys[c];
                        if ((x > y) == ((a & k) == 0)) {
                            keys[a] = y;
                            keys[c] = x;
                        }
                    }
                    __syncthreads();
                }
        }
    }
    for (u32 i = t; i < m; i += kThreads) put_record(i, result[i]);
}

unsigned grid_for(unsigned long long count) {
    unsigned long long blocks = (count + 255) / 256;
    return (unsigned)(blocks > 65536ull ? 65536ull : (blocks ? blocks : 1));
}

}  // namespace

void SortBuffers::release() {
    if (alt) (void)hipFree(alt);
    if (temp) (void)hipFree(temp);
    if (tables) (void)hipFree(tables);
    if (hostWord) (void)hipHostFree(hostWord);
    alt = temp = tables = nullptr;
    hostWord = hostWordDev = nullptr;
    altBytes = tempBytes = tableBytes = 0;
}

namespace {

hipError_t grow(void** buffer, size_t* have, size_t need) {
    if (need <= *have) return hipSuccess;
    if (*buffer) (void)hipFree(*buffer);
    *buffer = nullptr;
    *have = 0;
    const hipError_t e = hipMalloc(buffer, need);
    if (e == hipSuccess) *have = need;
    return e;
}

hipError_t radix_temp_bytes(unsigned long long count, size_t* bytes) {
    *bytes = 0;
    const hipError_t e = rocprim::radix_sort_keys(nullptr, *bytes, static_cast<u64*>(nullptr), static_cast<u64*>(nullptr),
                                                  (size_t)count, 0u, 64u, hipStream_t(nullptr));
    if (e == hipSuccess && *bytes == 0) *bytes = 16;
    return e;
}

// How `count` records with keys up to `lastKey` are distributed, and where the tables lie.
struct SortPlan {
    bool twoLevels;
    int shift;               // first level: bin = key >> shift
    u32 target1, ids1, ids2; // two levels: records per first-level bucket; buckets of each level (one level: ids1 only)
    u32 target;              // records per bucket that is ordered in LDS
    u32 maxWindows;          // room for windows of buckets that are too large for the LDS
    size_t cursors1, cursors2, buckets1, buckets2, bins2, childOf1, childOf2, windowList, bytes;  // byte offsets in `tables`
};
constexpr u64 kTwoLevelsFrom = 1ull << 20;
constexpr u64 kTwoLevelsAfterOneFrom = 1ull << 18;  // fewer records go from a distribution that broke off to the radix sort
constexpr u64 kDistributeUpTo = 1ull << 29;
constexpr size_t kBins1At = 64;  // the SortState, then the first level's bins

// false: too many records, or keys of more than 42 bits (a first-level bin would cover more than 2^32 of them)
bool make_plan(u64 count, u64 lastKey, bool twoLevels, SortPlan* p) {
    if (count > kDistributeUpTo || lastKey >> 42) return false;
    p->shift = 0;
    while ((lastKey >> p->shift) >= (u64)kBins1) ++p->shift;
    const u32 windows = (u32)(lastKey >> 32) + 1;
    p->twoLevels = twoLevels;
    p->target = kTargetMax;
    if (!p->twoLevels) {
        // small joins: as many buckets as the chip has compute units to work on them, if that leaves them 512 records
        u64 target = (count + 255) / 256;
        if (target < 512) target = 512;
        if (target < p->target) p->target = (u32)target;
    }
    // Two levels: a bucket too large for the LDS is a single bin of at most 2^32 / kBins2 keys, 16 windows, so there are
    // fewer than count / 256 of them in all.
    p->maxWindows = twoLevels ? (u32)(count >> 8) : kWindowsOneLevel;
    // two levels: about as many buckets in the first as in each of those in the second
    p->target1 = p->twoLevels ? (u32)__builtin_sqrt((double)count * p->target) : p->target;
    p->ids1 = (u32)(count / p->target1) + windows + 1;
    if (p->ids1 > (u32)kMaxIds) return false;
    p->ids2 = p->twoLevels ? (u32)(count / p->target) + p->ids1 : 0u;
    size_t at = kBins1At;
    auto place = [&](size_t bytes) {
        const size_t here = at;
        at = (at + bytes + 255) / 256 * 256;
        return here;
    };
    (void)place(kBins1 * sizeof(u32));
    p->bins2 = place(p->twoLevels ? (size_t)p->ids1 * kBins2 * sizeof(u32) : 0);
    p->cursors1 = place(p->ids1 * sizeof(u32));
    p->cursors2 = place(p->ids2 * sizeof(u32));
    p->buckets1 = place(p->ids1 * sizeof(Bucket));
    p->buckets2 = place(p->ids2 * sizeof(Bucket));
    p->childOf1 = place(kBins1 * sizeof(unsigned short));
    p->childOf2 = place(p->twoLevels ? (size_t)p->ids1 * kBins2 * sizeof(unsigned short) : 0);
    p->windowList = place(p->maxWindows * sizeof(u32));
    p->bytes = at;
    return true;
}

// Orders the records by distribution.  *done stays false when a bucket became too large: the records are as they
// were then.  Synchronises the stream.
hipError_t distribute(u64* records, u32 count, const SortPlan& p, u64 lastKey, KeyForm form, hipStream_t stream,
                      SortBuffers* ws, bool* done) {
    hipError_t e = grow(&ws->alt, &ws->altBytes, (size_t)count * sizeof(u32) * (p.twoLevels ? 2 : 1));
    if (e != hipSuccess) return e;
    if (!ws->hostWordDev) {
        if (!ws->hostWord) e = hipHostMalloc(reinterpret_cast<void**>(&ws->hostWord), 64, hipHostMallocCoherent);
        if (e != hipSuccess) return e;
        *ws->hostWord = 0;
        e = hipHostGetDevicePointer(reinterpret_cast<void**>(&ws->hostWordDev), ws->hostWord, 0);
        if (e != hipSuccess) return e;
    }
    const size_t binsEnd = p.bins2 + (size_t)(p.twoLevels ? p.ids1 : 0u) * kBins2 * sizeof(u32);
    if (p.bytes > ws->tableBytes || binsEnd > ws->cleanBytes || ws->tablesDirty) {
        // the bins are zero before a sort and left zeroed by it: cleared here only when the layout moves or a sort broke off
        e = grow(&ws->tables, &ws->tableBytes, p.bytes);
        if (e == hipSuccess) e = hipMemsetAsync(ws->tables, 0, ws->tableBytes, stream);
        if (e != hipSuccess) return e;
    }
    ws->tablesDirty = true;
    char* const base = static_cast<char*>(ws->tables);
    auto* const state = reinterpret_cast<SortState*>(base);
    u32* const bins1 = reinterpret_cast<u32*>(base + kBins1At);
    u32* const bins2 = reinterpret_cast<u32*>(base + p.bins2);
    u32* const cursors1 = reinterpret_cast<u32*>(base + p.cursors1);
    u32* const cursors2 = reinterpret_cast<u32*>(base + p.cursors2);
    Bucket* const buckets1 = reinterpret_cast<Bucket*>(base + p.buckets1);
    Bucket* const buckets2 = reinterpret_cast<Bucket*>(base + p.buckets2);
    auto* const childOf1 = reinterpret_cast<unsigned short*>(base + p.childOf1);
    auto* const childOf2 = reinterpret_cast<unsigned short*>(base + p.childOf2);
    u32* const windowList = reinterpret_cast<u32*>(base + p.windowList);
    const u64 epoch = ++ws->epoch;
    const u32 lastHigh = (u32)(lastKey >> 32), lastLow = (u32)lastKey;
    const dim3 threads(kSortThreads);
    auto blocks = [](u64 n, u64 per) { return dim3((unsigned)((n + per - 1) / per)); };
    u32* const keysA = static_cast<u32*>(ws->alt);
    u32* const keysB = keysA + count;
    const Bucket none{};
    if (!p.twoLevels) {
        count_keys_kernel<true><<<blocks(count, 4096), threads, 0, stream>>>(records, count, form, p.shift, nullptr, 0u, 4096u, bins1, state);
        plan_buckets_kernel<true><<<1, threads, 0, stream>>>(bins1, count, p.shift, lastHigh, lastLow, nullptr, p.target, p.ids1, 0u,
                                                             buckets1, childOf1, cursors1, windowList, p.maxWindows, state, epoch,
                                                             ws->hostWordDev);
        scatter_keys_kernel<true, 4><<<blocks(count, 4096), threads, 0, stream>>>(records, count, form, p.shift, nullptr, 0u, p.target,
                                                                                  childOf1, cursors1, keysA, epoch, state);
        sort_bucket_kernel<false, kBucketThreads, kBucketCap><<<p.ids1 + kWindowWorkers, kBucketThreads, 0, stream>>>(
            keysA, buckets1, none, form, records, windowList, epoch, state);
    } else {
        const u32 chunk1 = (u32)((count / 1024 + 4095) / 4096 * 4096 + 4096), chunk2 = 32768;
        constexpr u32 kScatter = 8 * kSortThreads;
        count_keys_kernel<true><<<blocks(count, chunk1), threads, 0, stream>>>(records, count, form, p.shift, nullptr, 0u, chunk1, bins1, state);
        plan_buckets_kernel<true><<<1, threads, 0, stream>>>(bins1, count, p.shift, lastHigh, lastLow, nullptr, p.target1, p.ids1, p.target,
                                                             buckets1, childOf1, cursors1, windowList, 0u, state, epoch, ws->hostWordDev);
        scatter_keys_kernel<true, 8><<<blocks(count, kScatter), threads, 0, stream>>>(
            records, count, form, p.shift, nullptr, 0u, p.target1, childOf1, cursors1, keysA, epoch, state);
        count_keys_kernel<false><<<count / chunk2 + p.ids1, threads, 0, stream>>>(keysA, count, form, 0, buckets1, p.ids1, chunk2, bins2, state);
        plan_buckets_kernel<false><<<p.ids1, threads, 0, stream>>>(bins2, count, 0, 0u, 0u, buckets1, p.target, p.ids2, 0u,
                                                                   buckets2, childOf2, cursors2, windowList, p.maxWindows, state, epoch,
                                                                   ws->hostWordDev);
        scatter_keys_kernel<false, 8><<<count / kScatter + p.ids1, threads, 0, stream>>>(
            keysA, count, form, 0, buckets1, p.ids1, p.target, childOf2, cursors2, keysB, epoch, state);
        sort_bucket_kernel<false, kBucketThreads, kBucketCap><<<p.ids2 + kWindowWorkers, kBucketThreads, 0, stream>>>(
            keysB, buckets2, none, form, records, windowList, epoch, state);
    }
    e = hipGetLastError();
    const hipError_t s = hipStreamSynchronize(stream);
    if (e == hipSuccess) e = s;
    if (e != hipSuccess) return e;
    *done = *static_cast<volatile u64*>(ws->hostWord) != epoch;
    ws->tablesDirty = !*done;
    ws->cleanBytes = binsEnd;
    return hipSuccess;
}

hipError_t radix_sort(u64* keys, u64 count, KeyForm form, int keyBits, hipStream_t stream, SortBuffers* ws) {
    size_t tempBytes = 0;
    hipError_t e = radix_temp_bytes(count, &tempBytes);
    if (e == hipSuccess) e = grow(&ws->alt, &ws->altBytes, (size_t)count * sizeof(u64));
    if (e == hipSuccess) e = grow(&ws->temp, &ws->tempBytes, tempBytes);
    if (e == hipSuccess) {
        tempBytes = ws->tempBytes;
        auto* const alt = static_cast<u64*>(ws->alt);
        pack_pairs_kernel<<<grid_for(count), 256, 0, stream>>>(keys, keys, count, form.candidateBits);
        e = rocprim::radix_sort_keys(ws->temp, tempBytes, keys, alt, (size_t)count, 0u, (unsigned)keyBits, stream);
        if (e == hipSuccess) {
            unpack_pairs_kernel<<<grid_for(count), 256, 0, stream>>>(alt, keys, count, form.candidateBits);
            e = hipGetLastError();
        } else {
            // the keys are still in place, packed: put the records back as they were
            unpack_pairs_kernel<<<grid_for(count), 256, 0, stream>>>(keys, keys, count, form.candidateBits);
        }
    }
    const hipError_t s = hipStreamSynchronize(stream);
    return e == hipSuccess ? s : e;
}

}  // namespace

size_t sort_scratch_bytes(unsigned long long count) {
    size_t needTemp = 0;
    if (radix_temp_bytes(count, &needTemp) != hipSuccess) return 0;
    SortPlan p{};
    const size_t tables = make_plan(count ? count : 1, (1ull << 42) - 1, true, &p) ? p.bytes : 0;
    return needTemp + tables + (size_t)count * sizeof(u64);
}

hipError_t sort_pairs_row_major(void* pairs, unsigned long long count, hipStream_t stream, SortBuffers* ws,
                                long long firstQuery, long long nQueries, long long nCandidates) {
    if (count < 2) return hipSuccess;
    auto* const records = static_cast<u64*>(pairs);
    const int queryBits = index_bits(firstQuery + nQueries), candidateBits = index_bits(nCandidates);
    const u64 lastKey = ((u64)(nQueries - 1) << candidateBits) | (u64)(nCandidates - 1);
    const KeyForm form{candidateBits, (u32)firstQuery};
    if (count <= (u64)kAloneCap && lastKey >> 32 == 0) {
        const Bucket whole{0u, (u32)count, 0u, 0u, (u32)lastKey, 0u, {0u, 0u}};
        sort_bucket_kernel<true, kSortThreads, kAloneCap><<<1, kSortThreads, 0, stream>>>(records, nullptr, whole, form, records, nullptr, 0ull,
                                                                                                 nullptr);
        const hipError_t e = hipGetLastError(), s = hipStreamSynchronize(stream);
        return e == hipSuccess ? s : e;
    }
    bool done = false;
    for (bool twoLevels = count > kTwoLevelsFrom; !done; twoLevels = true) {
        SortPlan p{};
        if (!make_plan(count, lastKey, twoLevels, &p)) break;
        const hipError_t e = distribute(records, (u32)count, p, lastKey, form, stream, ws, &done);
        if (e == hipErrorOutOfMemory) {
            (void)hipGetLastError();  // nothing was launched; the radix sort may need less
            break;
        }
        if (e != hipSuccess) return e;
        if (twoLevels || count < kTwoLevelsAfterOneFrom) break;
    }
    return done ? hipSuccess : radix_sort(records, count, form, queryBits + candidateBits, stream, ws);
}

}  // namespace fasted
