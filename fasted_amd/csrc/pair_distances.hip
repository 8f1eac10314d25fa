// pair_distances.hip -- Euclidean distance of every listed pair: FP32 sum of squared differences (no cancellation, unlike
// the expansion the join itself tests).  Pairs that name a point outside its set get NaN.
#include <type_traits>

#include "join_kernels.h"

namespace fasted {
namespace {

typedef unsigned int u32;
typedef unsigned long long u64;
typedef u32 u32x4 __attribute__((ext_vector_type(4)));

constexpr int kDistThreads = 256;
constexpr u32 kListCap = 1024;        // pairs that a workgroup holds in LDS
constexpr u32 kTurnPairs = 8u << 20;  // (the list of a stretch, 64 MB, stays in the Infinity Cache for all XCDs)
constexpr u32 kNoRow = ~0u;

// Where the rows of a pair begin, in 16-byte units; kNoRow: the pair names no point.
struct RowPair {
    u32 q, c;
};

// The difference of the low, of the high halves of two words, widened and rounded once, in one instruction (the compiler
// widens both operands first).
__device__ __forceinline__ float diff_lo(u32 a, u32 b) {
    float d;
    asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel_hi:[1,0,1]" : "=v"(d) : "v"(a), "v"(b));
    return d;
}
__device__ __forceinline__ float diff_hi(u32 a, u32 b) {
    float d;
    asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel:[1,0,1] op_sel_hi:[1,0,1]" : "=v"(d) : "v"(a), "v"(b));
    return d;
}

template <int kControl>
__device__ __forceinline__ float add_dpp(float x) {
    return x + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), kControl, 0xf, 0xf, true));
}
// Sum over the kLanes lanes of a group, in every lane of it.
template <int kLanes>
__device__ __forceinline__ float group_sum(float x) {
    x = add_dpp<0xb1>(x);                     // quad_perm 1,0,3,2
    x = add_dpp<0x4e>(x);                     // quad_perm 2,3,0,1
    x = add_dpp<0x141>(x);                    // row_half_mirror: the other quad of 8 lanes
    if (kLanes >= 16) x = add_dpp<0x140>(x);  // row_mirror: the other 8 lanes of 16
    if (kLanes >= 32) x += __shfl_xor(x, 16, 64);
    if (kLanes >= 64) x += __shfl_xor(x, 32, 64);
    return x;
}

// The distances of `n` pairs by one workgroup.  kLanes lanes share a pair, kChunks chunks of 16 bytes of either row each, all
// in registers; a group of lanes takes consecutive pairs, and a query row stays while the pairs that follow name the same
// query.  A lane keeps the sum of every kLanes-th pair of its group, so that a wave takes 64 roots and stores 64 distances
// at a time.  (The next candidate row on its way while this one is worked on costs the registers of half the waves: the
// same time within 2 %, 354 instead of 285 us at 4096 dimensions.)
template <int kLanes, int kChunks, bool kChecked, typename Put>
__device__ __forceinline__ void group_distances(const u32x4* __restrict__ ptsQ, const u32x4* __restrict__ ptsC, int chunksPerRow,
                                                const RowPair* list, u32 n, Put&& put) {
    constexpr u32 kGroups = kDistThreads / kLanes;
    const u32 group = threadIdx.x / kLanes, sub = threadIdx.x % kLanes;
    const u32 per = (n + kGroups - 1) / kGroups, begin = min(group * per, n), end = min(begin + per, n);
    const u32 last = end > begin ? end - 1 : n - 1;  // (a group without pairs goes along with the last)
    const bool whole = (int)sub + (kChunks - 1) * kLanes < chunksPerRow;  // this lane has a last chunk
    auto load = [&](u32x4 (&r)[kChunks], const u32x4* pts, u32 row) {
        const u32x4* const p = pts + (u64)(kChecked && row == kNoRow ? 0u : row) + sub;
#pragma unroll
        for (int k = 0; k + 1 < kChunks; ++k) r[k] = p[k * kLanes];
        if (kLanes == 8) {
            r[kChunks - 1] = p[(kChunks - 1) * kLanes];  // (rows are multiples of 8 chunks)
        } else {
            r[kChunks - 1] = p[whole ? (kChunks - 1) * kLanes : 0];
            if (!whole) r[kChunks - 1] = u32x4{0u, 0u, 0u, 0u};
        }
    };
    u32x4 a[kChunks], b[kChunks];
    float mine = 0.0f;
    u32 query = kNoRow - 1u;
    for (u32 j = 0; j < per; ++j) {
        const RowPair pair = list[min(begin + j, last)];
        load(b, ptsC, pair.c);
        if (pair.q != query) load(a, ptsQ, pair.q);
        query = pair.q;
        float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int k = 0; k < kChunks; ++k) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float lo = diff_lo(a[k][e], b[k][e]), hi = diff_hi(a[k][e], b[k][e]);
                acc[(2 * e) & 3] = __builtin_fmaf(lo, lo, acc[(2 * e) & 3]);
                acc[(2 * e + 1) & 3] = __builtin_fmaf(hi, hi, acc[(2 * e + 1) & 3]);
            }
        }
        float sum = group_sum<kLanes>((acc[0] + acc[1]) + (acc[2] + acc[3]));
        if (kChecked && pair.c == kNoRow) sum = __builtin_nanf("");
        const u32 turn = j % kLanes;
        if (turn == sub) mine = sum;
        if (turn == kLanes - 1 || j + 1 == per) {
            const u32 at = begin + j - turn + sub;
            if (at < end && sub <= turn) put(at, __builtin_sqrtf(mine));
        }
    }
}

// Pairs in the order of the list, `batch` to a workgroup.  Bound by fetching the candidate rows, which come in no order, from
// the Infinity Cache, and for short rows by the vector unit.  Against 16 lanes that walk both rows of every pair, widen
// before they subtract and take one root at a time: 60000 x 64 with 6 million pairs 212 -> 87 us, 16000 x 150 with 640
// thousand 48 -> 29, 15000 x 260 with 300 thousand 38 -> 31, 50021 x 384 with 1 million 116 -> 112.
template <int kLanes, int kChunks>
__global__ void __launch_bounds__(kDistThreads, kChunks <= 6 ? 6 : 5) listed_distances_kernel(const u32x4* __restrict__ ptsQ, u32 ldQ16, int nQ,
                                                                         const u32x4* __restrict__ ptsC, u32 ldC16, int nC,
                                                                         int chunksPerRow, const int2* __restrict__ pairs,
                                                                         u32 count, u32 batch, float* __restrict__ out) {
    __shared__ RowPair list[kListCap];
    const u32 first = blockIdx.x * batch, here = min(batch, count - first);
    for (u32 i = threadIdx.x; i < here; i += kDistThreads) {
        const int2 pr = pairs[first + i];
        const bool valid = pr.x >= 0 && pr.x < nQ && pr.y >= 0 && pr.y < nC;
        list[i] = valid ? RowPair{(u32)pr.x * ldQ16, (u32)pr.y * ldC16} : RowPair{kNoRow, kNoRow};
    }
    __syncthreads();
    group_distances<kLanes, kChunks, true>(ptsQ, ptsC, chunksPerRow, list, here, [&](u32 at, float v) { out[first + at] = v; });
}

// Where the candidates fit the eight L2 caches together but not one of them: the candidates are cut into 8 slices (or a
// multiple), and the workgroups of one XCD -- workgroups are dealt to the XCDs in turn; nothing but time depends on it --
// look through all pairs for those of one slice, whose rows then stay in that XCD's L2.  Bound by what still misses the L2
// (50021 x 384 with 5 million pairs, 4.8 MB to a slice: 16.4 of 38.6 million requests).  With a candidate row in registers ahead
// of its turn, 16 lanes for such rows and a root per pair, of 175 million vector instructions 61 were the arithmetic: 354 -> 291
// us; 20000 x 300 with 2 million 155 (not in slices) -> 92, 60000 x 192 with 3 million 174 (not in slices) -> 108, 5000 x 1000
// with 500 thousand 104 (not in slices) -> 67.  Pairs put in the order of the slices first, by a kernel of its own, so that
// every slice reads its own only: 324 us, 28 of them for the kernel.
template <int kLanes, int kChunks>
__global__ void __launch_bounds__(kDistThreads, kChunks <= 6 ? 6 : 5) sliced_distances_kernel(const u32x4* __restrict__ ptsQ, u32 ldQ16, int nQ,
                                                                      const u32x4* __restrict__ ptsC, u32 ldC16, int nC,
                                                                      int chunksPerRow, const int2* __restrict__ pairs,
                                                                      u32 count, float* __restrict__ out, u32 batchPairs,
                                                                      u32 slices, int sliceRows, u32 stretch) {
    constexpr u32 kWaves = kDistThreads / 64, kPer = kListCap / kDistThreads;
    __shared__ RowPair found[kListCap];  // a workgroup looks through batchPairs <= kListCap pairs
    __shared__ unsigned short where[kListCap];
    __shared__ u32 total;
    // workgroup number = ((pass * batches) + batch) * 8 + XCD, slice = pass * 8 + XCD; the XCDs go through every `stretch`
    // batches from different ones on, each from where its slice lies in a list whose candidates ascend
    const u32 batches = gridDim.x / slices;
    const u32 slice = blockIdx.x / (8 * batches) * 8 + blockIdx.x % 8;
    u32 batch = blockIdx.x / 8 % batches;
    if (stretch != 0) {
        const u32 start = batch / stretch * stretch, length = min(stretch, batches - start);
        batch = start + (batch - start + slice * length / slices) % length;
    }
    const u32 first = batch * batchPairs;
    const u32 here = min(batchPairs, count - first);
    const int lane = threadIdx.x & 63;
    if (threadIdx.x == 0) total = 0;
    __syncthreads();
    {
        const u32 perWave = batchPairs / kWaves, waveFirst = threadIdx.x / 64 * perWave + lane;
        const u32 waveEnd = min(threadIdx.x / 64 * perWave + perWave, here);
        int2 pr[kPer];
#pragma unroll
        for (u32 e = 0; e < kPer; ++e) pr[e] = pairs[first + min(waveFirst + e * 64, here - 1)];
        // the pairs of this slice, in order within a wave
        u64 take[kPer];
        u32 mine = 0;
#pragma unroll
        for (u32 e = 0; e < kPer; ++e) {
            const bool valid = pr[e].x >= 0 && pr[e].x < nQ && pr[e].y >= 0 && pr[e].y < nC;
            const bool real = waveFirst + e * 64 < waveEnd;
            if (!valid && real && slice == 0) out[first + waveFirst + e * 64] = __builtin_nanf("");
            take[e] = __builtin_amdgcn_ballot_w64(real && valid && (u32)pr[e].y - slice * (u32)sliceRows < (u32)sliceRows);
            mine += __builtin_popcountll(take[e]);
        }
        u32 base = 0;
        if (lane == 0) base = atomicAdd(&total, mine);
        base = __builtin_amdgcn_readfirstlane(base);
#pragma unroll
        for (u32 e = 0; e < kPer; ++e) {
            const u32 at = base + __builtin_amdgcn_mbcnt_hi((u32)(take[e] >> 32), __builtin_amdgcn_mbcnt_lo((u32)take[e], 0u));
            if (take[e] >> lane & 1) {
                found[at] = RowPair{(u32)pr[e].x * ldQ16, (u32)pr[e].y * ldC16};
                where[at] = (unsigned short)(waveFirst + e * 64);
            }
            base += __builtin_popcountll(take[e]);
        }
    }
    __syncthreads();
    if (total == 0) return;
    group_distances<kLanes, kChunks, false>(ptsQ, ptsC, chunksPerRow, found, total, [&](u32 at, float v) { out[first + where[at]] = v; });
}

// Rows of any length: 16 lanes walk the two rows of a pair, chunk by chunk.
__global__ void __launch_bounds__(256) pair_distances_kernel(const u32x4* __restrict__ ptsQ, long long ldQ16, int nQ,
                                                                  const u32x4* __restrict__ ptsC, long long ldC16, int nC,
                                                                  int chunksPerRow, const int2* __restrict__ pairs,
                                                                  unsigned long long count, float* __restrict__ out) {
    const int sub = threadIdx.x & 15;
    const unsigned long long groups = ((unsigned long long)gridDim.x * blockDim.x) >> 4;
    for (unsigned long long g = ((unsigned long long)blockIdx.x * blockDim.x + threadIdx.x) >> 4; g < count; g += groups) {
        const int2 pr = pairs[g];
        const bool valid = pr.x >= 0 && pr.x < nQ && pr.y >= 0 && pr.y < nC;
        float acc = 0.0f;
        if (valid) {
            const u32x4* a = ptsQ + (long long)pr.x * ldQ16;
            const u32x4* b = ptsC + (long long)pr.y * ldC16;
            for (int c = sub; c < chunksPerRow; c += 16) {
                const u32x4 x = a[c], y = b[c];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float lo = diff_lo(x[e], y[e]), hi = diff_hi(x[e], y[e]);
                    acc = __builtin_fmaf(lo, lo, acc);
                    acc = __builtin_fmaf(hi, hi, acc);
                }
            }
        }
        acc = group_sum<16>(acc);
        if (sub == 0) out[g] = valid ? __builtin_sqrtf(acc) : __builtin_nanf("");
    }
}

// f(lanes, chunks per lane) as constants: as few lanes per pair as hold the row in six chunks each, up to 64 lanes (of up to
// 8 chunks).  8 lanes hold whole rows; with more, only a lane's last chunk may lie beyond the row.
template <typename F>
void for_row_length(int chunks, F&& f) {
    using std::integral_constant;
    const int lanes = chunks <= 48 ? 8 : chunks <= 96 ? 16 : chunks <= 192 ? 32 : 64;
    const int perLane = (chunks + lanes - 1) / lanes;
    auto up_to = [&](auto lanesC, auto first, auto last) {
        auto each = [&](auto self, auto k) {
            if (perLane == decltype(k)::value) f(lanesC, k);
            if constexpr (decltype(k)::value < decltype(last)::value) self(self, integral_constant<int, decltype(k)::value + 1>{});
        };
        each(each, first);
    };
    integral_constant<int, 1> one;
    integral_constant<int, 4> four;
    integral_constant<int, 6> six;
    integral_constant<int, 8> eight;
    if (lanes == 8) up_to(integral_constant<int, 8>{}, one, six);
    if (lanes == 16) up_to(integral_constant<int, 16>{}, four, six);
    if (lanes == 32) up_to(integral_constant<int, 32>{}, four, six);
    if (lanes == 64) up_to(integral_constant<int, 64>{}, four, eight);
}

}  // namespace

hipError_t launch_pair_distances(const void* queries, long long ldQ, int nQ, const void* candidates, long long ldC,
                                 int nC, int dPad, const void* pairs, unsigned long long count, float* out,
                                 hipStream_t stream) {
    if (count == 0) return hipSuccess;
    const auto* const q = static_cast<const u32x4*>(queries);
    const auto* const c = static_cast<const u32x4*>(candidates);
    const auto* const list = static_cast<const int2*>(pairs);
    const int chunks = dPad / 8;
    const u32 ldQ16 = (u32)(ldQ / 8), ldC16 = (u32)(ldC / 8);
    const u64 rowBytes = (u64)dPad * 2, bytes = rowBytes * (u64)nC, sliceBytes = 5ull << 20;
    const u64 slices = 8 * ((bytes + 8 * sliceBytes - 1) / (8 * sliceBytes));
    const u64 batches = (count + kListCap - 1) / kListCap, maxGroups = (1ull << 32) / kDistThreads - 1;  // of a launch
    const bool addressable = (u64)nQ * (u64)(ldQ / 8) < kNoRow && (u64)nC * (u64)(ldC / 8) < kNoRow && count <= 1ull << 30;
    // Slices pay where the candidates do not fit one L2 (10000 x 100 with 600 thousand pairs, 2.6 MB: 22 us in the order of the
    // list, 29 sliced; 3000 x 1000 with 300 thousand, 6 MB: 46 and 49; 12000 x 512 with 360 thousand, 12 MB: 49 and 42), where
    // looking through the list once per slice, 8 bytes a pair, is little against a row (60000 x 64, 128 bytes a row: 81 and
    // 115; 60000 x 128: 111 and 93), and where a query has some pairs to a slice, since its row is fetched again in every
    // slice: three, or two of longer rows (8 slices: 50021 x 384 with 20 a query 112 and 120, 20000 x 300 with 30 51 and 46; 16:
    // 25000 x 1088 with 24 184 and 190, 40000 x 700 with 40 303 and 292; 24: 30000 x 2048 with 60 1003 and 920; 40: 50000 x
    // 2048 with 24 700 and 975).  Less than 100 thousand pairs leave too little for every XCD (2000 x 2500 with 60 thousand 37
    // and 41; 3000 x 2000 with 120 thousand 55 and 47).  Slices of up to 5 MB: 50021 x 384 in 8 of 4.8 MB 291 us, in 16 of
    // 2.4 313; 12000 x 2048 with 1.2 million in 8 of 6.1 MB 354, in 16 of 3.1 285.
    // Between 4 and 8 MB the rows that pass the L2 are few; rows of 1 KB and more pay all the same where there is much to fetch (in
    // the order of the list, sliced: 2000 x 2000, 8.2 MB, with 400 thousand pairs 117 and 93 us, 1 million 266 and 191, in no order
    // 509 and 357; 4000 x 800 with 1.2 million 136 and 130; but 3000 x 1000 with 600 thousand 82 and 73, near candidates 73 and 87).
    const bool large = bytes >= 8ull << 20 || (rowBytes >= 1024 && bytes > 4ull << 20 && count * rowBytes >= 3ull << 29);
    const bool sliced = rowBytes >= 256 && large && slices * 32 <= rowBytes &&
                        count / ((rowBytes < 1024 ? 3 : 2) * slices) >= (u64)nQ && batches >= 96 && batches * slices <= maxGroups && chunks <= 64 * 8 && addressable;
    // In the order of the list, rows of more than 192 chunks are walked by 16 lanes as well as held by 64 (50000 x 2048 with 1.2
    // million pairs 696 and 740 us, near candidates 302 and 277; 6000 x 3000 with 180 thousand 128 and 157).
    if (!sliced && (chunks > 192 || !addressable)) {
        const u64 blocks = (count * 16 + 255) / 256;
        pair_distances_kernel<<<dim3((unsigned)(blocks > 16384ull ? 16384ull : blocks)), dim3(256), 0, stream>>>(
            q, ldQ / 8, nQ, c, ldC / 8, nC, chunks, list, count, out);
        return hipGetLastError();
    }
    for_row_length(chunks, [&](auto lanes, auto perLane) {
        constexpr int kLanes = decltype(lanes)::value, kChunks = decltype(perLane)::value;
        if (sliced) {
            // Where the pairs of a query are few and its candidates are its neighbours in the set, whole batches belong to one
            // slice: all XCDs but one would pass over them at the same time, and the one would have too few.  For longer rows,
            // whose batches take long, the XCDs then start in different places.
            const bool turned = kLanes >= 16 && count / (16 * slices) < (u64)nQ;
            const int sliceRows = (int)(((u64)nC + slices - 1) / slices);
            // Where candidates are the query's neighbours in the set, the pairs of a slice are one piece of the list, and its
            // batches are all the workgroups that its XCD has: less than 50 are halved, and of longer rows less than 20 again.
            // Near candidates, batches of 1024 / 512 / 256 pairs: 3000 x 2000 with 120 thousand pairs (15 batches of 1024 to a
            // slice) 117 / 67 / 46 us, 5000 x 4096 with 150 thousand (18) 176 / 117 / 85, 11000 x 2048 with 396 thousand (24) 197 /
            // 140 / 115, 25000 x 2048 with 1.2 million (51) 505 / 348 / 307, 25000 x 2048 with 2 million (81) 587 / 425 / 480.
            // Others: 47 / 45 / 44, 128 / 130 / 134, 165 / 167 / 172, 637 / 660 / 642, 823 / 865 / 797; 16000 x 384 with 800
            // thousand (98) 57 / 61 / 74.
            const u32 batchPairs = count >= 50ull * kListCap * slices ? kListCap
                                   : kLanes < 32 || count >= 20ull * kListCap * slices ? kListCap / 2 : kListCap / 4;
            const u64 groups = (count + batchPairs - 1) / batchPairs * slices;
            sliced_distances_kernel<kLanes, kChunks><<<dim3((unsigned)groups), dim3(kDistThreads), 0, stream>>>(
                q, ldQ16, nQ, c, ldC16, nC, chunks, list, (u32)count, out, batchPairs, (u32)slices, sliceRows, turned ? kTurnPairs / batchPairs : 0u);
        } else if constexpr (kLanes < 64) {
            // Up to four pairs to a group of 8 lanes, two to a larger one, fewer where that leaves less than 8192 waves (4000 x 64
            // with 32 thousand pairs 14.1 us with one, 14.8 with four; 60000 x 64 with 1.2 million 41 with one, 29 with four;
            // 60000 x 512 with 1.2 million 180 with two, 190 with four).
            const u64 waves = count * kLanes / 64;
            u32 batch = (waves < 2 * 8192 ? 1 : waves < 4 * 8192 || kLanes > 8 ? 2 : 4) * (kDistThreads / kLanes);
            while ((count + batch - 1) / batch > maxGroups) batch *= 2;
            listed_distances_kernel<kLanes, kChunks><<<dim3((unsigned)((count + batch - 1) / batch)), dim3(kDistThreads), 0, stream>>>(
                q, ldQ16, nQ, c, ldC16, nC, chunks, list, (u32)count, batch, out);
        }
    });
    return hipGetLastError();
}

}  // namespace fasted
