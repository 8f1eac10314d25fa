// pair_bits.hip -- the row-major pair list of a join of few points, out of the hit bits that the join kernel has left
// (BitsLayout in join_kernels.h).  It takes the place of staged records and their sort (the reference: source/pair.cuh:123-133,
// 151-158): the bits of a row are in order as they lie, so the list needs counting and nothing else, whatever its length
// and however it crowds, and no count has to come back to the host in between.
#include "join_device.hpp"

namespace fasted {
namespace {

constexpr int kThreads = 512, kWaves = kThreads / 64;
constexpr int kRowsPerWave = kBandRows / kWaves;
constexpr int kMaxRowWords = (kMaxBitRows / 32) | 1;  // an odd pitch: a column of the band is spread over the banks

// Bound by latency: load the band's words, mark, count, write, with a barrier between; 1 to 2 workgroups share a CU (64 KB of
// LDS each).  In place of count, plan, scatter and bucket sort, their launches and the host's wait for the count; join kernel and
// what follows it, us: 1000 x 64 with 5 thousand records 12 + 21 -> 9 + 3.4, 4096 x 128 with
// 123 thousand 17 + 35 -> 14 + 7.6, 9733 x 257 with 954 thousand 54 + 43 -> 47 + 16, 7500 x 128 with 6.9 million 126 + 153 ->
// 25 + 25, 16000 x 128 with 1.0 million 58 + 45 -> 59 + 23, with 15.6 million 287 + 253 -> 61 + 57.
// One workgroup makes the records of a band of 32 query rows.  Its bits come from the tiles of its own row of tiles and, where
// only the tiles above the diagonal were computed, from the tiles above it in its own column, whose columns are its rows.
__global__ void __launch_bounds__(kThreads) expand_bits_kernel(const unsigned* __restrict__ bits, BitsLayout layout, int words, int nQ,
                                                               int nC, unsigned long long* __restrict__ counters,
                                                               unsigned long long* __restrict__ pairs, unsigned long long cap) {
    __shared__ unsigned rows[kBandRows * kMaxRowWords];  // the band, row by row, bit col % 32 of word col / 32
    __shared__ unsigned rowCount[kBandRows], below[kWaves];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const unsigned band = blockIdx.x;
    const unsigned long long started = wall_clock64();
    // where the band's records begin: behind those of the bands before it
    const unsigned hits = threadIdx.x < gridDim.x ? reinterpret_cast<const unsigned*>(counters + kCounterBands)[threadIdx.x * kBandStride] : 0u;
    const unsigned before = wave_sum(threadIdx.x < band || band == 0 ? hits : 0u);  // (the first band adds up all)
    const unsigned pitch = (unsigned)(nC + 31) / 32 | 1u;
    for (unsigned i = threadIdx.x; i < kBandRows * pitch; i += kThreads) rows[i] = 0u;
    if (lane == 0) below[wave] = before;
    __syncthreads();

    const unsigned bandsPerTile = (unsigned)layout.tileRows / kBandRows;
    const unsigned T = band / bandsPerTile, s = band % bandsPerTile;
    const unsigned perTile = 8u * (unsigned)words * 64u;
    const int quad = lane >> 4, l16 = lane & 15;
    auto mark = [&](unsigned row, unsigned col) { atomicOr(&rows[row * pitch + (col >> 5)], 1u << (col & 31u)); };
    // four words at a time: the four waves' sub-tiles beside each other in a tile of the band's own row
    for (unsigned tc = (layout.upper ? T : 0u) + (unsigned)wave; tc < layout.tileCols; tc += kWaves) {
        const unsigned* const p = bits + (size_t)(T * layout.tileCols + tc) * perTile + (s / (unsigned)words) * 4u * (unsigned)words * 64u +
                                  (s % (unsigned)words) * 64u;
        unsigned v[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = p[k * words * 64 + lane];
#pragma unroll
        for (int k = 0; k < 4; ++k)
            while (v[k]) {
                const unsigned e = (unsigned)__builtin_clz(v[k]);
                v[k] &= ~(0x80000000u >> e);
                mark((e >> 4) * 16u + (unsigned)quad * 4u + (e & 3u), tc * 256u + k * 64u + (e >> 2 & 3u) * 16u + (unsigned)l16);
            }
    }
    // and the four words of a sub-tile of a tile above the diagonal, those bits of them that lie in the band's columns
    if (layout.upper) {
        const unsigned mine = s % 2 ? 0x00ff00ffu : 0xff00ff00u;
        for (unsigned u = (unsigned)wave; u < 2 * T; u += kWaves) {
            const unsigned t = u / 2, half = u % 2;
            const unsigned* const p = bits + (size_t)(t * layout.tileCols + T) * perTile + (half * 4u + s / 2) * 256u;
            unsigned v[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) v[k] = p[k * 64 + lane] & mine;
#pragma unroll
            for (int k = 0; k < 4; ++k)
                while (v[k]) {
                    const unsigned e = (unsigned)__builtin_clz(v[k]);
                    v[k] &= ~(0x80000000u >> e);
                    mark((e >> 2 & 1u) * 16u + (unsigned)l16, t * 256u + half * 128u + k * 32u + (e >> 4) * 16u + (unsigned)quad * 4u + (e & 3u));
                }
        }
    }
    __syncthreads();

    const unsigned rowWords = (unsigned)(nC + 31) / 32;
#pragma unroll
    for (int r = 0; r < kRowsPerWave; ++r) {
        const unsigned* const row = &rows[(wave * kRowsPerWave + r) * pitch];
        unsigned n = 0;
        for (unsigned i = lane; i < rowWords; i += 64) n += (unsigned)__builtin_popcount(row[i]);
        n = wave_sum(n);
        if (lane == 0) rowCount[wave * kRowsPerWave + r] = n;
    }
    __syncthreads();
    unsigned first = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) first += below[w];
    if (band == 0) {
        if (threadIdx.x == 0) {
            unsigned long long* const host = reinterpret_cast<unsigned long long*>(counters[kCounterHostWords]);
            counters[kCounterFound] = first;
            if (host) {
                __hip_atomic_store(&host[0], (unsigned long long)first, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                __hip_atomic_store(&host[1], counters[kCounterStampNorms], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                __hip_atomic_store(&host[3], started | 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            }
        }
        first = 0;
    }
    const unsigned count = lane < kBandRows ? rowCount[lane] : 0u;
    const unsigned rowEnd = wave_inclusive_scan(count);
#pragma unroll
    for (int r = 0; r < kRowsPerWave; ++r) {
        const unsigned inBand = (unsigned)(wave * kRowsPerWave + r);
        const unsigned* const row = &rows[inBand * pitch];
        const unsigned long long query = band * kBandRows + inBand;
        unsigned at = first + (unsigned)__builtin_amdgcn_readlane((int)(rowEnd - count), (int)inBand);
        for (unsigned i = 0; i < rowWords; i += 64) {
            unsigned word = i + lane < rowWords ? row[i + lane] : 0u;
            const unsigned n = (unsigned)__builtin_popcount(word);
            const unsigned end = wave_inclusive_scan(n);
            unsigned slot = at + end - n;
            while (word) {
                const unsigned long long col = (i + (unsigned)lane) * 32u + (unsigned)__builtin_ctz(word);
                word &= word - 1u;
                if (slot < cap) pairs[slot] = query | col << 32;
                ++slot;
            }
            at += (unsigned)__builtin_amdgcn_readlane((int)end, 63);
        }
    }
    if (band + 1 == gridDim.x) {
        __syncthreads();
        if (threadIdx.x == 0) {
            unsigned long long* const host = reinterpret_cast<unsigned long long*>(counters[kCounterHostWords]);
            if (host) __hip_atomic_store(&host[4], wall_clock64(), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
}

}  // namespace

hipError_t launch_expand_bits(const unsigned* bits, const BitsLayout& layout, int nQ, int nC, unsigned long long* counters,
                              void* pairs, unsigned long long cap, hipStream_t stream) {
    if (nQ > kMaxBitRows || nC > kMaxBitRows) return hipErrorInvalidValue;
    const int bands = (nQ + kBandRows - 1) / kBandRows;
    expand_bits_kernel<<<dim3((unsigned)bands), dim3(kThreads), 0, stream>>>(bits, layout, layout.tileRows / 64, nQ, nC, counters,
                                                                             static_cast<unsigned long long*>(pairs), cap);
    return hipGetLastError();
}

}  // namespace fasted
