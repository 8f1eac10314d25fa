// pair_bits.hip -- the row-major pair list of a join of few points, out of the hit bits that the join kernel has left
// (BitsLayout in join_kernels.h).  It takes the place of staged records and their sort (the reference: source/pair.cuh:123-133,
// 151-158): the bits of a row are in order as they lie, so the list needs counting and nothing else, whatever its length
// and however it crowds, and no count has to come back to the host in between.
#include "join_device.hpp"

namespace fasted {
namespace {

constexpr int kThreads = 1024, kWaves = kThreads / 64;
constexpr int kRowsPerWave = kBandRows / kWaves;
constexpr int kMaxRowWords = (kMaxBitRows / 32) | 1;  // an odd pitch: a column of the band is spread over the banks
static_assert(2 * (kBandRows * kMaxRowWords * 4 + 256) <= 160 * 1024, "two workgroups to a CU");
static_assert(kMaxBands <= kThreads, "a thread per band");

template <int kControl>
__device__ __forceinline__ unsigned moved(unsigned v) {
    return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, kControl, 0xf, 0xf, true);
}
// One step of a transposition between lanes and fields of a word: fields whose number has the bit clear stay in lanes that have
// it clear, the others change places with those of the lane that differs in it (`other`), `distance` bits away.
__device__ __forceinline__ unsigned exchange(unsigned x, unsigned other, bool set, unsigned distance, unsigned low) {
    const unsigned keep = set ? ~low : low, turned = __builtin_amdgcn_alignbit(other, other, set ? distance : 32u - distance);
    return (x & keep) | (turned & ~keep);
}

// One workgroup makes the records of a band of 32 query rows.  Its bits come from the tiles of its own row of tiles and, where
// only the tiles above the diagonal were computed, from the tiles above it in its own column, whose columns are its rows.
// Instructions bound it, 16 lanes of a vector unit at a time: hence bits that are transposed a word at a time and not marked one
// by one (9733 x 257 with 954 thousand records, a band in the middle: 7.3 -> 3.6 us), and sixteen waves, each with two rows whose
// chains of instructions do not wait for each other (from marked to written 6.5 -> 3.9).  In place of count, plan, scatter and bucket sort, their launches and the host's wait
// for the count; join kernel and what follows it, us: 1000 x 64 with 5 thousand records 12 + 21 -> 9 + 3.4, 4096 x 128 with 123
// thousand 17 + 35 -> 13 + 5, 9733 x 257 with 954 thousand 54 + 43 -> 44 + 12, 4096 x 64 with 2.0 million 47 + 86 -> 12 + 10, 16000 x 128 with
// 1.0 million 58 + 45 -> 50 + 19, with 15.6 million 287 + 253 -> 50 + 46.  Up to 79 tiles a side, two such workgroups share a CU.
__global__ void __launch_bounds__(kThreads, 8) expand_bits_kernel(const unsigned* __restrict__ bits, BitsLayout layout, int words, int nC,
                                                               unsigned long long* __restrict__ counters,
                                                               unsigned long long* __restrict__ pairs, unsigned long long cap) {
    __shared__ unsigned rows[kBandRows * kMaxRowWords];  // the band, row by row, bit col % 32 of word col / 32
    __shared__ unsigned rowCount[kBandRows], below[kWaves];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const unsigned band = blockIdx.x;
    const unsigned long long started = wall_clock64();
    // where the band's records begin: behind those of the bands before it (the first band adds up all)
    const unsigned hits = threadIdx.x < gridDim.x ? reinterpret_cast<const unsigned*>(counters + kCounterBands)[threadIdx.x * kBandStride] : 0u;
    const unsigned before = wave_sum(threadIdx.x < band || band == 0 ? hits : 0u);
    if (lane == 0) below[wave] = before;

    const unsigned bandsPerTile = (unsigned)layout.tileRows / kBandRows;
    const unsigned T = band / bandsPerTile, s = band % bandsPerTile;
    const unsigned pitch = layout.tileCols * 8u | 1u;
    const unsigned perTile = 8u * (unsigned)words * 64u;
    const unsigned quad = (unsigned)lane >> 4, l16 = (unsigned)lane & 15u;
    // Four words of a lane at a time: those of the four sub-tiles beside each other in a tile of the band's own row, or, from a
    // tile above the diagonal in its own column, of one sub-tile, and of them the bits in the band's columns.  A wave loads two
    // such units before it looks at the first: they come from other XCDs, through the Infinity Cache.
    const unsigned firstCol = layout.upper ? T : 0u, direct = layout.tileCols - firstCol, units = direct + (layout.upper ? 2 * T : 0u);
    constexpr unsigned kAhead = 2;
    for (unsigned u0 = (unsigned)wave; u0 < units; u0 += kAhead * kWaves) {
        unsigned v[kAhead][4];
#pragma unroll
        for (unsigned a = 0; a < kAhead; ++a) {
            const unsigned u = u0 + a * kWaves;
            if (u < direct) {
                const unsigned* const p = bits + (size_t)(T * layout.tileCols + firstCol + u) * perTile +
                                          ((s / (unsigned)words) * 4u * (unsigned)words + s % (unsigned)words) * 64u;
#pragma unroll
                for (int k = 0; k < 4; ++k) v[a][k] = p[k * words * 64 + lane];
            } else if (u < units) {
                const unsigned t = (u - direct) / 2, half = (u - direct) % 2;
                const unsigned* const p = bits + (size_t)(t * layout.tileCols + T) * perTile + (half * 4u + s / 2) * 256u;
#pragma unroll
                for (int k = 0; k < 4; ++k) v[a][k] = p[k * 64 + lane];
            }
        }
        // (bit e of a reversed word: row (e >> 4) * 16 + quad * 4 + e % 4, column (e >> 2) % 4 * 16 + l16)
#pragma unroll
        for (unsigned a = 0; a < kAhead; ++a) {
            const unsigned u = u0 + a * kWaves;
            if (u < direct) {
                // Lanes of a group of 16 (columns) and fields of one bit change places: lane (quad, j) then holds 16 columns, of
                // the row and block of columns that bits j and 16 + j stood for.
                unsigned short* const at = reinterpret_cast<unsigned short*>(rows) + (quad * 4u + (l16 & 3u)) * 2u * pitch +
                                           (firstCol + u) * 16u + (l16 >> 2);
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    unsigned x = __builtin_bitreverse32(v[a][k]);
                    x = exchange(x, moved<0x128>(x), l16 & 8u, 8u, 0x00ff00ffu);               // row_ror:8
                    x = exchange(x, moved<0x1b>(moved<0x141>(x)), l16 & 4u, 4u, 0x0f0f0f0fu);  // half mirror, quad 3,2,1,0
                    x = exchange(x, moved<0x4e>(x), l16 & 2u, 2u, 0x33333333u);                // quad 2,3,0,1
                    x = exchange(x, moved<0xb1>(x), l16 & 1u, 1u, 0x55555555u);                // quad 1,0,3,2
                    at[k * 4] = (unsigned short)x;
                    at[16u * 2u * pitch + k * 4] = (unsigned short)(x >> 16);
                }
            } else if (u < units) {
                // The tile's columns are the rows here, and a lane's column stays its row: of every word the four bits of one of
                // the two blocks of columns, for either half; then the groups of 16 lanes and the four words change places.
                unsigned* const at = rows + l16 * pitch + (u - direct) * 4u + quad;
#pragma unroll
                for (unsigned f = 0; f < 2; ++f) {
                    const unsigned block = s % 2 * 2 + f;
                    unsigned x = 0;
#pragma unroll
                    for (unsigned k = 0; k < 4; ++k) {
                        const unsigned w = __builtin_bitreverse32(v[a][k]);
                        x |= __builtin_amdgcn_alignbit(w, w, (4u * block - 4u * k) & 31u) & (0x000f000fu << (4u * k));
                    }
                    x = exchange(x, __shfl_xor(x, 16, 64), quad & 1u, 4u, 0x0f0f0f0fu);
                    x = exchange(x, __shfl_xor(x, 32, 64), quad & 2u, 8u, 0x00ff00ffu);
                    at[f * 16u * pitch] = x;
                }
            }
        }
    }
    __syncthreads();

    const unsigned rowWords = (unsigned)(nC + 31) / 32;
    const unsigned* const row = &rows[wave * kRowsPerWave * pitch];
    unsigned n[kRowsPerWave] = {};
    for (unsigned i = (unsigned)lane; i < rowWords; i += 64) {
#pragma unroll
        for (int r = 0; r < kRowsPerWave; ++r) n[r] += (unsigned)__builtin_popcount(row[r * pitch + i]);
    }
#pragma unroll
    for (int r = 0; r < kRowsPerWave; ++r) {
        const unsigned all = wave_sum(n[r]);
        if (lane == 0) rowCount[wave * kRowsPerWave + r] = all;
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
    unsigned at[kRowsPerWave];
#pragma unroll
    for (int r = 0; r < kRowsPerWave; ++r)
        at[r] = first + (unsigned)__builtin_amdgcn_readlane((int)(rowEnd - count), wave * kRowsPerWave + r);
    const unsigned limit = cap < ~0u ? (unsigned)cap : ~0u;
    for (unsigned i = 0; i < rowWords; i += 64) {
        // (the wave's rows together: their chains of instructions do not wait for each other)
        unsigned word[kRowsPerWave], slot[kRowsPerWave], any = 0;
#pragma unroll
        for (int r = 0; r < kRowsPerWave; ++r) {
            word[r] = i + lane < rowWords ? row[r * pitch + i + lane] : 0u;
            any |= word[r];
        }
#pragma unroll
        for (int r = 0; r < kRowsPerWave; ++r) {
            const unsigned here = (unsigned)__builtin_popcount(word[r]), end = wave_inclusive_scan(here);
            slot[r] = at[r] + end - here;
            at[r] += (unsigned)__builtin_amdgcn_readlane((int)end, 63);
        }
        while (any) {
            any = 0;
#pragma unroll
            for (int r = 0; r < kRowsPerWave; ++r) {
                const unsigned long long col = (i + (unsigned)lane) * 32u + (unsigned)__builtin_ctz(word[r]);
                if (word[r] != 0u && slot[r] < limit) pairs[slot[r]] = (band * kBandRows + (unsigned)(wave * kRowsPerWave + r)) | col << 32;
                word[r] &= word[r] - 1u;
                ++slot[r];
                any |= word[r];
            }
        }
    }
    // The last workgroup to start stands for the last to end.  (With a reading by every workgroup, or by the one with the most
    // records as well, a call of 1000 x 64 took 26.4 us instead of 25.9, of 9733 x 257 69.5 instead of 68.6.)
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
    expand_bits_kernel<<<dim3((unsigned)bands), dim3(kThreads), 0, stream>>>(bits, layout, layout.tileRows / 64, nC, counters,
                                                                             static_cast<unsigned long long*>(pairs), cap);
    return hipGetLastError();
}

}  // namespace fasted
