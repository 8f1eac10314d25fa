// join_kernels.h -- host-callable launchers of the gfx950 kernels (internal to libfasted).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace fasted {

constexpr int kTile = 256;       // points per tile side (queries x candidates)
constexpr int kSlabK = 64;       // halves of K staged in LDS per pipeline stage
constexpr int kSquareTiles = 256; // tiles of a super-square of the work queues: one per workgroup of a full chip

// A self-join's distance matrix is bitwise symmetric, so the tiles on and above the diagonal hold every pair; the
// pairs of the tiles above it are emitted in both orientations.
enum class Triangle {
    kFull,   // every tile
    kUpper,  // tiles on and above the diagonal
    kAuto    // whichever is the faster one at this size (launch_join)
};

// Hit bits: what a join of few points leaves instead of pairs, one bit per element of the distance matrix, for
// launch_expand_bits to make the row-major pair list from.  Tile (row, col) of tileRows x 256 elements fills the
// words [(row * tileCols + col) * 8 * tileWords, ...): per wave (2 x 4 of them, sub-tiles of tileRows / 2 x 64) tileWords
// of 64 lanes, word p of lane l at p * 64 + l, as the matrix instruction leaves its elements: bit 31 - e of it is
// row p * 32 + (e >> 4) * 16 + (l >> 4) * 4 + e % 4, column (e >> 2) % 4 * 16 + l % 16 of the sub-tile.
struct BitsLayout {
    int tileRows = 0;     // 256, or 128
    unsigned rowsOfTiles = 0, tileCols = 0;
    bool upper = false;   // tiles on and above the diagonal only
};
constexpr int kMaxBitRows = 79 * kTile;            // points of either set of a join that leaves hit bits
constexpr int kBandRows = 32, kMaxBands = 640;     // query rows are counted, and expanded, in bands
static_assert(kMaxBitRows / kBandRows <= kMaxBands, "a counter per band");

struct JoinLaunch {
    const void* queries;         // FP16 rows
    const void* candidates;      // FP16 rows; the same buffer for a self-join
    long long ldQ, ldC;          // row strides in halves (multiples of 8)
    int nQ, nC;                  // real points
    bool selfJoin;               // same set on both sides: (i, i) always counts as a pair
    int forcedStride = 0;        // two sets where query i IS candidate i * forcedStride (a sample of the
                                 // candidates joined against all of them): that pair always counts
    Triangle triangle = Triangle::kFull;  // self-join: which part of the distance matrix is computed
    int d;                       // dimensions; the columns d .. dPad-1 of every row are zeros
    int dPad;                    // K extent, multiple of kSlabK
    const float* halfQ;          // per query point: eps^2/4 - s/2 (s = squared norm), see launch_sum_squared
    const float* halfC;          // ... per candidate point
    unsigned long long* counters;  // counter_words() words: [0] pairs found, [1] non-finite flag, ..., then the queue
                                   // heads.  Word host_words_slot() is the owner's: the device-side address of 4
                                   // words of pinned host memory, or 0.  If set, the join kernel's last workgroup
                                   // writes [0] = pairs found and the device's constant-rate clock [1] when the
                                   // join's first norm kernel started and [3] (never 0) when it was through itself,
                                   // its first workgroup [2] when it started; every pair record of the join is in
                                   // memory when [3] appears.  The kernels of this file never clear that word.
    unsigned long long epoch = 1;  // number of the join: what the norm kernels of THIS join write into the
                                   // non-finite flag (a flag left by an earlier join is not seen)
    void* pairs;                 // FastedPair[cap]
    unsigned long long cap;
    bool epilogue;               // false: contraction only (measurement)
    unsigned* bits = nullptr;    // hit bits are left here (bits_bytes(nQ, nC); neither set above kMaxBitRows points) and
                                 // the bands counted in the counter block; no pairs, no count, no report
};

// Device bytes of the hit bits of a join, in either tile height.
size_t bits_bytes(int nQ, int nC);
// The row-major list out of the hit bits that a launch_join has left: pairs[0, min(found, cap)).  Reports through the
// counter block's host words: [0] pairs found, [1] clock when the first norm kernel started, [3] (never 0) when this kernel
// did, [4] when its last band was through.
hipError_t launch_expand_bits(const unsigned* bits, const BitsLayout& layout, int nQ, int nC, unsigned long long* counters,
                              void* pairs, unsigned long long cap, hipStream_t stream);

// Host mirror of the device tile order.
// upperOnly: the order of a symmetric self-join (super-squares on and above the diagonal only).
unsigned long long raster_count(long long nQ, long long nC, bool upperOnly = false);
int raster_coord(unsigned long long idx, long long nQ, long long nC, bool upperOnly, int* row, int* col);
int counter_words();
int band_words();  // behind them, for joins that leave hit bits
int host_words_slot();
unsigned long long tile_count(long long nQ, long long nC);  // 256x256 tiles the kernel processes
// Slot (0..7) of 16-byte chunk `chunk` of slab row `row` in LDS (host mirror of the device swizzle).
int lds_chunk_slot(int row, int chunk);

enum class Reset { kNothing = 0, kCounters = 1, kCountersAndBands = 2 };
// Squared norms of n points into `sums` (may be null) and, when `halves` is given, the per-point start value of
// the join's accumulators  h = eps2/4 - s/2  (eps2 = (float)(eps*eps), source/findPairs.cuh:678): the join kernel
// tests  h_q + h_c + q.c >= 0.  A non-finite norm raises the flag in `counters` (the join then tests element
// by element): the flag word receives `epoch`.  With `reset` the kernel also clears the pair counter and the
// queue heads, and the counts of the bands, for the join that follows (no launch_reset_counters needed).
// One launch serves one set of points, or two where a launch can hold the workgroups of both (2^32 - 1 threads).
struct NormPoints {
    const void* points;
    long long ld;
    int n;
    float *sums, *halves;
};
constexpr int kNormThreads = 256;
// Lanes that share a row of dPad halves, and the workgroups of n such rows.
constexpr int norm_lanes(int dPad) {
    int lanes = 64;
    while (lanes > dPad / 8) lanes >>= 1;
    return lanes;
}
constexpr unsigned norm_groups(int n, int dPad) {
    const int rows = kNormThreads / norm_lanes(dPad);
    return (unsigned)(((long long)n + rows - 1) / rows);
}
constexpr bool norms_fit_one_launch(int first, int second, int dPad) {
    return ((unsigned long long)norm_groups(first, dPad) + norm_groups(second, dPad)) * kNormThreads < 1ull << 32;
}
hipError_t launch_sum_squared(const NormPoints& first, const NormPoints* second, int dPad, float eps2, unsigned long long* counters,
                              hipStream_t stream, unsigned long long epoch = 1, Reset reset = Reset::kNothing);
// The same halves from norms that are already there.
hipError_t launch_halves(const float* sums, int n, float eps2, float* halves, unsigned long long* counters,
                         hipStream_t stream, unsigned long long epoch = 1, Reset reset = Reset::kNothing);
// rows x d halves, packed -> rows x dPad halves, the columns d .. dPad-1 zero.  dst is 16-byte aligned, src 2-byte.
hipError_t launch_pad_rows(const void* src, int d, void* dst, int dPad, long long rows, hipStream_t stream);
// *badRows += number of rows whose columns d .. dPad-1 are not all zeros.
hipError_t launch_padding_check(const void* points, long long ld, int n, int d, int dPad, unsigned long long* badRows,
                                hipStream_t stream);
// Clears the queue heads and, unless keepFound, the pair counter (word 0 of `counters`).
hipError_t launch_reset_counters(unsigned long long* counters, bool keepFound, hipStream_t stream);
// pairs[first, last): QueryPoint += qOffset, CandidatePoint += cOffset.
hipError_t launch_offset_pairs(void* pairs, unsigned long long first, unsigned long long last, int qOffset, int cOffset,
                               hipStream_t stream);
// The same for the pairs [min(mark[0], cap), min(counter, cap)) that the join before this launch appended; leaves
// the counter in mark[1].  No host round trip: the range is read on the device.
hipError_t launch_offset_appended_pairs(void* pairs, unsigned long long* mark, const unsigned long long* counters,
                                        unsigned long long cap, int qOffset, int cOffset, hipStream_t stream);
// `layout` (may be null): how the hit bits lie.
hipError_t launch_join(const JoinLaunch& p, hipStream_t stream, BitsLayout* layout = nullptr);
// "" for the library proper; a measurement build of the join kernel (parts compiled out) names itself here.
const char* build_tag();


// Device buffers of the row-major sort: keys on their way, the distribution's tables, the radix sort's own storage.  They
// only grow; a caller that keeps a SortBuffers across calls sorts without allocating.
struct SortBuffers {
    void* alt = nullptr;
    size_t altBytes = 0;
    void* temp = nullptr;
    size_t tempBytes = 0;
    void* tables = nullptr;
    size_t tableBytes = 0, cleanBytes = 0;  // the first cleanBytes hold no counts but zeros (where bins lie)
    bool tablesDirty = false;               // a sort has not run to its end
    unsigned long long* hostWord = nullptr;  // pinned: number of the last sort in which a bucket became too large
    unsigned long long* hostWordDev = nullptr;
    unsigned long long epoch = 0;            // number of the sort
    void release();
};
// Row-major sort (pair_sort.hip) of `count` distinct stored pairs whose indices lie in [firstQuery, firstQuery + nQueries)
// and [0, nCandidates); synchronises the stream.  On failure (no memory for the buffers) the pairs are left as they
// were, unsorted.
hipError_t sort_pairs_row_major(void* pairs, unsigned long long count, hipStream_t stream, SortBuffers* ws,
                                long long firstQuery, long long nQueries, long long nCandidates);
// Device bytes a sort of `count` pairs needs beside the pairs themselves.
size_t sort_scratch_bytes(unsigned long long count);

// out[i] = Euclidean distance of pair i (FP32 sum of squared differences over dPad dimensions; pair_distances.hip); NaN for
// a pair that names a point outside [0, nQ) x [0, nC).
hipError_t launch_pair_distances(const void* queries, long long ldQ, int nQ, const void* candidates, long long ldC,
                                 int nC, int dPad, const void* pairs, unsigned long long count, float* out,
                                 hipStream_t stream);

}  // namespace fasted
