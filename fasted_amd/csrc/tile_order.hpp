// tile_order.hpp -- the order in which the join kernels walk the tiles of the distance matrix, and where
// the 16-byte chunks of an operand row go in LDS.  Plain C++ (host and device): the kernels use it with
// compile-time tile shapes, the library exports host mirrors of it, and a host-only build checks it
// under the address and undefined-behaviour sanitizers.
//
// Counterpart of Raster::OnDemandRasterizer (source/rasterizer/onDemandRasterizer.cuh:50-108) and
// SimSearch::SwizzleAddress (source/findPairs.cuh:161-166), re-cut for 8 accelerator dies (XCDs) with
// private L2 caches and for the 64-bank LDS of gfx950.
#pragma once

#if defined(__HIPCC__)
#define FASTED_HD __host__ __device__
#else
#define FASTED_HD
#endif
// (a call that is left in a kernel would take the kernel's variables out of its registers)
#define FASTED_INLINE FASTED_HD inline __attribute__((always_inline))

namespace fasted {

constexpr int kQueues = 8;     // one work queue per XCD
constexpr int kSubTiles = 32;  // tiles that a queue takes in a row: one to each of the workgroups resident on one XCD

// Work queues.  The matrix of tiles is cut into super-squares of 4 * subRows x 2 * subCols tiles; a
// super-square is cut into 8 sub-rectangles of subRows x subCols
// tiles, one per XCD, arranged 4 (down) x 2 (across).  Each XCD has its own queue head: position t of
// queue q is tile t % (subRows * subCols), row-major, of sub-rectangle q of super-square t / (subRows *
// subCols); the super-squares follow each other along a row of the matrix.  The workgroups resident on one
// XCD therefore work on a few query panels and candidate panels at a time and share them through that
// XCD's L2, all 8 XCDs stay inside one super-square, and from one super-square to the next the query
// panels stay (the Infinity Cache holds them) while only the candidate panels are new: the taller the
// super-square, the fewer bytes come from HBM.
struct TileOrder {
    unsigned tileRows, tileCols;  // tiles along the queries / the candidates
    unsigned squareCols;          // super-squares per row of super-squares
    unsigned upperOnly;           // symmetric self-join: only the super-squares that reach the diagonal or lie above it
    unsigned long long perQueue;  // positions each queue serves
};

// With `upperOnly` (square matrix, square tiles, super-squares a whole number of times taller than wide:
// ratio = height / width) row i of super-squares keeps the squares from column ratio * i on: those hold
// every tile on or above the diagonal.  Row i starts at position i * S - ratio * i * (i - 1) / 2 of that order.
FASTED_HD inline unsigned long long tile_order_row_start(unsigned long long squareCols, unsigned ratio, long long row) {
    return (unsigned long long)row * squareCols - (unsigned long long)ratio * (unsigned long long)(row * (row - 1) / 2);
}

FASTED_HD inline TileOrder make_tile_order(long long nQueries, long long nCandidates, int tileM, int tileN,
                                           int subRows, int subCols, bool upperOnly) {
    TileOrder r;
    r.tileRows = (unsigned)((nQueries + tileM - 1) / tileM);
    r.tileCols = (unsigned)((nCandidates + tileN - 1) / tileN);
    const unsigned height = 4u * (unsigned)subRows, width = 2u * (unsigned)subCols;  // of a super-square, in tiles
    const unsigned squareRows = (r.tileRows + height - 1) / height;
    r.squareCols = (r.tileCols + width - 1) / width;
    r.upperOnly = (upperOnly && height % width == 0 && tileM == tileN && r.tileRows == r.tileCols) ? 1u : 0u;
    const unsigned long long squares = r.upperOnly ? tile_order_row_start(r.squareCols, height / width, squareRows)
                                                   : (unsigned long long)squareRows * r.squareCols;
    r.perQueue = squares * (unsigned)(subRows * subCols);
    return r;
}

// Position t of queue q -> tile (row, col) in tile units, for the sub-rectangle shape the order was made
// with.  Tiles outside the tileRows x tileCols grid are padding of the last super-squares: the caller
// skips them.
FASTED_HD inline void tile_order_decode(const TileOrder& r, int subRows, int subCols, unsigned q,
                                        unsigned long long t, unsigned* tr, unsigned* tc) {
    const unsigned subTiles = (unsigned)(subRows * subCols);
    const unsigned long long sq = t / subTiles;
    const unsigned local = (unsigned)(t % subTiles);
    const unsigned height = 4u * (unsigned)subRows, width = 2u * (unsigned)subCols;
    unsigned squareRow, squareCol;
    if (r.upperOnly) {
        // smaller root of  ratio/2 * i^2 - (S + ratio/2) * i + sq = 0  as an estimate, then corrected
        const unsigned ratio = height / width;
        const unsigned long long S = r.squareCols;
        const long long rowsOfSquares = (long long)((r.tileRows + height - 1) / height);
        const double b = (double)S + 0.5 * (double)ratio;
        const double disc = b * b - 2.0 * (double)ratio * (double)sq;
        long long i = (long long)((b - __builtin_sqrt(disc > 0.0 ? disc : 0.0)) / (double)ratio);
        if (i < 0) i = 0;
        if (i >= rowsOfSquares) i = rowsOfSquares - 1;
        while (i > 0 && tile_order_row_start(S, ratio, i) > sq) --i;
        while (i + 1 < rowsOfSquares && tile_order_row_start(S, ratio, i + 1) <= sq) ++i;
        squareRow = (unsigned)i;
        squareCol = (unsigned)((long long)ratio * i + (long long)(sq - tile_order_row_start(S, ratio, i)));
    } else {
        squareRow = (unsigned)(sq / r.squareCols);
        squareCol = (unsigned)(sq % r.squareCols);
    }
    *tr = squareRow * height + (q >> 1) * (unsigned)subRows + local / (unsigned)subCols;
    *tc = squareCol * width + (q & 1) * (unsigned)subCols + local % (unsigned)subCols;
}

// Number b of the upper triangle of a square tile matrix, column by column ((0,0), (0,1), (1,1), (0,2), ...): tile
// (row, col), row <= col.  The square root is an estimate, then corrected.
FASTED_HD inline void tile_order_upper_decode(unsigned b, unsigned* tr, unsigned* tc) {
    unsigned c = (unsigned)((__builtin_sqrtf(8.0f * (float)b + 1.0f) - 1.0f) * 0.5f);
    while (c > 0 && c * (c + 1) / 2 > b) --c;
    while ((c + 1) * (c + 2) / 2 <= b) ++c;
    *tc = c;
    *tr = b - c * (c + 1) / 2;
}

// Tile `number` of a matrix of rows x cols tiles taken in strips of four columns, row by row in a strip: 32 consecutive
// numbers are 8 x 4 tiles.  upper: of its upper triangle (rows == cols), diagonal included.  Every number below
// rows * cols, or rows * (rows + 1) / 2, is a tile: no padding, whatever the shape.  (Both products fit 32 bits.)
FASTED_INLINE void tile_strip_decode(unsigned number, unsigned rows, unsigned cols, bool upper, unsigned* tr, unsigned* tc) {
    if (upper) {
        // strips 0 .. j - 1 hold 8 j^2 + 2 j tiles; the root is an estimate, then corrected
        unsigned j = (unsigned)((__builtin_sqrtf(8.0f * (float)number + 1.0f) - 1.0f) * 0.125f);
        while (j > 0 && 8 * j * j + 2 * j > number) --j;
        while (8 * (j + 1) * (j + 1) + 2 * (j + 1) <= number) ++j;
        const unsigned first = 4 * j, width = cols - first < 4 ? cols - first : 4;
        unsigned s = number - (8 * j * j + 2 * j);
        if (s < first * width) {
            *tr = s / width;
            *tc = first + s % width;
        } else {
            s -= first * width;
            unsigned i = 0;  // rows first + i of the strip start at the diagonal
            for (; s >= width - i; ++i) s -= width - i;
            *tr = first + i;
            *tc = first + i + s;
        }
    } else {
        const unsigned strip = number / (4 * rows), s = number % (4 * rows);
        const unsigned width = cols - 4 * strip < 4 ? cols - 4 * strip : 4;
        *tr = s / width;
        *tc = 4 * strip + s % width;
    }
}

// Number, in that order, of the tile at position `pos` of queue q: 32 tiles to a queue in turn.
FASTED_INLINE unsigned long long tile_strip_number(unsigned q, unsigned long long pos) {
    return pos / kSubTiles * (kQueues * kSubTiles) + q * kSubTiles + pos % kSubTiles;
}

// LDS placement of operand rows.  gfx950 serves a ds_read_b128 in four phases of 16 lanes --
// {0-3,12-15,20-23,24-27}, {4-7,8-11,16-19,28-31} and the same two groups +32 -- and the fragment read
// of v_mfma_f32_16x16x32_f16 has lane l on row l%16, 16-byte chunk l/16 of a 32-wide k-step.  A phase is
// conflict free when its 16 lanes touch all 64 four-byte banks once.
//
// Rows of 128 bytes (a 64-wide k-slab, 8 chunks): chunk c of row r is stored at slot c ^ ((r>>1)&7).
FASTED_HD inline int lds_swizzle128(int row) { return (row >> 1) & 7; }
// Rows of 64 bytes (a 32-wide k-step, 4 chunks): chunk c of row r is stored at slot c ^ ((r>>2)&2).
FASTED_HD inline int lds_swizzle64(int row) { return (row >> 2) & 2; }

}  // namespace fasted
