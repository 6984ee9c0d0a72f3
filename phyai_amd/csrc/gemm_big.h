// What the pipelined tile kernels share (gemm_big.hip; gemm_tall.hip: tiles of 144 .. 256 rows x 256 columns): the order of the tiles over XCDs, the swizzle and operand blocks of the staged rows.
#pragma once

#include "fp8_device.h"
#include "launch.h"
#include "tuning.h"
#include <stdlib.h>

namespace phyai {

constexpr int BIG_BK = 128;   // bytes of K per LDS row: one L2 cache line

// Workgroup id -> tile.  Workgroups go to the 8 XCDs round-robin (id % 8) and each XCD has its own
// L2, so ids are laid out for the tiles that share an XCD at a time to share operands: the tile
// grid is cut into bands of 4 tile rows; inside a band, 8 consecutive ids are 8 neighbouring
// tile columns (one per XCD), and the next 8 ids the same columns one tile row further down.  An
// XCD thus works on all (up to 4) tile rows of one tile column together - the weight rows come
// from HBM once per band - while the activation rows of the band stay in its L2.
// Tile columns beyond the last multiple of 8 would leave some XCDs a whole column more than
// others (20 columns: three for XCDs 0-3, two for the rest, and the launch lasts as long as the
// busiest XCD).  The tiles of those last columns are therefore taken in column-major order and
// cut into 8 runs of equal length (within one), one per XCD: still whole or half columns per
// XCD, and every XCD gets the same number of tiles.  Ids past an XCD's run have no tile.
struct BigTile { int m, n; };
// Tile order, weight layout, kind of row scale and of rows (GemmProblem::xq_padded) in one argument.
inline int big_order(int band, int by_rows, int operand_w, int scale_is_scalar, int padded) {
    return band | by_rows << 8 | operand_w << 10 | scale_is_scalar << 11 | padded << 12;
}
// Quotients of uniform values below 2^24 through the reciprocal: what stands between a wavefront's start and its first
// request, five of them in a row, at a third of the instructions of an integer division.
__device__ __forceinline__ int big_div(int n, int d) {
    int quot = (int)((float)n * __builtin_amdgcn_rcpf((float)d));
    const int rest = n - quot * d;
    quot += rest >= d ? 1 : 0;
    quot -= rest < 0 ? 1 : 0;
    return __builtin_amdgcn_readfirstlane(quot);
}
__device__ __forceinline__ BigTile big_tile_of(int id, int m_tiles, int n_tiles, int band_rows) {
    const int full = n_tiles >> 3, rest = n_tiles & 7;   // whole groups of 8 tile columns; columns after them
    const int per_band = 8 * (band_rows * full + ((rest * band_rows + 7) >> 3));
    const int band = big_div(id, per_band);
    const int local = id - band * per_band;
    const int bm = m_tiles - band_rows * band < band_rows ? m_tiles - band_rows * band : band_rows;
    BigTile t;
    if (local < 8 * bm * full) {
        const int col = big_div(local >> 3, bm);
        t.n = col * 8 + (local & 7);
        t.m = band_rows * band + (local >> 3) - col * bm;
    } else {
        const int j = local - 8 * bm * full, x = j & 7, total = rest * bm;
        const int e = ((x * total) >> 3) + (j >> 3);                  // (j / 8)-th tile of XCD x's run
        const int col = big_div(e, bm);
        t.n = e < (((x + 1) * total) >> 3) ? 8 * full + col : n_tiles;   // n_tiles: no tile
        t.m = band_rows * band + e - col * bm;
    }
    return t;
}
// The same order as each XCD's own list: its i-th tile, without the ids that have none (n = n_tiles past the end of the list).
__device__ __forceinline__ BigTile big_tile_of_xcd(int x, int i, int m_tiles, int n_tiles, int band_rows) {
    const int full = n_tiles >> 3, rest = n_tiles & 7, bands = big_div(m_tiles, band_rows);
    auto run = [&](int total) { return (((x + 1) * total) >> 3) - ((x * total) >> 3); };
    const int per_band = band_rows * full + run(rest * band_rows);
    int band = per_band ? big_div(i, per_band) : bands;
    band = band < bands ? band : bands;
    const int local = i - band * per_band, bm = band < bands ? band_rows : m_tiles - bands * band_rows;
    BigTile t = {0, n_tiles};
    if (local < bm * full) {
        const int col = big_div(local, bm);
        t.n = col * 8 + x;
        t.m = band_rows * band + local - col * bm;
    } else if (local - bm * full < run(rest * bm)) {
        const int e = ((x * rest * bm) >> 3) + local - bm * full, col = big_div(e, bm);
        t.n = 8 * full + col;
        t.m = band_rows * band + e - col * bm;
    }
    return t;
}
// Tiles of the busiest XCD under that order (host side; the same arithmetic: whole bands and the last one).
inline int big_max_tiles_per_xcd(int m_tiles, int n_tiles, int band_rows) {
    const int full = n_tiles >> 3, rest = n_tiles & 7, bands = m_tiles / band_rows, last = m_tiles % band_rows;
    int mx = 0;
    for (int x = 0; x < 8; ++x) {
        const int of_band = (((x + 1) * rest * band_rows) >> 3) - ((x * rest * band_rows) >> 3);
        const int of_last = (((x + 1) * rest * last) >> 3) - ((x * rest * last) >> 3);
        const int n = m_tiles * full + bands * of_band + of_last;
        mx = n > mx ? n : mx;
    }
    return mx;
}
// Ids that order needs (host side).
inline int big_grid_ids(int m_tiles, int n_tiles, int band_rows) {
    const int full = n_tiles >> 3, rest = n_tiles & 7;
    const int bands = m_tiles / band_rows, last = m_tiles % band_rows;
    return bands * 8 * (band_rows * full + ((rest * band_rows + 7) >> 3)) +
           (last ? 8 * (last * full + ((rest * last + 7) >> 3)) : 0);
}

// Swizzle of the eight 16-byte chunks of a 128-byte row.  LDS has 64 banks of 4 bytes, so one
// pass over the banks spans two rows and a 128-bit read is served 16 lanes at a time: the eight
// rows of equal parity among 16 consecutive ones must land in different chunk columns.
__device__ __forceinline__ int big_swizzle(int row) { return (row >> 1) & 7; }

// Operand block of v_mfma_f32_16x16x128: 16 rows x 128 bytes of K; lane (l16, q) supplies 32 of the 128 bytes of row
// l16.  Which 32 is free as long as A and B agree: chunks q and 4 + q, so that a quarter of a wavefront reads one chunk
// column.  `row`: the block's first row plus l16.
__device__ __forceinline__ v8i big_join(v4i lo, v4i hi) {
    v8i f;
    f[0] = lo[0]; f[1] = lo[1]; f[2] = lo[2]; f[3] = lo[3];
    f[4] = hi[0]; f[5] = hi[1]; f[6] = hi[2]; f[7] = hi[3];
    return f;
}
__device__ __forceinline__ v8i big_frag(const uint8_t* buf, int row, int q) {
    const int sw = big_swizzle(row);
    const uint8_t* r = buf + row * BIG_BK;
    return big_join(*reinterpret_cast<const v4i*>(r + ((q ^ sw) << 4)), *reinterpret_cast<const v4i*>(r + (((4 + q) ^ sw) << 4)));
}
// ---- host side -------------------------------------------------------------------------------------

inline int big_ceil_div(int a, int b) { return (a + b - 1) / b; }

inline int big_tiles(int M, int N, int epilogue, int bm, int bn) {
    const bool gated = epi_is_gated(epilogue);
    return big_ceil_div(M, bm) * big_ceil_div(gated ? N / 2 : N, gated ? bn / 2 : bn);
}

// Whether an XCD takes tile rows instead of tile columns, the bytes from HBM that this was chosen by, and the tiles that the
// busiest XCD then has.
// By default an XCD takes tile columns: its L2 then holds the weight rows of those columns once, but every XCD streams all
// activation rows it meets.  With few tile columns and long rows of activations (816 x B tokens into a 16384 -> 2048
// projection) that is eight copies of the larger operand; then the roles are exchanged.  Estimated bytes: the operand an XCD
// does not own is read once per XCD (up to 8 times), the other once per band.  (6528 x 2048 x 16384: 187 us by tile columns,
// 168 by tile rows.)
// ... unless the busiest XCD then needs one more round of tiles than in the other order (13056 x 2560 x 2048 in 256 x 256
// tiles: 510 tiles are 64 per XCD by tile columns, two rounds on 32 CUs, but 65 on some XCDs by tile rows: 93 against 75 us).
inline bool big_takes_rows(int M, int N, int K, int m_tiles, int n_tiles, int slots, double* bytes, int* busiest) {
    const double a_bytes = (double)M * K, b_bytes = (double)N * K;
    const int band_c = 4, band_r = 4;
    const double by_cols = a_bytes * (n_tiles < 8 ? n_tiles : 8) + b_bytes * big_ceil_div(m_tiles, band_c);
    const double by_rows = b_bytes * (m_tiles < 8 ? m_tiles : 8) + a_bytes * big_ceil_div(n_tiles, band_r);
    bool rows = by_rows < 0.8 * by_cols;
    const int most_c = big_max_tiles_per_xcd(m_tiles, n_tiles, 4), most_r = big_max_tiles_per_xcd(n_tiles, m_tiles, 4);
    const int rounds_c = big_ceil_div(most_c, slots), rounds_r = big_ceil_div(most_r, slots);
    if (rounds_c != rounds_r) rows = rounds_r < rounds_c;
    *bytes = rows ? by_rows : by_cols;
    *busiest = rows ? most_r : most_c;
    return rows;
}


// Tile rows per band: 4; a grid of up to 8 tile rows whose activation rows still fit an XCD's L2 beside the weight stream is
// one band, so that the weights come from HBM once.
inline int big_band(int by_rows, int m_tiles, int tile_rows, int K) {
    int band = 4;
    if (!by_rows && m_tiles <= 8 && (int64_t)m_tiles * tile_rows * (K < 4096 ? K : 4096) <= (5 << 19)) band = m_tiles;
    if (const char* e = tuning_env("PHYAI_FP8_BAND")) { const int b = atoi(e); if (b >= 1 && b <= 16) band = b; }
    return band;
}

}  // namespace phyai
