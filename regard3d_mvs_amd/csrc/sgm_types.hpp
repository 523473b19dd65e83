// Descriptors shared by the host driver and the gfx950 kernels.
//
// A *job* is one matching direction of one pyramid level of one pair: a base
// image matched against a partner image (the left-to-right match, or the
// right-to-left match on the mirrored pair, stereo_matcher.cpp:842-863).  A
// *tile* is one of the job's overlapping tiles (stereo_matcher.cpp:613-653);
// aggregation restarts at tile borders, so tiles are independent work units
// and one launch can cover the tiles of many jobs (both directions of a level,
// or every pair of a batch).
//
// HBM layout of the costs C (uint8), of the paths' planes (uint8) and of the
// aggregated costs S (uint16): every tile owns a contiguous volume at
// cell_base, its rows one after the other, a row's pixels in order; a pixel's
// labels follow each other (the TileLabels ranges of stereo_matcher.cpp:172-224).
// rowbase[row_base + y * strips + s] is the first cell of strip s of row y, the
// pixel record pix[px_base + y*w + x] holds the offset from there (tiles of at
// most 2^16 columns, nearly all, have one strip a row).  Label counts are
// multiples of 16, so every pixel's labels are whole chunks of 16 cells.
//
// Pixel record (uint64): bits 0-23 chunk offset inside the strip, bits
// 24-31 label count / 16, bits 32-47 first label `lo`, bits 48-63 intensity.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace r3dg {

constexpr int kLabelAlign = 16;
constexpr int kMaxLabels = 4000;           // per pixel and level: a record keeps label count / 16 in 8 bits
// A tile row is counted in strips of 2^16 columns: a record keeps a chunk offset
// inside its strip in 24 bits, a map entry a column in 16.
constexpr int kStripShift = 16;
static_assert((std::uint64_t{kMaxLabels / kLabelAlign} << kStripShift) < (1U << 24));
__host__ __device__ constexpr int strips_of(int columns) { return (columns + (1 << kStripShift) - 1) >> kStripShift; }
constexpr int kPaths = 8;
constexpr int kMaxByteP2 = 255;  // largest P2 with which a path's M = L - C is a byte

__host__ __device__ constexpr std::uint64_t pix_record(std::uint64_t off, int lo, int num, int val) {
  return ((off / kLabelAlign) & 0xFFFFFFU) | (std::uint64_t((num / kLabelAlign) & 0xFF) << 24) |
         (std::uint64_t(std::uint16_t(lo)) << 32) | (std::uint64_t(std::uint16_t(val)) << 48);
}
__host__ __device__ constexpr std::uint32_t pix_off(std::uint64_t r) { return std::uint32_t(r & 0xFFFFFFU) * kLabelAlign; }
__host__ __device__ constexpr int pix_num(std::uint64_t r) { return int((r >> 24) & 0xFFU) * kLabelAlign; }
__host__ __device__ constexpr int pix_lo(std::uint64_t r) { return int((r >> 32) & 0xFFFFU); }
__host__ __device__ constexpr int pix_val(std::uint64_t r) { return int(r >> 48); }
// Chunk map entry: the chunk's column in its strip and its place in the pixel.
__host__ __device__ constexpr std::uint32_t map_entry(int col, int place) {
  return std::uint32_t(col) | std::uint32_t(place) << kStripShift;
}
__host__ __device__ constexpr int map_col(std::uint32_t m) { return int(m & ((1U << kStripShift) - 1)); }
__host__ __device__ constexpr int map_place(std::uint32_t m) { return int(m >> kStripShift); }
constexpr int kMaxLevels = 13;

struct JobDesc {
  const std::uint16_t* img;  // base image (P2 intensities), width x height
  const std::uint64_t* cl;   // base Census
  const std::uint64_t* cr;   // partner Census, pwidth x height
  const std::int32_t* rows4; // [height][4] valid columns of the row: base first, last; partner first, last
  const std::uint16_t* lo;   // per-pixel label ranges (nullptr: full range)
  const std::uint16_t* num;
  std::int64_t img_stride;   // elements
  std::int64_t cl_stride;
  std::int64_t cr_stride;
  std::int64_t r_stride;
  std::int32_t width;
  std::int32_t height;
  std::int32_t pwidth;
  std::int32_t dmin;
  std::int32_t D;            // aligned label count of the level
  std::int32_t p1;
  std::int32_t invalid_cost;
  std::int32_t confidence;   // select writes confidence
  // 1: a mirrored job whose img, cl and cr are those of the unmirrored
  // images: base column X reads img[width - 1 - X] and cl[width - 1 - X],
  // partner column c reads cr[pwidth - 1 - c].  The Census of a mirrored
  // image is that of the image read backwards with its bits permuted
  // (neighbour (dy, dx) <-> (dy, -dx)), and a permutation applied to both
  // sides leaves Hamming distances unchanged.
  std::int32_t mirrored;
  std::uint16_t lut[256];    // P2 by 8-bit intensity step (stereo_matcher.cpp:69-79)
};

struct TileDesc {
  std::int32_t x0, y0, w, h;  // in the job's base image
  std::int32_t job;
  std::int32_t max_num;       // largest label count of the tile
  std::uint64_t cell_base;    // first cell of the tile in S
  std::uint64_t px_base;      // first tile pixel in per-pixel arrays
  std::uint64_t row_base;     // first strip of the first row in per-strip arrays
  std::uint32_t cells;        // cells of the tile
  std::int32_t strips;        // per row
};

// Tile grid of one job for blending (stereo_matcher.cpp:688-766): tile (i, j)
// of the grid is tile tile_base + j * nx + i; cols[i] / rows[j] hold the tile
// extent [x0, x1) and its core [c0, c1).
struct GridDesc {
  const std::int32_t* cols;  // [nx][4]
  const std::int32_t* rows;  // [ny][4]
  std::int32_t nx, ny;
  std::int32_t width, height;
  std::int32_t blend;
  std::int32_t tile_base;
};

struct SelectParams {
  std::int32_t subpixel;     // r3dg_subpixel
  float uniqueness;
  std::int32_t lr_max_diff;
  std::int32_t diagonal_lr;  // check against the right WTA of the same volume
};

}  // namespace r3dg
