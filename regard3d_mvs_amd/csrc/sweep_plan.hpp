// Launch shape of the row sweeps (k_sweep, kernels_sgm.hip): host arithmetic
// only, so that it can be checked without a device.
#pragma once

#include <algorithm>
#include <cstdint>

namespace r3dg {

constexpr int kSweepThreads = 1024;  // a block's threads: the columns and the chunks of a row it takes at once
constexpr int kSweepRowPad = 8;      // words after an LDS row that a window may read

// Launch shape for tiles of at most max_w columns and max_chunks chunks a row:
// words of an LDS row, words of a scratch row (0: none needed), the blocks
// that run at once, the chunks a thread holds.  ok is false where the kernel
// does not apply.
struct SweepPlan {
  bool ok;
  int wpad, cap, swords, lds_bytes, blocks, held;
};

// The same on a device of `cus` compute units with `lds` bytes of LDS a block.
// mean_chunks: of the rows of the tile with most.  A row of k chunks takes
// words 0 .. 8 k + max_w + 1 (8 per chunk, a sentinel before each pixel and
// after the last): a scratch row holds all of them, however many (rows of 1024
// columns have at most 1024 x 250 chunks).
//
// Two chunks held per thread, where three paths leave no registers for more or
// no tile's mean row has more chunks than threads (rows past twice that are
// rare there, and the sweep of one path is 3 % faster than with four: 2.94 ms
// against 3.02 for the 1080p pair's aggregation); four for wider rows (the 24 MP
// pair's: 17.5 ms against 17.7 with two).
inline SweepPlan size_sweep(int np, int max_w, std::uint32_t max_chunks, std::uint64_t mean_chunks, int cus, int lds) {
  SweepPlan p{};
  const std::uint64_t need = 8 * std::uint64_t(max_chunks) + std::uint64_t(std::max(max_w, 0)) + 2;
  if (max_w > kSweepThreads || need > (std::uint64_t{1} << 30)) return p;
  const int fixed = 4 * (6 * max_w + 2 * np * max_w + 128 + 4);
  p.held = np == 3 || mean_chunks <= kSweepThreads ? 2 : 4;
  p.wpad = max_w;
  const int room = (lds - fixed) / (4 * np) - kSweepRowPad;
  if (room < 1024) return p;
  // At least 16 words: a window that is not used reads the row's first ten.
  p.cap = std::min({room, 8 * kSweepThreads * p.held, std::max(static_cast<int>(need), 16)});
  p.lds_bytes = fixed + 4 * np * (p.cap + kSweepRowPad);
  p.swords = std::uint64_t(p.cap) >= need ? 0 : static_cast<int>(need) + 16;
  p.blocks = std::max(cus, 1);
  p.ok = true;
  return p;
}

// Whether sweeps take the `tiles` tiles with label ranges of a level, of `cells`
// cells in all, where a range of tiles may hold `cap` cells (`scan_cap` of path
// scans); path scans otherwise.  A sweep is one block's chain of rows, six a
// tile, as long with few tiles as with many: with 12 (one tile and its mirror)
// path scans are over sooner (384x288 with a half-size level 0.97 and 0.93 ms,
// 480x270 1.02 and 0.96), with 48 sweeps (960x540 1.37 and 1.52 ms; 800x600 1.29 and
// 1.26).  The line is at a sixteenth of the compute units, at an eighth where a
// path's slices are uint16 (P2 past a byte; 640x480, 24 sweeps: 1.86 and 1.60 ms).
//
// Where the level is cut into ranges, each waits for its slowest tile.  Path
// scans hold five times the cells in the same memory; where they are cut into
// fewer ranges, sweeps have to have four blocks a compute unit in each of theirs
// (aggregation of 24 MP in 10 GiB, 32 tiles a range: 52 ms by sweeps and 37 by path
// scans, of 1080p in 1.2 GiB, 8 tiles a range: 12.5 and 7.4; the 24 MP pair in 30
// GiB, 96 tiles a range: 33.7 and 34).  Where both are cut alike, at the most
// cells a range may have, a quarter is enough (24 MP with 400 labels a pixel, 48
// tiles a range: 149 and 174 ms; 3 MP with 900, 12 tiles a range: 51 and 53).
inline bool sweeps_fit(std::uint64_t tiles, std::uint64_t cells, std::uint64_t cap, std::uint64_t scan_cap, bool bytes,
                       int cus) {
  const auto cut = [&](std::uint64_t most) { return cells / std::max<std::uint64_t>(most, 1) + 1; };
  const std::uint64_t ranges = cut(cap), units = 6 * tiles / ranges;
  const auto n = std::uint64_t(std::max(cus, 0));
  if (ranges == 1) return (bytes ? 16 : 8) * units >= n;
  return ranges > cut(scan_cap) ? units >= 4 * n : 4 * units >= n;
}

}  // namespace r3dg
