// gfx950 kernels of the SGM core: tile label layout, matching costs, the 8
// path scans, winner-takes-all selection and tile blending.
//
// Aggregation dataflow (no MFMA: nothing here is a contraction).  k_cost
// writes the matching cost of every tile cell once per level as one byte
// (popcount of the Census XOR, or invalid_cost).  Three kernels aggregate it:
//   k_full   tiles without label ranges: all eight paths in one launch, path
//            costs in registers, a byte plane M = L - C per path;
//   k_sweep  tiles with label ranges: the vertical and diagonal paths, a block
//            per tile and direction sweeping row by row, lanes packed with
//            16-label chunks, up to three paths at once;
//   k_path   one path direction over every tile by waves of 8 scanlines: the
//            horizontal paths beside the sweeps, and all eight where the
//            memory left, the tiles' width, labels or P2 rule the others out
//            or sweeps would be too few to fill the device.
// Each writes uint16 slices of S (uint16 wrap-around, so the order of the
// paths does not matter) or byte planes; the selection sums them.
//
// Recurrence (sgm_kernels.cpp:176-228, 387-403; stereo_matcher.cpp:1280-1362):
//   L(p,d) = C(p,d) + min(L(q,d), sat16(min(L(q,d-1), L(q,d+1)) + P1),
//                         sat16(min_q + P2(p,q))) - min_q            (mod 2^16)
// with L = C at the first pixel of a path inside the tile.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>
#include <utility>

#include "kernels.hpp"

namespace r3dg {
namespace {

constexpr float kInf = __builtin_huge_valf();

__device__ __forceinline__ int find_tile(const std::uint64_t* __restrict__ prefix, int ntiles, std::uint64_t id) {
  int lo = 0, hi = ntiles - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (prefix[mid] <= id) {
      lo = mid;
    } else {
      hi = mid - 1;
    }
  }
  return lo;
}

// The same search by a whole wave (every lane active, the same id in every
// lane): each round samples 64 evenly spaced prefixes and keeps the interval
// between the last sample <= id and the next, so 4096 tiles take two rounds
// of loads instead of twelve.
__device__ __forceinline__ int find_tile_wave(const std::uint64_t* __restrict__ prefix, int ntiles, std::uint64_t id) {
  const int lane = static_cast<int>(__lane_id());
  int lo = 0, span = ntiles;  // prefix[lo] <= id; the tile lies in [lo, lo + span)
  while (span > 1) {
    const int step = (span + 63) >> 6;
    const int i = lane * step;
    const bool le = i < span && prefix[lo + i] <= id;
    const int c = __popcll(__ballot(le));
    lo += (c - 1) * step;
    span = min(step, span - (c - 1) * step);
  }
  return lo;
}

// Pointers read out of JobDesc / TileDesc are generic to the compiler; these
// views make their loads and stores global_* instructions (flat ones also count
// against the LDS wait counter, which would serialise the prefetch below).
template <typename T>
__device__ __forceinline__ const __attribute__((address_space(1))) T* gptr(const T* p) {
  return (const __attribute__((address_space(1))) T*)(p);
}
template <typename T>
__device__ __forceinline__ __attribute__((address_space(1))) T* gptr_mut(T* p) {
  return (__attribute__((address_space(1))) T*)(p);
}

// Descriptors that no kernel writes, read through the scalar cache where the
// address is the same in every lane.
template <typename T>
__device__ __forceinline__ const __attribute__((address_space(4))) T* cptr(const T* p) {
  return (const __attribute__((address_space(4))) T*)(p);
}

__device__ __forceinline__ void label_range(const JobDesc& J, int X, int Y, int& lo, int& num) {
  if (J.lo != nullptr) {
    lo = J.lo[Y * J.r_stride + X];
    num = J.num[Y * J.r_stride + X];
  } else {
    lo = 0;
    num = J.D;
  }
}

// ------------------------------------------------------------------ layout
// Inclusive scan of v over a block of W waves: shuffles inside each wave, the
// wave totals through LDS (wsum[W]).  Returns this thread's inclusive prefix
// and the block total; every thread of the block must call it.
template <int W, typename U>
__device__ __forceinline__ U block_scan_incl(U v, U* wsum, U& total) {
  const int lane = static_cast<int>(threadIdx.x & 63), wave = static_cast<int>(threadIdx.x >> 6);
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const U t = __shfl_up(v, d);
    if (lane >= d) v += t;
  }
  if (lane == 63) wsum[wave] = v;
  __syncthreads();
  U off = 0, all = 0;
#pragma unroll
  for (int k = 0; k < W; ++k) {
    off += k < wave ? wsum[k] : U(0);
    all += wsum[k];
  }
  total = all;
  __syncthreads();  // wsum is reused by the next call
  return v + off;
}

// Inclusive scan of v over the 64 lanes of a wave.
__device__ __forceinline__ std::uint32_t wave_scan_incl(std::uint32_t v) {
  const int lane = static_cast<int>(threadIdx.x & 63);
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const std::uint32_t t = __shfl_up(v, static_cast<unsigned>(d));
    if (lane >= d) v += t;
  }
  return v;
}

// Exclusive scan of the label counts of one tile row into the pixel records:
// chunk offset inside the row, chunks, lo, intensity.  One wave per row (4
// rows per block), 64 x kItems pixels per pass, the pass's label ranges and
// intensities loaded before its scans; no block barriers, so a row waits only
// on its own loads.
__global__ __launch_bounds__(256) void k_tile_row_scan(const JobDesc* __restrict__ jobs,
                                                       const TileDesc* __restrict__ tiles,
                                                       const std::uint64_t* __restrict__ row_prefix, int ntiles,
                                                       std::uint64_t total_rows,
                                                       std::uint64_t* __restrict__ pix,
                                                       std::uint64_t* __restrict__ row_cells,
                                                       std::uint32_t* __restrict__ row_max) {
  constexpr int kItems = 8;
  const int lane = static_cast<int>(threadIdx.x & 63);
  const std::uint64_t r = std::uint64_t(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (r >= total_rows) return;  // whole waves
  const int t = find_tile_wave(row_prefix, ntiles, r);
  const TileDesc T = tiles[t];
  const JobDesc& J = jobs[T.job];
  const int y = static_cast<int>(r - row_prefix[t]);
  const int Y = T.y0 + y;
  const auto jlo = gptr(J.lo), jnum = gptr(J.num);
  const std::int64_t rbase = std::int64_t(Y) * J.r_stride + T.x0;
  const auto img = gptr(J.img) + std::int64_t(Y) * J.img_stride;
  // Base columns of a mirrored job read the unmirrored image backwards.
  const int img_x0 = J.mirrored != 0 ? J.width - 1 - T.x0 : T.x0, img_dx = J.mirrored != 0 ? -1 : 1;
  std::uint64_t* prow = pix + T.px_base + std::uint64_t(y) * T.w;
  constexpr int kStrip = 1 << kStripShift;
  static_assert(kStrip % (64 * kItems) == 0, "strips end where a pass does");
  std::uint64_t strip = T.row_base + static_cast<std::uint32_t>(y * T.strips);
#pragma unroll 1
  for (int xs = 0; xs < T.w; xs += kStrip, ++strip) {
    const int xe = min(T.w, xs + kStrip);
    std::uint64_t carry = 0;
    std::uint32_t vmax = 0;
    for (int base = xs; base < xe; base += 64 * kItems) {
      int lo[kItems], num[kItems], val[kItems];
#pragma unroll
      for (int k = 0; k < kItems; ++k) {
        const int x = base + 64 * k + lane;
        lo[k] = 0;
        num[k] = 0;
        val[k] = 0;
        if (x < T.w) {
          val[k] = img[img_x0 + img_dx * x];
          if (jlo != nullptr) {
            lo[k] = jlo[rbase + x];
            num[k] = jnum[rbase + x];
          } else {
            num[k] = J.D;
          }
        }
      }
#pragma unroll
      for (int k = 0; k < kItems; ++k) {
        const int x = base + 64 * k + lane;
        const std::uint32_t v = static_cast<std::uint32_t>(num[k]);
        const std::uint32_t incl = wave_scan_incl(v);
        if (x < T.w) prow[x] = pix_record(carry + incl - v, lo[k], num[k], val[k]);
        carry += static_cast<std::uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(incl), 63));
        vmax = max(vmax, v);
      }
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) vmax = max(vmax, static_cast<std::uint32_t>(__shfl_xor(vmax, d)));
    if (lane == 0) {
      row_cells[strip] = carry;
      row_max[strip] = vmax;
    }
  }
}

// Totals of one tile (cells, largest label count, most chunks in a strip) and
// the first cell of each of its strips: an exclusive scan of their counts.
constexpr int kCellsThreads = 1024;  // k_tile_cells: one block of 16 waves per tile
__global__ __launch_bounds__(kCellsThreads) void k_tile_cells(const TileDesc* __restrict__ tiles,
                                                    const std::uint64_t* __restrict__ row_cells,
                                                    const std::uint32_t* __restrict__ row_max,
                                                    std::uint32_t* __restrict__ rowbase,
                                                    std::uint64_t* __restrict__ tile_cells,
                                                    std::uint32_t* __restrict__ tile_max,
                                                    std::uint32_t* __restrict__ tile_row) {
  const TileDesc T = tiles[blockIdx.x];
  __shared__ std::uint64_t wsum[kCellsThreads / 64];
  __shared__ std::uint32_t smax, srow;
  if (threadIdx.x == 0) {
    smax = 0;
    srow = 0;
  }
  __syncthreads();
  std::uint64_t carry = 0;
  const int strips = T.h * T.strips;
  for (int base = 0; base < strips; base += kCellsThreads) {
    const int y = base + static_cast<int>(threadIdx.x);
    std::uint64_t v = 0;
    if (y < strips) {
      v = row_cells[T.row_base + y];
      atomicMax(&smax, row_max[T.row_base + y]);
      atomicMax(&srow, static_cast<std::uint32_t>(min(v / kLabelAlign, std::uint64_t{0xFFFFFFFFU})));
    }
    std::uint64_t total;
    const std::uint64_t before = carry + block_scan_incl<kCellsThreads / 64>(v, wsum, total) - v;
    if (y < strips) rowbase[T.row_base + y] = static_cast<std::uint32_t>(before);
    carry += total;
  }
  if (threadIdx.x == 0) {
    tile_cells[blockIdx.x] = carry;
    tile_max[blockIdx.x] = smax;
    tile_row[blockIdx.x] = srow;
  }
}

// ------------------------------------------------------------------ paths
// Path directions (dx, dy): the predecessor of p is p - (dx, dy).
//   0 (1,0)  1 (-1,0)  2 (0,1)  3 (0,-1)  4 (1,1)  5 (-1,-1)  6 (-1,1)  7 (1,-1)
// Scanlines of a w x h tile: rows (dy == 0), columns (dx == 0), diagonals
// x - y = s - (h - 1) (dx == dy) or anti-diagonals x + y = s (dx == -dy).
template <int DX, int DY>
__device__ __forceinline__ int scanlines(int w, int h) {
  return DY == 0 ? h : (DX == 0 ? w : w + h - 1);
}

template <int DX, int DY>
__device__ __forceinline__ void scan_start(int s, int w, int h, int& x, int& y, int& len) {
  if (DY == 0) {
    y = s;
    x = DX > 0 ? 0 : w - 1;
    len = w;
  } else if (DX == 0) {
    x = s;
    y = DY > 0 ? 0 : h - 1;
    len = h;
  } else if (DX == DY) {
    const int c = s - (h - 1);
    const int x0 = c >= 0 ? c : 0, y0 = c >= 0 ? 0 : -c;
    len = min(w - x0, h - y0);
    x = DX > 0 ? x0 : x0 + len - 1;
    y = DX > 0 ? y0 : y0 + len - 1;
  } else {
    const int x0 = min(s, w - 1), y0 = s - x0;  // end on the top / right border
    len = min(x0 + 1, h - y0);
    x = DX < 0 ? x0 : x0 - (len - 1);
    y = DX < 0 ? y0 : y0 + (len - 1);
  }
}

// ------------------------------------------------------------------ costs
// Matching costs of every tile cell (stereo_matcher.cpp:233-247, census_costs):
// the Hamming distance of the base Census and the partner Census at column
// X - dmin - lo - j when that column lies in the partner row's valid interval,
// invalid_cost when it does not, 0 for base pixels outside the base row's
// valid interval.  One block per tile row; a thread per 16-label chunk writes
// 16 bytes.  Rows of at most kPx pixels stage everything a chunk reads in
// LDS (pixel cell offsets and lo, base Census, a chunk-to-pixel map, the
// partner Census window), so the chunk loop touches
// global memory only to store; wider rows search their pixel records in
// global memory.
constexpr int kCostThreads = 256;
__global__ __launch_bounds__(kCostThreads) void k_cost(const JobDesc* __restrict__ jobs, const TileDesc* __restrict__ tiles,
                                              const std::uint64_t* __restrict__ row_prefix, int ntiles,
                                              const std::uint32_t* __restrict__ rowbase,
                                              const std::uint64_t* __restrict__ pix, std::uint8_t* __restrict__ C,
                                              std::uint32_t* __restrict__ cmap) {
  // Sized for the tiles of the default options (at most 600 columns, 512
  // labels): 24 KB of LDS, six blocks per CU.
  constexpr int kPx = 640;          // row pixels staged in LDS
  constexpr int kMap = 2048;        // chunks mapped to their pixel
  constexpr int kWin = 1280;        // partner Census columns staged
  __shared__ std::uint32_t soff[kPx];
  __shared__ std::uint16_t slo[kPx];
  __shared__ std::uint64_t scl[kPx];
  __shared__ std::uint16_t smap[kMap];
  __shared__ std::uint64_t swin[kWin];
  const std::uint64_t r = blockIdx.x;
  const int t = find_tile_wave(row_prefix, ntiles, r);
  const TileDesc T = tiles[t];
  const JobDesc& J = jobs[T.job];
  const int y = static_cast<int>(r - row_prefix[t]);
  const int Y = T.y0 + y;
  const auto rec = gptr(pix + T.px_base + std::uint64_t(y) * T.w);
  const auto rows = gptr(J.rows4) + 4 * Y;
  const auto cl = gptr(J.cl) + std::size_t(Y) * J.cl_stride;
  const auto cr = gptr(J.cr) + std::size_t(Y) * J.cr_stride;
  const int pw1 = J.pwidth - 1;
  const bool mir = J.mirrored != 0;
  auto bcol = [&](int X) { return mir ? J.width - 1 - X : X; };  // column of cl
  auto pcol = [&](int c) { return mir ? pw1 - c : c; };         // column of cr
  // Partner columns a cost of this row can use: X - dmin - label for X in the
  // tile and label in [0, D); every valid column lies in [c0, c1].
  const int c0 = max(0, T.x0 - J.dmin - (J.D - 1)), c1 = min(pw1, T.x0 + T.w - 1 - J.dmin);
  const bool windowed = c1 >= c0 && c1 - c0 < kWin;
  const bool staged = T.w <= kPx;
  constexpr int kStrip = 1 << kStripShift;
  const std::uint64_t last = rec[min(T.w, kStrip) - 1];  // of the first strip: the only one where staged
  // Staging: every global load of a thread is issued before the first LDS
  // store, so that the block waits for one memory latency, not one per
  // element (the launch has kCostThreads threads).
  constexpr int kWinIt = (kWin + kCostThreads - 1) / kCostThreads;
  constexpr int kPxIt = (kPx + kCostThreads - 1) / kCostThreads;
  const int tid = static_cast<int>(threadIdx.x);
  std::uint64_t wv[kWinIt], pv[kPxIt], cv[kPxIt];
#pragma unroll
  for (int i = 0; i < kWinIt; ++i) {
    const int k = tid + kCostThreads * i;
    wv[i] = windowed && k <= c1 - c0 ? cr[pcol(c0 + k)] : 0;
  }
  if (staged) {
#pragma unroll
    for (int i = 0; i < kPxIt; ++i) {
      const int x = tid + kCostThreads * i;
      pv[i] = x < T.w ? rec[x] : 0;
      cv[i] = x < T.w ? cl[bcol(T.x0 + x)] : 0;
    }
  }
#pragma unroll
  for (int i = 0; i < kWinIt; ++i) {
    const int k = tid + kCostThreads * i;
    if (windowed && k <= c1 - c0) swin[k] = wv[i];
  }
  if (staged) {
#pragma unroll
    for (int i = 0; i < kPxIt; ++i) {
      const int x = tid + kCostThreads * i;
      if (x < T.w) {
        const std::uint64_t pr = pv[i];
        const std::uint32_t off = pix_off(pr);
        soff[x] = off;
        slo[x] = static_cast<std::uint16_t>(pix_lo(pr));
        scl[x] = cv[i];
        const std::uint32_t e =
            min((off + static_cast<std::uint32_t>(pix_num(pr))) >> 4, static_cast<std::uint32_t>(kMap));
        for (std::uint32_t k = off >> 4; k < e; ++k) smap[k] = static_cast<std::uint16_t>(x);
      }
    }
  }
  __syncthreads();
  auto chunks_to = [](std::uint64_t r) { return (pix_off(r) + static_cast<std::uint32_t>(pix_num(r))) >> 4; };
  const int bfirst = rows[0], blast = rows[1], pfirst = rows[2], plast = rows[3];
  const std::uint32_t invalid = static_cast<std::uint32_t>(J.invalid_cost);
  const std::uint32_t* strip_base = rowbase + T.row_base + static_cast<std::uint32_t>(y * T.strips);
  const bool costs = C != nullptr, map = cmap != nullptr;
  // Output of the strip in hand.
  std::uint64_t strip_cell = T.cell_base + strip_base[0];
  std::uint8_t* out = C + strip_cell;
  std::uint32_t* mout = cmap + strip_cell / kLabelAlign;
  auto partner = [&](int xr) {
    return windowed ? swin[min(max(xr, c0), c1) - c0] : cr[pcol(min(max(xr, 0), pw1))];
  };
  // Costs of the strip's chunk k, of pixel xa (first cell off, first label lo, Census c).
  auto chunk = [&](std::uint32_t k, int xa, std::uint32_t off, int lo, std::uint64_t c) {
    const int X = T.x0 + xa;
    const int jb = static_cast<int>(16 * k - off);
    const int xr0 = X - J.dmin - lo - jb;
    const bool lvalid = X >= bfirst && X <= blast;
    std::uint32_t w[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      std::uint32_t v = 0;
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const int xr = xr0 - 4 * q - b;
        std::uint32_t cost = xr >= pfirst && xr <= plast ? static_cast<std::uint32_t>(__popcll(c ^ partner(xr)))
                                                         : invalid;
        cost = lvalid ? cost : 0U;
        v |= cost << (8 * b);
      }
      w[q] = v;
    }
    if (costs) *reinterpret_cast<uint4*>(out + 16 * std::size_t(k)) = make_uint4(w[0], w[1], w[2], w[3]);
    if (map) mout[k] = map_entry(xa & (kStrip - 1), jb / kLabelAlign);
  };
  if (staged) {
    const std::uint32_t chunks = chunks_to(last);
    const bool mapped = chunks <= static_cast<std::uint32_t>(kMap);
    for (std::uint32_t k = threadIdx.x; k < chunks; k += blockDim.x) {
      int xa;
      if (mapped) {
        xa = smap[k];
      } else {
        // Every pixel holds at least one chunk, so the pixel of chunk k is at most k.
        xa = 0;
        int xb = min(static_cast<int>(k), T.w - 1);
        while (xa < xb) {
          const int mid = (xa + xb + 1) >> 1;
          if (soff[mid] <= 16 * k) {
            xa = mid;
          } else {
            xb = mid - 1;
          }
        }
      }
      chunk(k, xa, soff[xa], slo[xa], scl[xa]);
    }
  } else {
    for (int xs = 0; xs < T.w; xs += kStrip) {
      const int xn = min(T.w - xs, kStrip);
      if (xs > 0) {
        strip_cell = T.cell_base + strip_base[xs >> kStripShift];
        out = C + strip_cell;
        mout = cmap + strip_cell / kLabelAlign;
      }
      const std::uint32_t chunks = chunks_to(xs > 0 ? rec[xs + xn - 1] : last);
      for (std::uint32_t k = threadIdx.x; k < chunks; k += blockDim.x) {
        int xa = xs, xb = xs + min(static_cast<int>(k), xn - 1);
        while (xa < xb) {
          const int mid = (xa + xb + 1) >> 1;
          if (pix_off(rec[mid]) <= 16 * k) {
            xa = mid;
          } else {
            xb = mid - 1;
          }
        }
        const std::uint64_t pr = rec[xa];
        chunk(k, xa, pix_off(pr), pix_lo(pr), cl[bcol(T.x0 + xa)]);
      }
    }
  }
}

// ------------------------------------------------------------------ path scans
// Packed pairs of uint16 path costs: v_pk_* instructions process two labels.
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ u16x2 as_pair(std::uint32_t v) { return __builtin_bit_cast(u16x2, v); }
__device__ __forceinline__ std::uint32_t as_u32(u16x2 v) { return __builtin_bit_cast(std::uint32_t, v); }

// Min over the 8 lanes of a scanline (quad swaps, then the half-row mirror).
__device__ __forceinline__ std::uint32_t min8(std::uint32_t v) {
  v = min(v, static_cast<std::uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0xB1, 0xF, 0xF, false)));
  v = min(v, static_cast<std::uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x4E, 0xF, 0xF, false)));
  v = min(v, static_cast<std::uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x141, 0xF, 0xF, false)));
  return v;
}

typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// Loads and stores at a byte offset from a wave-uniform base (SGPR base +
// 32-bit VGPR offset addressing).
template <typename T>
__device__ __forceinline__ T ldb(const void* base, std::uint32_t off) {
  const auto p = (const __attribute__((address_space(1))) char*)(base);
  return *reinterpret_cast<const __attribute__((address_space(1))) T*>(p + off);
}
template <typename T>
__device__ __forceinline__ void stb(void* base, std::uint32_t off, T v) {
  const auto p = (__attribute__((address_space(1))) char*)(base);
  *reinterpret_cast<__attribute__((address_space(1))) T*>(p + off) = v;
}

// The same past the caches, for what is written whole and read only once the
// launch is over: the volumes of k_full and k_sweep then leave the costs they
// read in the memory-side cache (aggregation of 1024x768 with 128 labels 0.83 to
// 0.76 ms, of the 1080p pair 2.93 to 2.81).  Not for scans along rows, whose
// lines fill 16 bytes at a time.
template <typename T>
__device__ __forceinline__ void stb_nt(void* base, std::uint32_t off, T v) {
  const auto p = (__attribute__((address_space(1))) char*)(base);
  __builtin_nontemporal_store(v, reinterpret_cast<__attribute__((address_space(1))) T*>(p + off));
}

// s_waitcnt immediate (gfx9 encoding) that waits for every vector memory
// operation and nothing else: vmcnt 0, expcnt 7, lgkmcnt 15.
constexpr int kVmcnt0 = 0x0F70;
constexpr int kWaves = 4;                     // waves per block
constexpr int kDist = 3;                      // steps between a segment prefetch and its use
constexpr int kNarrow = 368;                  // labels whose path costs stay in LDS
constexpr int kPad = 12;                      // sentinel slots before label 0 and after the last label
constexpr int kRow = kPad + kNarrow + kPad;   // uint16 slots of an LDS row

// Label segments of a pixel: segment 0 holds labels [0, 32), lane l holds
// four of them from 4l; segment s >= 1 holds [32 + 64 (s - 1), 32 + 64 s),
// lane l eight of them from 32 + 64 (s - 1) + 8l.  A lane's labels lie all
// inside or all outside a pixel's range (label counts are multiples of 16).
template <int P>
__device__ __forceinline__ int seg_first(int s, int l8) {
  return P == 4 ? 4 * l8 : 32 + 64 * (s - 1) + 8 * l8;
}
__device__ __forceinline__ int segments(int num) { return num <= 32 ? 1 : 1 + (num - 32 + 63) / 64; }

// Costs (P bytes) and S (P uint16) of one lane in one segment.
template <int P>
struct SegIn {
  std::uint32_t c[P / 4];
  std::uint32_t s[P / 2];
};

// Per-step values of one scanline pixel, read from the wave's step ring:
// the pixel's first cell in the tile volume and a packed word holding its
// first label (bits 0-15), the P2 table index |I - I_prev| >> 8 of the step
// (bits 16-23) and its label count / 16 (bits 24-31); p2 is the table
// entry itself, read kDist steps before the step.
struct StepIn {
  std::uint32_t cell;
  std::uint32_t meta;
  std::uint32_t p2;
};
static_assert(kMaxLabels / kLabelAlign <= 255, "label count / 16 must fit 8 bits");
__device__ __forceinline__ int step_lo(const StepIn& u) { return static_cast<int>(u.meta & 0xFFFFU); }
__device__ __forceinline__ std::uint32_t step_p2_index(const StepIn& u) { return (u.meta >> 16) & 0xFFU; }
__device__ __forceinline__ int step_num(const StepIn& u) { return static_cast<int>(u.meta >> 24) * kLabelAlign; }
// Pixel record and row offset of step 8 b + l of a scanline, held by lane l of
// its group: the loads of 8 steps are one batch.
struct StepBatch {
  std::uint64_t rec;
  std::uint32_t rs;
};
// Segments 0 and 1 of a pixel, loaded one step ahead.
struct StepSegs {
  SegIn<4> a;
  SegIn<8> b;
};

// One path direction over every tile.  A wave scans 8 adjacent scanlines of a
// tile, 8 lanes per scanline, a lane holding 4 or 8 consecutive labels of a
// segment as packed uint16 pairs.  Recursion (stereo_matcher.cpp:258-330):
//   L(j) = C(j) + min(Lp(k), sat(min(Lp(k-1), Lp(k+1)) + P1), sat(mp + P2)) - mp
// with k = j + lo - lo_prev, mp the predecessor's minimum, Lp = 0xFFFF outside
// its labels and L = C at the first pixel.  The predecessor's path costs sit
// in a row with 0xFFFF sentinels around its labels, in LDS for pixels of at
// most kNarrow labels and in a global scratch row for wider ones; a lane reads
// its window of P + 2 values as aligned words (the window clamped into the
// sentinels) and shifts them into place.  Segments 0 and 1 use data prefetched
// kDist steps ahead; segments from 2 on (pixels of more than 96 labels) are
// loaded in the step, one segment ahead.  The pixel records and row offsets
// of a scanline are loaded 8 steps at a time (lane l of the group loads step
// 8 b + l) and unpacked into an 8-slot ring in LDS, read one step before the
// segment prefetch that needs them.
template <int DX, int DY, int MODE>
__global__ __launch_bounds__(64 * kWaves) void k_path(
    const JobDesc* __restrict__ jobs, const TileDesc* __restrict__ tiles, const std::uint64_t* __restrict__ gprefix,
    int ntiles, std::uint64_t groups, const std::uint32_t* __restrict__ rowbase,
    const std::uint64_t* __restrict__ pix, const std::uint8_t* __restrict__ C, void* __restrict__ out_volume,
    std::uint16_t* __restrict__ scratch, int scratch_row, std::uint32_t* __restrict__ queue) {
  constexpr bool kAcc = MODE == kAddSum, kByte = MODE == kByteM;
  __shared__ __attribute__((aligned(16))) std::uint16_t lut[kWaves][256];
  __shared__ __attribute__((aligned(16))) std::uint32_t rows[kWaves][kScanPerWave][2][kRow / 2];
  __shared__ __attribute__((aligned(16))) u32x2 ring[kWaves][8][kScanPerWave];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, grp = lane / kLanesPerScan, l8 = lane % kLanesPerScan;
  // Resident wave index: the wave keeps its LDS rows and its scratch rows for
  // every scanline group it takes from the queue.
  const std::uint64_t slot = std::uint64_t(blockIdx.x) * kWaves + wave;
  if (l8 < kPad / 2) {  // lead sentinels of both rows (never overwritten)
    rows[wave][grp][0][l8] = 0xFFFFFFFFU;
    rows[wave][grp][1][l8] = 0xFFFFFFFFU;
  }
  __attribute__((address_space(1))) std::uint32_t* srow =
      reinterpret_cast<__attribute__((address_space(1))) std::uint32_t*>(
          gptr_mut(scratch + (slot * kScanPerWave + grp) * 2 * std::uint64_t(scratch_row)));
  const int swords = scratch_row / 2;
  if (l8 < kPad / 2) {
    srow[l8] = 0xFFFFFFFFU;
    srow[swords + l8] = 0xFFFFFFFFU;
  }
  int lut_job = -1;
  for (;;) {
  // Next scanline group from the queue (one atomic per wave).
  std::uint32_t item = 0;
  if (lane == 0) item = atomicAdd(queue, 1U);
  item = static_cast<std::uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(item), 0));
  if (item >= groups) break;
  const int t = find_tile(gprefix, ntiles, item);
  const TileDesc T = tiles[t];
  const JobDesc& J = jobs[T.job];
  if (T.job != lut_job) {
    for (int k = lane; k < 256; k += 64) lut[wave][k] = J.lut[k];
    lut_job = T.job;
  }
  __builtin_amdgcn_wave_barrier();
  const int ns = scanlines<DX, DY>(T.w, T.h);
  // Diagonal scanlines are longest in the middle of a tile: take those
  // groups first so that a launch ends with short ones.
  int rank = static_cast<int>(item - gprefix[t]);
  if constexpr (DX != 0 && DY != 0) {
    const int G = static_cast<int>(gprefix[t + 1] - gprefix[t]), mid = G / 2;
    rank = (rank & 1) ? mid - 1 - (rank >> 1) : mid + (rank >> 1);
  }
  const int s0 = rank * kScanPerWave;
  const int sl = min(s0 + grp, ns - 1);  // idle groups shadow the last scanline
  const bool grp_active = s0 + grp < ns;
  int x0, y0, len;
  scan_start<DX, DY>(sl, T.w, T.h, x0, y0, len);
  auto wave_max = [](int v) {
    v = max(v, __shfl_xor(v, 8));
    v = max(v, __shfl_xor(v, 16));
    v = max(v, __shfl_xor(v, 32));
    return __builtin_amdgcn_readfirstlane(v);
  };
  const int steps = wave_max(grp_active ? len : 0);

  const std::uint32_t P1x2 = static_cast<std::uint32_t>(J.p1) * 0x10001U;
  const std::uint64_t* tpix = pix + T.px_base;
  const std::uint32_t* trow = rowbase + T.row_base;
  const std::uint8_t* Ct = C + T.cell_base;
  std::uint16_t* St = static_cast<std::uint16_t*>(out_volume) + T.cell_base;  // not kByte
  std::uint8_t* Mt = static_cast<std::uint8_t*>(out_volume) + T.cell_base;    // kByte

  // Batch of steps [base, base + 8): lane l8 loads step base + l8 (steps past
  // the scanline repeat its last pixel; they are never active).
  auto load_batch = [&](int base, StepBatch& b) {
    const int i = min(base + l8, len - 1);
    const int x = x0 + i * DX, y = y0 + i * DY;
    b.rec = ldb<std::uint64_t>(tpix, static_cast<std::uint32_t>(y * T.w + x) * 8U);
    b.rs = ldb<std::uint32_t>(trow, static_cast<std::uint32_t>(y * T.strips + (x >> kStripShift)) * 4U);
  };
  // Unpacks a batch into the ring (slot l8 of the group); last_ip carries the
  // intensity of the batch's last step to the next batch's first.
  std::uint32_t last_ip = 0;
  auto write_batch = [&](const StepBatch& b) {
    const std::uint32_t ip = static_cast<std::uint32_t>(pix_val(b.rec));
    std::uint32_t prev = __shfl_up(ip, 1U, kLanesPerScan);
    prev = l8 == 0 ? last_ip : prev;
    const std::uint32_t d = static_cast<std::uint32_t>(abs(static_cast<int>(ip) - static_cast<int>(prev))) >> 8;
    ring[wave][l8][grp] = u32x2{b.rs + pix_off(b.rec), static_cast<std::uint32_t>(pix_lo(b.rec)) | d << 16 |
                                                           static_cast<std::uint32_t>(pix_num(b.rec) / kLabelAlign) << 24};
    last_ip = __shfl(ip, kLanesPerScan - 1, kLanesPerScan);
    __builtin_amdgcn_wave_barrier();
    // Keep the shuffles of b ahead of the loads that refill it: otherwise the
    // new record lands in a temporary whose copy into b waits for the load.
    __builtin_amdgcn_sched_barrier(0);
  };
  auto read_step = [&](int i, StepIn& u) {
    const u32x2 e = ring[wave][i & 7][grp];
    u.cell = e.x;
    u.meta = e.y;
  };
  // Costs and S of segment s (lanes past the pixel's labels read its last ones;
  // those values are never used).
  auto load_seg4 = [&](const StepIn& u, SegIn<4>& d) {
    const std::uint32_t cell = u.cell;
    const std::uint32_t j0 = static_cast<std::uint32_t>(min(4 * l8, step_num(u) - 4));
    d.c[0] = ldb<std::uint32_t>(Ct, cell + j0);
    if constexpr (kAcc) {
      const u32x2 v = ldb<u32x2>(St, (cell + j0) * 2U);
      d.s[0] = v.x;
      d.s[1] = v.y;
    }
  };
  auto load_seg8 = [&](const StepIn& u, int s, SegIn<8>& d) {
    const std::uint32_t cell = u.cell;
    const std::uint32_t j0 = static_cast<std::uint32_t>(min(seg_first<8>(s, l8), step_num(u) - 8));
    const u32x2 c = ldb<u32x2>(Ct, cell + j0);
    d.c[0] = c.x;
    d.c[1] = c.y;
    if constexpr (kAcc) {
      const u32x4 v = ldb<u32x4>(St, (cell + j0) * 2U);
      d.s[0] = v.x;
      d.s[1] = v.y;
      d.s[2] = v.z;
      d.s[3] = v.w;
    }
  };
  // Segment 1 only when a scanline of the wave needs it at that step (its
  // pixel has more than 32 labels); the step tests the same condition.
  // The label count / 16 is the top byte of meta: more than 32 labels is
  // meta > 0x02FFFFFF, never for idle groups.
  const std::uint32_t seg1_meta = grp_active ? 0x02FFFFFFU : 0xFFFFFFFFU;
  auto load_segs = [&](const StepIn& u, StepSegs& d) {
    load_seg4(u, d.a);
    if (__builtin_amdgcn_ballot_w64(u.meta > seg1_meta) != 0) load_seg8(u, 1, d.b);
  };

  int prev_lo = 0, prev_num = 0, flip = 0;
  std::uint32_t prev_min = 0;
  StepBatch B;
  // Step i: u, v are its pixel values and segments; it reads the pixel values
  // of step i + kDist + 1 into u_load (first unpacking the batch of that step
  // and loading the next one when it starts a batch), the P2 entry of step
  // i + kDist into u_seg and loads that step's segments into v_load.  The
  // batch of steps [8 b, 8 b + 8) is unpacked at step 8 b - kDist - 1, after
  // the last read of the slots it overwrites (steps 8 b - 8 .. 8 b - 1, read
  // by step 8 b - kDist - 2).
  auto step = [&](int i, const StepIn& u, const StepSegs& v, StepIn& u_load, StepIn& u_seg,
                  StepSegs& v_load) __attribute__((always_inline)) {
    u_seg.p2 = lut[wave][step_p2_index(u_seg)];
    if (((i + kDist + 1) & 7) == 0) {
      write_batch(B);
      load_batch(i + kDist + 1 + 8, B);
    }
    read_step(i + kDist + 1, u_load);
    load_segs(u_seg, v_load);
    const bool act = grp_active && i < len;
    const bool first = i == 0;
    const int lo = step_lo(u), num = step_num(u);
    const std::uint32_t cell = u.cell;
    const std::uint32_t pen = min(prev_min + u.p2, 0xFFFFU);
    const std::uint32_t PENx2 = pen * 0x10001U, MPx2 = prev_min * 0x10001U;
    const int delta = lo - prev_lo;
    const bool prev_wide = prev_num > kNarrow, cur_wide = num > kNarrow;
    const int n_lds = min(prev_num, kNarrow);
    // Label counts of active lanes (0 elsewhere): each ballot is one compare.
    const int num_act = act ? num : 0, prev_act = act ? prev_num : 0;
    const bool any_seg1 = __builtin_amdgcn_ballot_w64(num_act > 32) != 0;
    const bool any_seg2 = __builtin_amdgcn_ballot_w64(num_act > 96) != 0;
    const bool any_prev_wide = __builtin_amdgcn_ballot_w64(prev_act > kNarrow) != 0;
    const bool any_cur_wide = __builtin_amdgcn_ballot_w64(num_act > kNarrow) != 0;
    std::uint32_t* cur = rows[wave][grp][flip];
    const std::uint32_t* prv = rows[wave][grp][flip ^ 1];
    __attribute__((address_space(1))) std::uint32_t* scur = srow + flip * swords;
    const __attribute__((address_space(1))) std::uint32_t* sprv = srow + (flip ^ 1) * swords;
    std::uint32_t m = 0xFFFFFFFFU;

    // Byte position of predecessor label k - 1 for the window of a lane whose
    // first label is j0; k is clamped into [-(P + 1), n + 1] so that the
    // window stays inside the sentinels.
    auto wpos = [&](int P, int j0, int n) {
      return static_cast<std::uint32_t>(min(max(j0 + delta, -(P + 1)), n + 1) - 1 + kPad) * 2U;
    };
    // New path costs of P labels from their window words W (shift sh) and costs.
    // M: L - C.
    auto recur = [&](auto Pc, const std::uint32_t* W, std::uint32_t sh, const std::uint32_t* c, std::uint32_t* L,
                     std::uint32_t* M) {
      constexpr int P = decltype(Pc)::value;
      std::uint32_t Q[P / 2 + 1];
#pragma unroll
      for (int k = 0; k <= P / 2; ++k) Q[k] = __builtin_amdgcn_alignbyte(W[k + 1], W[k], sh);
#pragma unroll
      for (int k = 0; k < P / 2; ++k) {
        const std::uint32_t Cx2 = __builtin_amdgcn_perm(0U, c[k >> 1], (k & 1) ? 0x0c030c02U : 0x0c010c00U);
        if (first) {
          L[k] = Cx2;
          M[k] = 0;
        } else {
          const std::uint32_t p12 = __builtin_amdgcn_alignbyte(Q[k + 1], Q[k], 2U);
          const u16x2 nb =
              __builtin_elementwise_add_sat(__builtin_elementwise_min(as_pair(Q[k]), as_pair(Q[k + 1])), as_pair(P1x2));
          const u16x2 best = __builtin_elementwise_min(__builtin_elementwise_min(as_pair(p12), nb), as_pair(PENx2));
          M[k] = as_u32(best - as_pair(MPx2));
          L[k] = as_u32(as_pair(M[k]) + as_pair(Cx2));
        }
      }
    };
    // LDS window of a lane.
    auto lds_window = [&](auto Pc, int j0, std::uint32_t* W, std::uint32_t& sh) {
      constexpr int P = decltype(Pc)::value;
      sh = wpos(P, j0, n_lds);
      const std::uint32_t* wp = prv + (sh >> 2);
#pragma unroll
      for (int k = 0; k < P / 2 + 2; ++k) W[k] = wp[k];
    };
    // Scratch window of a lane (in range for every lane; used where prev_wide).
    auto scr_window = [&](auto Pc, int j0, std::uint32_t* W, std::uint32_t& sh) {
      constexpr int P = decltype(Pc)::value;
      sh = wpos(P, j0, prev_num);
      const auto wp = sprv + (sh >> 2);
#pragma unroll
      for (int k = 0; k < P / 2 + 2; ++k) W[k] = wp[k];
    };
    // Stores of a lane's new path costs (next step's row) and S; running min.
    // kLow: segments 0 and 1, whose labels (below 96) lie inside the LDS row
    // of every lane.  Their row store needs no condition: a lane past its
    // pixel's labels, or of a finished scanline, writes only positions the
    // next step does not read (the sentinels after the labels are written
    // later in the step, and reads stop inside them), and a wide pixel's row
    // is read from scratch.
    auto emit = [&](auto Pc, auto kLow, int j0, const std::uint32_t* L, const std::uint32_t* M, const std::uint32_t* sv) {
      constexpr int P = decltype(Pc)::value;
      const bool on = act && j0 < num;
      const int w0 = (kPad + j0) >> 1;
      if (decltype(kLow)::value || (on && !cur_wide)) {
#pragma unroll
        for (int k = 0; k < P / 2; k += 2) *reinterpret_cast<u32x2*>(cur + w0 + k) = u32x2{L[k], L[k + 1]};
      }
      if (any_cur_wide) {
        if (on && cur_wide) {
#pragma unroll
          for (int k = 0; k < P / 2; ++k) scur[w0 + k] = L[k];
        }
      }
      std::uint32_t out[P / 2];
      std::uint32_t mm = L[0];
#pragma unroll
      for (int k = 0; k < P / 2; ++k) {
        out[k] = kAcc ? as_u32(as_pair(sv[k]) + as_pair(L[k])) : L[k];
        if (k > 0) mm = as_u32(__builtin_elementwise_min(as_pair(mm), as_pair(L[k])));
      }
      if (on) {
        const std::uint32_t off = (cell + static_cast<std::uint32_t>(j0)) * 2U;
        if constexpr (kByte && P == 4) {
          stb<std::uint32_t>(Mt, cell + static_cast<std::uint32_t>(j0), __builtin_amdgcn_perm(M[1], M[0], 0x06040200U));
        } else if constexpr (kByte) {
          stb<u32x2>(Mt, cell + static_cast<std::uint32_t>(j0),
                     u32x2{__builtin_amdgcn_perm(M[1], M[0], 0x06040200U),
                           __builtin_amdgcn_perm(M[3], M[2], 0x06040200U)});
        } else if constexpr (P == 4) {
          stb<u32x2>(St, off, u32x2{out[0], out[1]});
        } else {
          stb<u32x4>(St, off, u32x4{out[0], out[1], out[2], out[3]});
        }
      }
      m = on ? as_u32(__builtin_elementwise_min(as_pair(m), as_pair(mm))) : m;
    };
    using P4 = std::integral_constant<int, 4>;
    using P8 = std::integral_constant<int, 8>;
    // A lane's window: from LDS, or from its scratch row where prev_wide.  The
    // scratch loads are retired inside their block, so that the shared code
    // after it never waits on them.
    auto window = [&](auto Pc, int j0, std::uint32_t* W, std::uint32_t& sh) {
      constexpr int P = decltype(Pc)::value;
      lds_window(Pc, j0, W, sh);
      if (any_prev_wide) {
        std::uint32_t G[P / 2 + 2], gsh;
        scr_window(Pc, j0, G, gsh);
        __builtin_amdgcn_s_waitcnt(kVmcnt0);
#pragma unroll
        for (int k = 0; k < P / 2 + 2; ++k) W[k] = prev_wide ? G[k] : W[k];
        sh = prev_wide ? gsh : sh;
      }
    };
    auto seg8 = [&](int s, const SegIn<8>& d) {
      const int j0 = seg_first<8>(s, l8);
      std::uint32_t W[6], sh, L[4], M[4];
      window(P8{}, j0, W, sh);
      recur(P8{}, W, sh, d.c, L, M);
      emit(P8{}, std::true_type{}, j0, L, M, d.s);
    };
    auto seg4 = [&](const SegIn<4>& d) {
      const int j0 = seg_first<4>(0, l8);
      std::uint32_t W[4], sh, L[2], M[2];
      window(P4{}, j0, W, sh);
      recur(P4{}, W, sh, d.c, L, M);
      emit(P4{}, std::true_type{}, j0, L, M, d.s);
    };
    // Segments from 2 on (pixels of more than 96 labels): costs, S and the
    // scratch window of every lane (used where prev_wide) loaded one segment
    // ahead.  No load in the loop is conditional and the loop has one exit,
    // so the waits inside it only cover the segment being computed.
    auto wide = [&]() {
      const int segmax = wave_max(act ? segments(num) : 0);
      struct Ahead {
        SegIn<8> d;
        std::uint32_t G[6];
      } A, B;
      auto load = [&](int s, Ahead& x) {
        load_seg8(u, s, x.d);
        std::uint32_t gsh;
        scr_window(P8{}, seg_first<8>(s, l8), x.G, gsh);
      };
      auto run = [&](int s, const Ahead& x) {
        const int j0 = seg_first<8>(s, l8);
        std::uint32_t W[6], sh, L[4], M[4];
        lds_window(P8{}, j0, W, sh);
        const std::uint32_t gsh = wpos(8, j0, prev_num);
#pragma unroll
        for (int k = 0; k < 6; ++k) W[k] = prev_wide ? x.G[k] : W[k];
        sh = prev_wide ? gsh : sh;
        recur(P8{}, W, sh, x.d.c, L, M);
        emit(P8{}, std::false_type{}, j0, L, M, x.d.s);
      };
      load(2, A);
      for (int s = 2; s < segmax; s += 2) {
        load(s + 1, B);
        run(s, A);
        load(s + 2, A);
        if (s + 1 < segmax) run(s + 1, B);
      }
      // Retire the loads of the segments past the end.
      __builtin_amdgcn_s_waitcnt(kVmcnt0);
    };
    seg4(v.a);
    if (any_seg1) seg8(1, v.b);
    if (any_seg2) wide();
    // Sentinels after the labels (in the LDS row also for finished
    // scanlines, whose rows are not read again).
    if (l8 < kPad / 2) {
      const int w = ((kPad + num) >> 1) + l8;
      if (!cur_wide) cur[w] = 0xFFFFFFFFU;
      if (any_cur_wide && act && cur_wide) scur[w] = 0xFFFFFFFFU;
    }
    prev_min = min8(min(m & 0xFFFFU, m >> 16));
    prev_lo = lo;
    prev_num = num;
    flip ^= 1;
    __builtin_amdgcn_wave_barrier();  // this step's row writes before the next step's reads
  };

  // Register rotation: kDist + 2 sets of pixel values, kDist + 1 of segments,
  // the loop unrolled over a full period so every index is a constant.
  constexpr int NU = kDist + 2, NV = kDist + 1;
  StepIn U[NU];
  StepSegs V[NV];
  static_assert(kDist + 1 < 8, "the prologue reads the first batch only");
  load_batch(0, B);
  write_batch(B);
  load_batch(8, B);
  for (int j = 0; j <= kDist; ++j) read_step(j, U[j]);
  for (int j = 0; j < kDist; ++j) U[j].p2 = lut[wave][step_p2_index(U[j])];
  for (int j = 0; j < kDist; ++j) load_segs(U[j], V[j]);
  auto body = [&](auto Kc, int i) __attribute__((always_inline)) {
    constexpr int K = decltype(Kc)::value;
    step(i, U[K % NU], V[K % NV], U[(K + kDist + 1) % NU], U[(K + kDist) % NU], V[(K + kDist) % NV]);
  };
  for (int i = 0; i < steps; i += NU * NV) {
    [&]<int... K>(std::integer_sequence<int, K...>) __attribute__((always_inline)) {
      (body(std::integral_constant<int, K>{}, i + K), ...);
    }(std::make_integer_sequence<int, NU * NV>{});
  }
  // Retire this group's loads before the next group reuses their registers.
  __builtin_amdgcn_s_waitcnt(kVmcnt0);
  }
}

// ------------------------------------------------------------------ full-range scans
// The eight path scans of tiles whose pixels all have the same D labels (no
// label ranges: single-level matches, the coarsest level of a hierarchy).
// Nothing has to be aligned, so a scanline is LPS lanes (the power of two from
// D / PL on, lane q holding labels PL q .. PL q + PL - 1 as packed pairs) and the
// predecessor's path costs never leave their registers: the two neighbours
// across lanes and the minimum over the labels are DPP moves.  A wave scans
// 64 / LPS neighbouring scanlines in lockstep: columns of a tile row for the
// vertical and diagonal paths (a diagonal scanline moves one column per row
// and re-enters at the other side of the tile, as a new scanline, when it
// leaves), rows of a tile column for the horizontal ones.  Each path stores
// M = L - C, at most P2 and so one byte, into its own plane: no path waits
// for another's sums, and all eight are one launch.
//
// Bound by the chain of a step at small sizes and by HBM at large ones (a byte
// read and a byte written per label and path).  Aggregation of a 640x480 pair
// with 64 labels: 0.92 ms with eight k_path launches, 0.19 ms with 16 labels a
// lane, 0.147 ms here; 1024x768 with 128 labels: 3.4 ms, 0.92 ms, 0.76 ms (1.9 GB
// written and 2 GB read).
// Value of the lane below (above) in a wave; 0 in the first (last) lane.  Like
// the moves of the minima these fold into the operation that takes them.
template <int LPS>
__device__ __forceinline__ std::uint32_t lane_below(std::uint32_t v) {
  const int i = static_cast<int>(v);
  return static_cast<std::uint32_t>(LPS <= 16 ? __builtin_amdgcn_update_dpp(0, i, 0x111, 0xF, 0xF, true)
                                              : __builtin_amdgcn_update_dpp(0, i, 0x138, 0xF, 0xF, true));
}
template <int LPS>
__device__ __forceinline__ std::uint32_t lane_above(std::uint32_t v) {
  const int i = static_cast<int>(v);
  return static_cast<std::uint32_t>(LPS <= 16 ? __builtin_amdgcn_update_dpp(0, i, 0x101, 0xF, 0xF, true)
                                              : __builtin_amdgcn_update_dpp(0, i, 0x130, 0xF, 0xF, true));
}
template <int CTRL>
__device__ __forceinline__ std::uint32_t dpp_min(std::uint32_t v) {
  const int i = static_cast<int>(v);
  return min(v, static_cast<std::uint32_t>(__builtin_amdgcn_update_dpp(0, i, CTRL, 0xF, 0xF, true)));
}
// Minimum over aligned groups of LPS lanes.
template <int LPS>
__device__ __forceinline__ std::uint32_t group_min(std::uint32_t v) {
  if constexpr (LPS >= 2) v = dpp_min<0xB1>(v);   // quad_perm 1 0 3 2
  if constexpr (LPS >= 4) v = dpp_min<0x4E>(v);   // quad_perm 2 3 0 1
  if constexpr (LPS >= 8) v = dpp_min<0x141>(v);  // row_half_mirror
  if constexpr (LPS >= 16) v = dpp_min<0x140>(v); // row_mirror
  if constexpr (LPS >= 32) {
    const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    v = min(r[0], r[1]);
  }
  if constexpr (LPS >= 64) {
    const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    v = min(r[0], r[1]);
  }
  return v;
}

template <int LPS, int PL>
__global__ __launch_bounds__(64 * kWaves) void k_full(FullArgs A) {
  constexpr int S = 64 / LPS, W = PL / 2, B = PL / 4;
  using Bytes = std::uint32_t __attribute__((ext_vector_type(B)));
  __shared__ std::uint32_t lut[256];
  // The P2 table depends on the options only: the same for every job.
  for (int k = threadIdx.x; k < 256; k += 64 * kWaves) lut[k] = A.jobs[0].lut[k] * 0x10001U;
  __syncthreads();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, sc = lane / LPS, q = lane % LPS;
  const std::uint64_t item = std::uint64_t(blockIdx.x) * kWaves + wave;
  if (item >= A.groups) return;
  const auto gprefix = cptr(A.gprefix);
  int t = 0;
  for (int hi = A.ntiles - 1; t < hi;) {
    const int mid = (t + hi + 1) >> 1;
    if (gprefix[mid] <= item) {
      t = mid;
    } else {
      hi = mid - 1;
    }
  }
  const auto& T = cptr(A.tiles)[t];
  const auto& J = cptr(A.jobs)[T.job];
  const int tw = T.w, th = T.h, D = J.D;
  int path = 0, g = static_cast<int>(item - gprefix[t]);
  for (; path < kPaths - 1; ++path) {
    const int n = ((path < 2 ? th : tw) + S - 1) / S;
    if (g < n) break;
    g -= n;
  }
  // Paths 0, 1: along rows; 2, 3: along columns; 4 .. 7: diagonals.  dx:
  // columns a scanline moves per step; odd paths run from the last row
  // (column) to the first.
  const bool horiz = path < 2, rev = (path & 1) != 0;
  const int dx = path < 4 ? 0 : (path == 4 || path == 7 ? 1 : -1);
  const int nscan = horiz ? th : tw, steps = horiz ? tw : th;
  const int s = min(g * S + sc, nscan - 1);
  const bool on = g * S + sc < nscan && PL * q < D;
  const std::uint8_t* Ct = A.C + T.cell_base;
  std::uint8_t* Mt = A.M + std::uint64_t(path) * A.mstride + T.cell_base;
  const std::uint16_t* img = J.img + std::int64_t(T.y0) * J.img_stride;
  const int img_stride = static_cast<int>(J.img_stride);
  // Base columns of a mirrored job read the unmirrored image backwards.
  const int ix0 = J.mirrored != 0 ? J.width - 1 - T.x0 : T.x0, idx = J.mirrored != 0 ? -1 : 1;
  const u16x2 P1x2 = as_pair(static_cast<std::uint32_t>(J.p1) * 0x10001U);
  // Sentinels for the neighbours of the first and the last label, and for the labels of idle lanes.
  const std::uint32_t left_inf = q == 0 ? 0xFFFFFFFFU : 0U, right_inf = PL * (q + 1) >= D ? 0xFFFFFFFFU : 0U;
  const std::uint32_t off_inf = on ? 0U : 0xFFFFFFFFU;

  // Offsets of the next pixel to load: they move by a constant per step, and
  // by another at the step a diagonal leaves the tile (left steps from now).
  const int x0 = horiz ? (rev ? tw - 1 : 0) : s, y0 = horiz ? s : (rev ? th - 1 : 0);
  const int sx = horiz ? (rev ? -1 : 1) : dx, sy = horiz ? 0 : (rev ? -1 : 1);
  std::uint32_t cell = static_cast<std::uint32_t>(y0 * tw + x0) * static_cast<std::uint32_t>(D) +
                       static_cast<std::uint32_t>(PL * min(q, D / PL - 1));
  std::uint32_t pix = static_cast<std::uint32_t>(y0 * img_stride + ix0 + idx * x0) * 2U;
  const std::uint32_t cmove = static_cast<std::uint32_t>((sy * tw + sx) * D);
  const std::uint32_t pmove = static_cast<std::uint32_t>(sy * img_stride + idx * sx) * 2U;
  const std::uint32_t cwrap = cmove - static_cast<std::uint32_t>(dx * tw * D);
  const std::uint32_t pwrap = pmove - static_cast<std::uint32_t>(idx * dx * tw) * 2U;
  int left = dx == 0 ? 1 << 30 : (dx > 0 ? nscan - s : s + 1);
  bool start = true;
  struct In {
    Bytes c;
    std::uint32_t cell, val;
    bool first;  // starts a scanline
  };
  auto load = [&](In& d) __attribute__((always_inline)) {
    d.cell = cell;
    d.c = ldb<Bytes>(Ct, cell);
    d.val = ldb<std::uint16_t>(img, pix);
    d.first = start;
    start = --left == 0;
    left = start ? nscan : left;
    cell += start ? cwrap : cmove;
    pix += start ? pwrap : pmove;
  };
  // Path costs, their minimum and the next step's P2, as pairs.
  std::uint32_t L[W], pmin = 0, p2 = 0;
#pragma unroll
  for (int j = 0; j < W; ++j) L[j] = 0xFFFFFFFFU;
  auto step = [&](const In& in, const In& next) __attribute__((always_inline)) {
    const u16x2 MP = as_pair(in.first ? 0U : pmin), PEN = as_pair(in.first ? 0U : pmin + p2);
    // P2 of the next step, read while this one computes.
    p2 = lut[__builtin_amdgcn_sad_u16(in.val, next.val, 0U) >> 8];
    const std::uint32_t below = lane_below<LPS>(L[W - 1]) | left_inf, above = lane_above<LPS>(L[0]) | right_inf;
    std::uint32_t Q[W + 1], M[W];
    Q[0] = __builtin_amdgcn_alignbyte(L[0], below, 2U);
#pragma unroll
    for (int j = 1; j < W; ++j) Q[j] = __builtin_amdgcn_alignbyte(L[j], L[j - 1], 2U);
    Q[W] = __builtin_amdgcn_alignbyte(above, L[W - 1], 2U);
#pragma unroll
    for (int j = 0; j < W; ++j) {
      const std::uint32_t Cx2 = __builtin_amdgcn_perm(0U, in.c[j >> 1], (j & 1) ? 0x0c030c02U : 0x0c010c00U);
      const u16x2 nb = __builtin_elementwise_add_sat(__builtin_elementwise_min(as_pair(Q[j]), as_pair(Q[j + 1])), P1x2);
      const u16x2 best = __builtin_elementwise_min(__builtin_elementwise_min(as_pair(L[j]), nb), PEN);
      M[j] = as_u32(best - MP);
      L[j] = as_u32(as_pair(M[j]) + as_pair(Cx2));
    }
    u16x2 m[W];
#pragma unroll
    for (int j = 0; j < W; ++j) m[j] = as_pair(L[j]);
#pragma unroll
    for (int n = W / 2; n > 0; n /= 2)
#pragma unroll
      for (int j = 0; j < n; ++j) m[j] = __builtin_elementwise_min(m[j], m[j + n]);
    const std::uint32_t both = as_u32(m[0]) | off_inf;
    // Equal halves from here on: the order of the words is the order of the costs.
    pmin = group_min<LPS>(as_u32(__builtin_elementwise_min(as_pair(both), as_pair(both >> 16 | both << 16))));
    if (on) {
      Bytes o;
#pragma unroll
      for (int j = 0; j < B; ++j) o[j] = __builtin_amdgcn_perm(M[2 * j + 1], M[2 * j], 0x06040200U);
      stb_nt<Bytes>(Mt, in.cell, o);
    }
  };
  // Costs and intensities N - 1 steps ahead; the loops are unrolled over the N
  // sets so that every index is a constant.  The first one loads in every step.
  constexpr int N = 8;
  In in[N];
#pragma unroll
  for (int j = 0; j < N; ++j) {
    in[j] = In{};  // all N: a scanline of N - 1 steps reads the one that none of its loads fills
    if (j < N - 1 && j < steps) load(in[j]);
  }
  int i = 0;
  for (; i + 2 * N - 1 <= steps; i += N) {
#pragma unroll
    for (int j = 0; j < N; ++j) {
      load(in[(j + N - 1) % N]);
      step(in[j], in[(j + 1) % N]);
    }
  }
  for (; i < steps; i += N) {
#pragma unroll
    for (int j = 0; j < N; ++j) {
      if (i + j < steps) {
        if (i + j + N - 1 < steps) load(in[(j + N - 1) % N]);
        step(in[j], in[(j + 1) % N]);
      }
    }
  }
}

// ------------------------------------------------------------------ row sweeps
// The vertical and diagonal scans of tiles with label ranges.  A block sweeps
// one tile row by row, downwards or upwards, and advances NP paths at once:
// all three whose predecessors lie in the last row (NP = 3), so that a row's
// costs are read and its sums written once for three paths, or one of them
// (NP = 1, more blocks where there are few tiles).  A thread takes chunks (16
// labels of a pixel) of the row, whatever pixel they belong to, so that wide
// and narrow pixels keep the lanes equally busy; cmap holds each chunk's
// column and place in its pixel.
//
// The last row's path costs of every path stay in LDS as uint16: pixel x's
// labels from word 8 k + x + 1 on, k its first chunk, a word of sentinels
// between neighbouring pixels (odd strides between one-chunk pixels: no bank
// conflicts).  Pixels past the LDS rows (cap words, the end of rows with many
// wide pixels) use rows of the same layout in a global scratch, one per
// parity.  Each row is two phases between barriers: windows and minima of the
// last row are read, the new costs stay in registers (H chunks per thread;
// later ones are past cap and go to scratch) until every thread has read, then
// they replace the last row.  Costs, map and records are loaded one row ahead.
//
// Bound by CU time: a block fills its CU's LDS and registers, and its 16 waves
// issue vector instructions (about 180 per chunk and path with three paths, 260
// with one) in 60 to 75% of the time, between the two barriers of a row (with
// three paths at the limit of 128 registers, 76 bytes a lane in scratch).  The
// six paths of the 24 MP pair's finest level: 19 ms by k_path; 11.5 ms here.
// Barrier that orders LDS accesses only: loads in flight and stores of sums
// stay in flight across it.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <int NP, bool kByte, int H>
__global__ __launch_bounds__(kSweepThreads) void k_sweep(SweepArgs A) {
  static_assert(NP == 1 || !kByte, "a byte holds L - C of one path");
  constexpr int N = kSweepThreads;
  extern __shared__ __attribute__((aligned(16))) std::uint32_t lds[];
  // info[3][wpad] (pixel records of three rows), pmin[2][NP][wpad], lut, item, rows[NP][cap + pad].
  const int wpad = A.wpad, cap = A.cap, rstride = cap + kSweepRowPad;
  u32x2* const info = reinterpret_cast<u32x2*>(lds);
  std::uint32_t* const pmin = lds + 6 * wpad;
  std::uint16_t* const lut = reinterpret_cast<std::uint16_t*>(pmin + 2 * NP * wpad);
  std::uint32_t* const sitem = pmin + 2 * NP * wpad + 128;
  std::uint32_t* const rows = sitem + 4;
  const int tid = static_cast<int>(threadIdx.x), lane = tid & 63;
  const int wave0 = __builtin_amdgcn_readfirstlane(tid & ~63);  // first thread of the wave
  if (tid < 256) lut[tid] = A.jobs[0].lut[tid];
  auto* const scr = gptr_mut(A.scratch + std::uint64_t(blockIdx.x) * 2 * NP * A.swords);
  constexpr int kUnits = NP == 3 ? 2 : 6;
  for (;;) {
    if (tid == 0) *sitem = atomicAdd(A.queue, 1U);
    __syncthreads();
    const std::uint32_t item = static_cast<std::uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(*sitem)));
    if (item >= A.units) break;
    const int t = cptr(A.order)[item / kUnits], u = static_cast<int>(item % kUnits);
    const auto& T = cptr(A.tiles)[t];
    const int w = T.w, h = T.h;
    const bool rev = (u & 1) != 0;
    // Columns from the predecessor: 0, 1, -1 (paths 2/3, 4/5, 6/7; upwards 0, -1, 1).
    const int dx1 = (u >> 1) == 0 ? 0 : (((u >> 1) == 1) != rev ? 1 : -1);
    auto path_dx = [&](int p) { return NP == 3 ? (p == 0 ? 0 : (p == 1 ? 1 : -1)) : dx1; };
    const std::uint32_t P1x2 = static_cast<std::uint32_t>(cptr(A.jobs)[T.job].p1) * 0x10001U;
    const std::uint32_t* rbase = A.rowbase + T.row_base;
    const std::uint64_t* tpix = A.pix + T.px_base;
    const std::uint8_t* Ct = A.C + T.cell_base;
    const std::uint32_t* tmap = A.cmap + T.cell_base / kLabelAlign;
    std::uint16_t* St = static_cast<std::uint16_t*>(A.out[u]) + T.cell_base;  // not kByte
    std::uint8_t* Mt = static_cast<std::uint8_t*>(A.out[u]) + T.cell_base;    // kByte
    const std::uint32_t tcells = T.cells;
    auto row_y = [&](int i) { return rev ? h - 1 - i : i; };
    // First cells of 64 rows at a time, one per lane; fcell(i) is that of row
    // i, and of the row past the last one the other end of the volume.
    std::uint32_t rb = 0;
    auto load_rb = [&](int i0) {
      rb = rbase[row_y(min(i0 + lane, h - 1))];
      __builtin_amdgcn_s_waitcnt(kVmcnt0);
    };
    auto fcell = [&](int i) {
      return i < h ? static_cast<std::uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(rb), i & 63)) : tcells;
    };
    load_rb(0);
    std::uint32_t first = fcell(0), next = h > 1 ? fcell(1) : tcells;
    int K = static_cast<int>((rev ? tcells - first : next - first) >> 4);
    // The record of column tid in row i (clamped: unused values).
    auto load_pix = [&](int i) {
      return ldb<u32x2>(tpix, static_cast<std::uint32_t>(row_y(min(i, h - 1)) * w + min(tid, w - 1)) * 8U);
    };
    u32x4 c[H];
    std::uint32_t cm[H];
    auto load_chunk = [&](int r, std::uint32_t f, int n) {
      const std::uint32_t k = static_cast<std::uint32_t>(min(tid + N * r, n - 1));
      c[r] = ldb<u32x4>(Ct, f + 16U * k);
      cm[r] = ldb<std::uint32_t>(tmap, ((f >> 4) + k) * 4U);
    };

    // Where chunk m's window of path p lies, for pixel records `own` in row
    // `info o` and predecessors in `info l`: bits 0-15 the window's first word
    // in the LDS row, bits 16-28 P2, bit 29 the window starts on an odd label,
    // bit 30 a predecessor exists, bit 31 the window needs the general read
    // (past a sentinel on either side, or in scratch).
    auto window = [&](std::uint32_t m, const u32x2& own, const u32x2* linfo, int p) {
      const int x = map_col(m), xp = x - path_dx(p);
      const bool use = xp >= 0 && xp < w;
      const int xq = use ? xp : 0;
      const u32x2 pi = linfo[xq];
      const std::uint32_t ia = own.y >> 16, ib = pi.y >> 16;
      const std::uint32_t p2 = lut[(max(ia, ib) - min(ia, ib)) >> 8];
      const int pw = static_cast<int>(pi.x >> 24) * 8, base = 8 * static_cast<int>(pi.x & 0xFFFFFFU) + xq + 1;
      const int k0 = static_cast<int>(own.y & 0xFFFFU) + kLabelAlign * map_place(m) -
                     static_cast<int>(pi.y & 0xFFFFU);
      const bool far = static_cast<unsigned>(k0 + 1) > static_cast<unsigned>(2 * pw - 14) || base + pw >= cap;
      const std::uint32_t at = use && !far ? static_cast<std::uint32_t>(base + ((k0 - 1) >> 1)) : 0U;
      return at | p2 << 16 | (static_cast<std::uint32_t>(k0) & 1U) << 29 | (use ? 1U << 30 : 0U) |
             (use && far ? 1U << 31 : 0U);
    };
    // A chunk's column, and what its row needs: bit 16 the pixel's first
    // chunk, bit 17 its last, bit 18 the pixel's costs go to LDS.
    auto place = [&](std::uint32_t m, const u32x2& own) {
      const int x = map_col(m), cc = map_place(m), n16 = static_cast<int>(own.x >> 24);
      const bool in_lds = 8 * (static_cast<int>(own.x & 0xFFFFFFU) + n16) + x + 1 < cap;
      return static_cast<std::uint32_t>(x) | (cc == 0 ? 1U << 16 : 0U) | (cc == n16 - 1 ? 1U << 17 : 0U) |
             (in_lds ? 1U << 18 : 0U);
    };
    std::uint32_t pre[H][NP], flags[H];
    // Windows and places of the held chunks of a row of n chunks.
    auto prepare = [&](const u32x2* cinfo, const u32x2* linfo, int n, bool top) __attribute__((always_inline)) {
#pragma unroll
      for (int r = 0; r < H; ++r) {
        flags[r] = 0;
#pragma unroll
        for (int p = 0; p < NP; ++p) pre[r][p] = 0;
        if (tid + N * r < n) {
          const u32x2 own = cinfo[map_col(cm[r])];
          flags[r] = place(cm[r], own);
#pragma unroll
          for (int p = 0; p < NP; ++p) pre[r][p] = top ? 0U : window(cm[r], own, linfo, p);
        }
      }
    };

#pragma unroll
    for (int r = 0; r < H; ++r) load_chunk(r, first, K);
    const u32x2 p0 = load_pix(0);
    u32x2 pr = load_pix(1);
    if (tid < w) {
      info[tid] = p0;
#pragma unroll
      for (int p = 0; p < NP; ++p) pmin[p * wpad + tid] = 0xFFFFU;
    }
    lds_barrier();
    prepare(info, info, K, true);
    int i0 = 0, i1 = 1, i2 = 2;  // info buffers of this, the next and the last row
    for (int i = 0; i < h; ++i) {
      std::uint32_t* const cmin = pmin + (i & 1) * NP * wpad;
      std::uint32_t* const lmin = pmin + ((i & 1) ^ 1) * NP * wpad;
      auto* const cscr = scr + (i & 1) * NP * A.swords;
      const auto* const lscr = scr + ((i & 1) ^ 1) * NP * A.swords;
      const u32x2* const cinfo = info + i0 * wpad;
      const u32x2* const linfo = info + i2 * wpad;
      // Chunks of the next row (of this one again after the last).
      if (((i + 2) & 63) == 0) load_rb(i + 2);
      const std::uint32_t after = fcell(i + 2);
      const bool last = i + 1 >= h;
      const std::uint32_t nfirst = last ? first : next;
      const int nK = last ? K : static_cast<int>((rev ? first - next : after - next) >> 4);

      // New path costs of chunk k (map entry m, windows pr, unpacked costs
      // Cx2) into L, their sum to S, their minima to cmin.
      auto chunk = [&](int k, std::uint32_t m, const std::uint32_t (&pp)[NP], const std::uint32_t (&Cx2)[8],
                       std::uint32_t (&L)[NP][8]) __attribute__((always_inline)) {
        const int x = map_col(m);
        std::uint32_t sum[8];
#pragma unroll
        for (int p = 0; p < NP; ++p) {
          const std::uint32_t v = pp[p];
          const bool use = (v & (1U << 30)) != 0, far = (v & (1U << 31)) != 0;
          const std::uint32_t pm = lmin[p * wpad + (use ? x - path_dx(p) : 0)];
          const std::uint32_t* const lrow = rows + p * rstride;
          std::uint32_t W[10], sh = ((v >> 29) & 1U) != 0 ? 0U : 16U;
          const std::uint32_t* wp = lrow + (v & 0xFFFFU);
#pragma unroll
          for (int j = 0; j < 10; ++j) W[j] = wp[j];
          if (__builtin_amdgcn_ballot_w64(far) != 0) {
            if (far) {
              const int xq = x - path_dx(p);
              const u32x2 own = cinfo[x], pi = linfo[xq];
              const int pw = static_cast<int>(pi.x >> 24) * 8, base = 8 * static_cast<int>(pi.x & 0xFFFFFFU) + xq + 1;
              const int k0 = static_cast<int>(own.y & 0xFFFFU) + kLabelAlign * map_place(m) -
                             static_cast<int>(pi.y & 0xFFFFU);
              const int w0 = (k0 - 1) >> 1;
              if (base + pw < cap) {
#pragma unroll
                for (int j = 0; j < 10; ++j) W[j] = lrow[base + min(max(w0 + j, -1), pw)];
              } else {
                const auto* sp = lscr + p * A.swords + base;
#pragma unroll
                for (int j = 0; j < 10; ++j) W[j] = sp[min(max(w0 + j, -1), pw)];
                __builtin_amdgcn_s_waitcnt(kVmcnt0);
              }
            }
          }
          const std::uint32_t mpv = use ? pm : 0U, pen = use ? pm + ((v >> 16) & 0x1FFFU) : 0U;
          const std::uint32_t PENx2 = pen * 0x10001U, MPx2 = mpv * 0x10001U;
          std::uint32_t Q[9], mm = 0xFFFFFFFFU;
#pragma unroll
          for (int j = 0; j < 9; ++j) Q[j] = __builtin_amdgcn_alignbit(W[j + 1], W[j], sh);
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const std::uint32_t p12 = __builtin_amdgcn_alignbyte(Q[j + 1], Q[j], 2U);
            const u16x2 nb = __builtin_elementwise_add_sat(
                __builtin_elementwise_min(as_pair(Q[j]), as_pair(Q[j + 1])), as_pair(P1x2));
            const u16x2 best = __builtin_elementwise_min(__builtin_elementwise_min(as_pair(p12), nb), as_pair(PENx2));
            const u16x2 M = best - as_pair(MPx2);
            L[p][j] = as_u32(M + as_pair(Cx2[j]));
            sum[j] = kByte ? as_u32(M) : (p == 0 ? L[p][j] : as_u32(as_pair(sum[j]) + as_pair(L[p][j])));
            mm = as_u32(__builtin_elementwise_min(as_pair(mm), as_pair(L[p][j])));
          }
          atomicMin(&cmin[p * wpad + x], min(mm & 0xFFFFU, mm >> 16));
        }
        const std::uint32_t at = first + 16U * static_cast<std::uint32_t>(k);
        if constexpr (kByte) {
          u32x4 o;
#pragma unroll
          for (int j = 0; j < 4; ++j) o[j] = __builtin_amdgcn_perm(sum[2 * j + 1], sum[2 * j], 0x06040200U);
          stb_nt<u32x4>(Mt, at, o);
        } else {
          stb_nt<u32x4>(St, 2U * at, u32x4{sum[0], sum[1], sum[2], sum[3]});
          stb_nt<u32x4>(St, 2U * at + 16U, u32x4{sum[4], sum[5], sum[6], sum[7]});
        }
      };
      // A chunk's costs into a row, with the sentinels around its pixel.
      auto put = [&](auto* row, int k, std::uint32_t f, const std::uint32_t (&L)[8]) __attribute__((always_inline)) {
        auto* d = row + 8 * k + static_cast<int>(f & 0xFFFFU) + 1;
#pragma unroll
        for (int j = 0; j < 8; ++j) d[j] = L[j];
        if ((f & (1U << 16)) != 0) d[-1] = 0xFFFFFFFFU;
        if ((f & (1U << 17)) != 0) d[8] = 0xFFFFFFFFU;
      };
      auto unpack = [&](const u32x4& cw, std::uint32_t (&Cx2)[8]) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 8; ++j)
          Cx2[j] = __builtin_amdgcn_perm(0U, cw[j >> 1], (j & 1) ? 0x0c030c02U : 0x0c010c00U);
      };
      std::uint32_t L[H][NP][8];
      bool spilled = false;
#pragma unroll
      for (int r = 0; r < H; ++r) {
        // Waves without a chunk in this row and the next have nothing to do.
        if (wave0 + N * r >= max(K, nK)) continue;
        const int k = tid + N * r;
        std::uint32_t Cx2[8];
        unpack(c[r], Cx2);
        const std::uint32_t m = cm[r];
        load_chunk(r, nfirst, nK);
        if (k < K) {
          chunk(k, m, pre[r], Cx2, L[r]);
          if ((flags[r] & (1U << 18)) == 0) {
            spilled = true;
#pragma unroll
            for (int p = 0; p < NP; ++p) put(cscr + p * A.swords, k, flags[r], L[r][p]);
          }
        }
      }
      // Chunks past the held ones lie past cap.
      for (int k = tid + N * H; k < K; k += N) {
        std::uint32_t Cx2[8], X[NP][8], pp[NP];
        const std::uint32_t m = ldb<std::uint32_t>(tmap, ((first >> 4) + static_cast<std::uint32_t>(k)) * 4U);
        unpack(ldb<u32x4>(Ct, first + 16U * static_cast<std::uint32_t>(k)), Cx2);
        const u32x2 own = cinfo[map_col(m)];
#pragma unroll
        for (int p = 0; p < NP; ++p) pp[p] = i == 0 ? 0U : window(m, own, linfo, p);
        chunk(k, m, pp, Cx2, X);
        spilled = true;
        const std::uint32_t f = place(m, own);
#pragma unroll
        for (int p = 0; p < NP; ++p) put(cscr + p * A.swords, k, f, X[p]);
      }
      if (tid < w) info[i1 * wpad + tid] = pr;
      pr = load_pix(i + 2);
      // Scratch rows have to be in place before another wave reads them.
      if (__builtin_amdgcn_ballot_w64(spilled) != 0) __builtin_amdgcn_s_waitcnt(kVmcnt0);
      lds_barrier();
#pragma unroll
      for (int r = 0; r < H; ++r) {
        if ((flags[r] & (1U << 18)) != 0) {
#pragma unroll
          for (int p = 0; p < NP; ++p) put(rows + p * rstride, tid + N * r, flags[r], L[r][p]);
        }
      }
      if (tid < w) {
#pragma unroll
        for (int p = 0; p < NP; ++p) lmin[p * wpad + tid] = 0xFFFFU;
      }
      prepare(info + i1 * wpad, cinfo, nK, false);
      lds_barrier();
      const int t0 = i2;
      i2 = i0;
      i0 = i1;
      i1 = t0;
      first = nfirst;
      next = after;
      K = nK;
    }
  }
}

// ------------------------------------------------------------------ partial sums
// Sum of the path-cost slices of scans that ran side by side (uint16
// wrap-around, so the grouping of the 8 paths does not matter).
__global__ __launch_bounds__(256) void k_sum_u16(std::uint16_t* __restrict__ dst, SumSrc src, std::uint64_t n8) {
  const std::uint64_t i = std::uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n8) return;
  uint4 acc = reinterpret_cast<const uint4*>(src.p[0])[i];
  for (int k = 1; k < src.n; ++k) {
    const uint4 v = reinterpret_cast<const uint4*>(src.p[k])[i];
    acc.x = as_u32(as_pair(acc.x) + as_pair(v.x));
    acc.y = as_u32(as_pair(acc.y) + as_pair(v.y));
    acc.z = as_u32(as_pair(acc.z) + as_pair(v.z));
    acc.w = as_u32(as_pair(acc.w) + as_pair(v.w));
  }
  reinterpret_cast<uint4*>(dst)[i] = acc;
}

// ------------------------------------------------------------------ selection
__device__ __forceinline__ float subpixel_offset(int method, float sm, float s0, float sp) {
  float delta = 0.0F;
  if (method == 1) {
    const float denom = sm - 2.0F * s0 + sp;
    delta = denom > 0.0F ? (sm - sp) / (2.0F * denom) : 0.0F;
  } else if (method == 2) {
    const float a = sm - s0, b = sp - s0;
    const float slope = a < b ? b : a;
    delta = slope > 0.0F ? (sm - sp) / (2.0F * slope) : 0.0F;
  }
  return delta < -0.5F ? -0.5F : (0.5F < delta ? 0.5F : delta);
}

// Minimum of (value << 16 | label) over the 16 packed values of a chunk whose
// first label is k0: the lowest value, the first label on ties.
__device__ __forceinline__ std::uint32_t chunk_key(const std::uint32_t (&V)[8], std::uint32_t k0) {
  std::uint32_t m = 0xFFFFFFFFU;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    m = min(m, (V[j] << 16) | (k0 + 2U * j));
    m = min(m, (V[j] & 0xFFFF0000U) | (k0 + 2U * j + 1U));
  }
  return m;
}

// select_disparities (stereo_matcher.cpp:446-525): the winner-takes-all
// (sgm_kernels.cpp:405-426) of one tile row (of kSelPx columns of it) per
// block.  A thread takes chunks (16 labels of a pixel) of the row, whatever
// pixel they belong to, and keeps their summed costs in registers: first the
// chunks' best (cost, label) keys meet in LDS, then each chunk gives its best
// cost outside the winner's neighbours and, where it holds them, the costs
// next to the winner; last a thread per pixel fits and checks.  Chunks past
// the kSelHeld a thread keeps are summed again for the second step.
//
// HBM-bound: the chunk's slices or planes once, 12 bytes per pixel (5.5 TB/s at
// 24 MP).  With a quad of lanes per pixel, 8 labels a lane, half
// the lanes idled on pixels of 16 labels: selection of 1024x768 with 128
// labels 1.17 ms, 0.69 ms here; of the 24 MP pair, whose paths then were eight
// uint16 slices, 5.75 and 5.38 ms, 4.07 with bytes and sums of three paths.
constexpr int kSelThreads = 256, kSelPx = 1024, kSelHeld = 4;
template <bool kBytes>
__global__ __launch_bounds__(kSelThreads) void k_select(const JobDesc* __restrict__ jobs,
                                                const TileDesc* __restrict__ tiles,
                                                const std::uint64_t* __restrict__ row_prefix, int ntiles,
                                                const std::uint32_t* __restrict__ rowbase,
                                                const std::uint64_t* __restrict__ pix,
                                                const std::uint32_t* __restrict__ cmap, SumSrc S, SelectParams p,
                                                float* __restrict__ tdisp, float* __restrict__ tconf,
                                                std::int16_t* __restrict__ tlab) {
  __shared__ std::uint32_t best[kSelPx], second[kSelPx];
  __shared__ std::uint16_t below[kSelPx], above[kSelPx];  // costs next to the winner
  extern __shared__ std::uint32_t keys[];
  const std::uint64_t r = blockIdx.x;
  const int t = find_tile_wave(row_prefix, ntiles, r);
  const TileDesc T = tiles[t];
  const int x0 = static_cast<int>(blockIdx.y) * kSelPx, x1 = min(x0 + kSelPx, T.w);
  if (x0 >= T.w) return;
  const JobDesc& J = jobs[T.job];
  const int y = static_cast<int>(r - row_prefix[t]);
  const int Y = T.y0 + y, tid = static_cast<int>(threadIdx.x);
  const auto rows = gptr(J.rows4) + 4 * Y;
  const int lf = rows[0], ll = rows[1], rf = rows[2], rl = rows[3];
  const int xb = min(max(lf - T.x0, 0), T.w);
  const int xe = min(max(ll + 1 - T.x0, xb), T.w);
  // A block's columns lie in one strip; the diagonal check's keys hold tiles of one.
  static_assert((1 << kStripShift) % kSelPx == 0);
  const int strip = x0 >> kStripShift, xs = x0 - (strip << kStripShift);  // the strip's column of x0
  const std::uint64_t row_cell = T.cell_base + rowbase[T.row_base + static_cast<std::uint32_t>(y * T.strips + strip)];
  const std::uint64_t px = T.px_base + std::uint64_t(y) * T.w;
  const bool split = T.cell_base < S.xcells;  // a slice or plane per path
  const int slices = split ? kPaths : S.n;
  const int D = J.D;
  const std::uint32_t* rmap = cmap + row_cell / kLabelAlign;
  // Chunks of the block's columns.
  const std::uint64_t rec0 = pix[px + x0], rec1 = pix[px + x1 - 1];
  const int ka = static_cast<int>(pix_off(rec0) / kLabelAlign);
  const int kb = static_cast<int>((pix_off(rec1) + pix_num(rec1)) / kLabelAlign);

  // Aggregated costs of chunk k.  With planes a path's bytes are M = L - C:
  // 8 C and the eight planes' sum, or 2 C, the horizontal paths' planes and
  // the sweeps' slices; else the sum of the slices.
  auto load = [&](int k, std::uint32_t (&V)[8]) __attribute__((always_inline)) {
    const std::uint64_t cell = row_cell + 16 * std::uint64_t(k);
    auto add_slice = [&](const std::uint16_t* q) __attribute__((always_inline)) {
      const u32x4* b = reinterpret_cast<const u32x4*>(q + cell);
      const u32x4 bl = b[0], bh = b[1];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        V[j] = as_u32(as_pair(V[j]) + as_pair(bl[j]));
        V[j + 4] = as_u32(as_pair(V[j + 4]) + as_pair(bh[j]));
      }
    };
    if constexpr (kBytes) {
      // Sum of n planes and n C: even and odd labels as packed 16-bit sums (at
      // most 16 x 255).
      auto planes = [&](auto Nc) __attribute__((always_inline)) {
        constexpr int n = decltype(Nc)::value;
        u32x4 v[n + 1];
#pragma unroll
        for (int i = 0; i < n; ++i) {
          const std::uint8_t* q = i < 2 ? S.m + i * S.mstride : S.mx + (i - 2) * S.mxstride;
          v[i] = *reinterpret_cast<const u32x4*>(q + cell);
        }
        v[n] = *reinterpret_cast<const u32x4*>(S.c + cell);
        constexpr int kShift = n == 8 ? 3 : 1;
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          std::uint32_t even = (v[n][h] & 0x00FF00FFU) << kShift, odd = ((v[n][h] >> 8) & 0x00FF00FFU) << kShift;
#pragma unroll
          for (int i = 0; i < n; ++i) {
            even += v[i][h] & 0x00FF00FFU;
            odd += (v[i][h] >> 8) & 0x00FF00FFU;
          }
          V[2 * h] = __builtin_amdgcn_perm(odd, even, 0x05040100U);
          V[2 * h + 1] = __builtin_amdgcn_perm(odd, even, 0x07060302U);
        }
      };
      if (split) {
        planes(std::integral_constant<int, kPaths>{});
      } else {
        planes(std::integral_constant<int, 2>{});
        add_slice(S.p[0]);
        add_slice(S.p[1]);
      }
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) V[j] = 0;
      for (int i = 0; i < slices; ++i) add_slice(S.p[i]);
    }
  };

  for (int i = tid; i < x1 - x0; i += kSelThreads) {
    best[i] = 0xFFFFFFFFU;
    second[i] = 0xFFFFU;
  }
  if (p.diagonal_lr) {
    // Right-image WTA along x - label (sgm_kernels.cpp:427-435): the first
    // (in x order) minimum of each diagonal, as a (cost, x) key minimum.
    for (int i = tid; i < T.w + D; i += kSelThreads) keys[i] = 0xFFFFFFFFU;
    __syncthreads();
    const std::uint64_t recl = pix[px + T.w - 1];
    const int kn = static_cast<int>((pix_off(recl) + pix_num(recl)) / kLabelAlign);
    for (int k = tid; k < kn; k += kSelThreads) {
      const std::uint32_t m = rmap[k];
      const int x = map_col(m);
      if (x < xb || x >= xe) continue;
      std::uint32_t V[8];
      load(k, V);
      const int d0 = x - pix_lo(pix[px + x]) - kLabelAlign * map_place(m) + D - 1;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        atomicMin(&keys[d0 - 2 * j], (V[j] << 16) | static_cast<std::uint32_t>(x));
        atomicMin(&keys[d0 - 2 * j - 1], (V[j] & 0xFFFF0000U) | static_cast<std::uint32_t>(x));
      }
    }
  }
  __syncthreads();

  std::uint32_t V[kSelHeld][8], m[kSelHeld];
#pragma unroll
  for (int i = 0; i < kSelHeld; ++i) {
    const int k = ka + tid + kSelThreads * i;
    m[i] = k < kb ? rmap[k] : 0U;
  }
#pragma unroll
  for (int i = 0; i < kSelHeld; ++i) {
    const int k = ka + tid + kSelThreads * i;
    if (k < kb) {
      load(k, V[i]);
      atomicMin(&best[map_col(m[i]) - xs], chunk_key(V[i], static_cast<std::uint32_t>(map_place(m[i]) * kLabelAlign)));
    }
  }
  for (int k = ka + tid + kSelThreads * kSelHeld; k < kb; k += kSelThreads) {
    std::uint32_t X[8];
    const std::uint32_t mm = rmap[k];
    load(k, X);
    atomicMin(&best[map_col(mm) - xs], chunk_key(X, static_cast<std::uint32_t>(map_place(mm) * kLabelAlign)));
  }
  __syncthreads();
  // Best cost of a chunk outside the winner and its neighbours (labels w - 1
  // .. w + 1, halves a .. a + 2 of the chunk: words a / 2 and a / 2 + 1).
  auto outside = [&](std::uint32_t mm, const std::uint32_t (&X)[8]) __attribute__((always_inline)) {
    const int x = map_col(mm) - xs;
    const int a = static_cast<int>(best[x] & 0xFFFFU) - 1 - map_place(mm) * kLabelAlign, j0 = a >> 1;
    std::uint32_t w0 = 0xFFFFFFFFU, w1 = 0xFFFFFFFFU, lowest = 0xFFFFFFFFU;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const bool e0 = j == j0, e1 = j == j0 + 1;
      w0 = e0 ? X[j] : w0;
      w1 = e1 ? X[j] : w1;
      lowest = as_u32(__builtin_elementwise_min(as_pair(lowest), as_pair(e0 || e1 ? 0xFFFFFFFFU : X[j])));
    }
    const bool odd = (a & 1) != 0;
    // Costs at w - 1 and w + 1 where this chunk holds them.
    if (j0 >= 0 && j0 < 8) below[x] = static_cast<std::uint16_t>(odd ? w0 >> 16 : w0);
    if (j0 + 1 >= 0 && j0 + 1 < 8) above[x] = static_cast<std::uint16_t>(odd ? w1 >> 16 : w1);
    lowest = as_u32(__builtin_elementwise_min(as_pair(lowest), as_pair(w0 | (odd ? 0xFFFF0000U : 0xFFFFFFFFU))));
    lowest = as_u32(__builtin_elementwise_min(as_pair(lowest), as_pair(w1 | (odd ? 0xFFFFFFFFU : 0x0000FFFFU))));
    atomicMin(&second[x], min(lowest & 0xFFFFU, lowest >> 16));
  };
#pragma unroll
  for (int i = 0; i < kSelHeld; ++i) {
    if (ka + tid + kSelThreads * i < kb) outside(m[i], V[i]);
  }
  for (int k = ka + tid + kSelThreads * kSelHeld; k < kb; k += kSelThreads) {
    std::uint32_t X[8];
    load(k, X);
    outside(rmap[k], X);
  }
  __syncthreads();

  for (int x = x0 + tid; x < x1; x += kSelThreads) {
    float d = kInf, conf = 0.0F;
    std::int16_t lab = INT16_MIN;
    if (x >= xb && x < xe) {
      const std::uint64_t rec = pix[px + x];
      const int lo = pix_lo(rec), n = pix_num(rec);
      const std::uint32_t key = best[x - x0], sec = second[x - x0], bcost = key >> 16;
      const int j = static_cast<int>(key & 0xFFFFU), label = lo + j;
      const int xr = T.x0 + x - J.dmin - label;
      bool ok = !(xr < rf || xr > rl);
      if (ok && ((j == 0 && lo > 0) || (j == n - 1 && lo + n < D))) ok = false;
      if (ok && p.diagonal_lr) {
        const std::uint32_t rkey = keys[x - label + D - 1];
        const int rbest = static_cast<int>(rkey & 0xFFFFU) - (x - label);
        if (abs(rbest - label) > p.lr_max_diff) ok = false;
      }
      const float best_cost = static_cast<float>(bcost);
      if (ok && p.uniqueness > 0.0F && sec != 0xFFFFU && best_cost > (1.0F - p.uniqueness) * static_cast<float>(sec))
        ok = false;
      if (ok) {
        float delta = 0.0F;
        if (j > 0 && j < n - 1)
          delta = subpixel_offset(p.subpixel, static_cast<float>(below[x - x0]), best_cost,
                                  static_cast<float>(above[x - x0]));
        d = static_cast<float>(J.dmin + label) + delta;
        conf = sec != 0xFFFFU && sec > 0 ? 1.0F - best_cost / static_cast<float>(sec) : 0.0F;
        lab = static_cast<std::int16_t>(J.dmin + label);
      }
    }
    tdisp[px + x] = d;
    if (J.confidence) tconf[px + x] = conf;
    if (tlab != nullptr) tlab[px + x] = lab;
  }
}

// ------------------------------------------------------------------ blending
// axis_weight (stereo_matcher.cpp:530-543).
__device__ __forceinline__ float axis_weight(int v, int c0, int c1, int size, int blend_px) {
  const float blend = static_cast<float>(blend_px);
  float w = 1.0F;
  const float pos = static_cast<float>(v) + 0.5F;
  auto clamp01 = [](float a) { return a < 0.0F ? 0.0F : (1.0F < a ? 1.0F : a); };
  if (c0 > 0) {
    const float a = blend_px > 0 ? clamp01((pos - static_cast<float>(c0) + 0.5F * blend) / blend) : (v >= c0 ? 1.0F : 0.0F);
    w = a < w ? a : w;
  }
  if (c1 < size) {
    const float a = blend_px > 0 ? clamp01((static_cast<float>(c1) + 0.5F * blend - pos) / blend) : (v < c1 ? 1.0F : 0.0F);
    w = a < w ? a : w;
  }
  return w;
}

// First grid index whose extent end exceeds v (extents sorted by start and
// end); e(k) is extent k's end.
template <typename E>
__device__ __forceinline__ int first_covering(E e, int n, int v) {
  int lo = 0, hi = n;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (e(mid) > v) {
      hi = mid;
    } else {
      lo = mid + 1;
    }
  }
  return lo;
}

// Blend of one job's tiles (stereo_matcher.cpp:688-766): per pixel, the tiles
// that cover it in tile-index order, the same float operations as the
// reference (weighted mean if the valid weight is at least half of the total,
// the dominant tile's value if the mean is more than 1 away from it).  The
// block copies the grid's extents into LDS first (grids of at most kGrid
// tiles per axis), so a pixel's searches wait on one coalesced load.
__global__ __launch_bounds__(256) void k_blend(GridDesc g, const TileDesc* __restrict__ tiles,
                                               const float* __restrict__ tdisp, const float* __restrict__ tconf,
                                               const std::int16_t* __restrict__ tlab, float* __restrict__ disp,
                                               float* __restrict__ conf, std::int16_t* __restrict__ lab) {
  constexpr int kGrid = 256;
  __shared__ std::int32_t scols[4 * kGrid], srows[4 * kGrid];
  const bool staged = g.nx <= kGrid && g.ny <= kGrid;
  if (staged) {
    const auto gc = gptr(g.cols), gr = gptr(g.rows);
    for (int k = threadIdx.x; k < 4 * g.nx; k += blockDim.x) scols[k] = gc[k];
    for (int k = threadIdx.x; k < 4 * g.ny; k += blockDim.x) srows[k] = gr[k];
  }
  __syncthreads();
  const int X = blockIdx.x * blockDim.x + threadIdx.x, Y = blockIdx.y;
  if (X >= g.width) return;
  float wall = 0.0F, wsum = 0.0F, dsum = 0.0F, csum = 0.0F, wbest = 0.0F, dbest = kInf;
  std::int16_t lbest = INT16_MIN;
  // cols(i, k) / rows(j, k): entry k of extent i / j.
  auto blend = [&](auto cols, auto rows) {
    const int j0 = first_covering([&](int k) { return rows(k, 1); }, g.ny, Y);
    const int i0 = first_covering([&](int k) { return cols(k, 1); }, g.nx, X);
    for (int j = j0; j < g.ny && rows(j, 0) <= Y; ++j) {
      const float wy = axis_weight(Y, rows(j, 2), rows(j, 3), g.height, g.blend);
      if (wy <= 0.0F) continue;
      for (int i = i0; i < g.nx && cols(i, 0) <= X; ++i) {
        const float wgt = wy * axis_weight(X, cols(i, 2), cols(i, 3), g.width, g.blend);
        if (wgt <= 0.0F) continue;
        const TileDesc& T = tiles[g.tile_base + j * g.nx + i];
        const std::uint64_t ti = T.px_base + std::uint64_t(Y - T.y0) * T.w + (X - T.x0);
        wall += wgt;
        const float dv = tdisp[ti];
        if (__builtin_isfinite(dv)) {
          wsum += wgt;
          dsum += wgt * dv;
          if (conf != nullptr) csum += wgt * tconf[ti];
          if (wgt > wbest) {
            wbest = wgt;
            dbest = dv;
            if (lab != nullptr) lbest = tlab[ti];
          }
        }
      }
    }
  };
  if (staged) {
    blend([&](int i, int k) { return scols[4 * i + k]; }, [&](int j, int k) { return srows[4 * j + k]; });
  } else {
    const auto gc = gptr(g.cols), gr = gptr(g.rows);
    blend([&](int i, int k) { return gc[4 * i + k]; }, [&](int j, int k) { return gr[4 * j + k]; });
  }
  float dv = kInf;
  float cv = 0.0F;
  std::int16_t lv = INT16_MIN;
  if (wsum > 0.0F && wsum >= 0.5F * wall) {
    dv = dsum / wsum;
    if (fabsf(dv - dbest) > 1.0F) dv = dbest;
    cv = csum / wsum;
    lv = lbest;
  }
  const std::int64_t o = std::int64_t(Y) * g.width + X;
  disp[o] = dv;
  if (conf != nullptr) conf[o] = cv;
  if (lab != nullptr) lab[o] = lv;
}

__global__ void k_pack_rows(const std::int32_t* __restrict__ base, const std::int32_t* __restrict__ partner, int h,
                            std::int32_t* __restrict__ rows4) {
  const int y = blockIdx.x * blockDim.x + threadIdx.x;
  if (y >= h) return;
  reinterpret_cast<int4*>(rows4)[y] = make_int4(base[2 * y], base[2 * y + 1], partner[2 * y], partner[2 * y + 1]);
}

// Blocks of a kernel that fit on the device at once.
template <typename K>
std::uint64_t resident_blocks(K kernel) {
  int dev = 0, cus = 0, per_cu = 0;
  (void)hipGetDevice(&dev);
  (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, 64 * kWaves, 0);
  return std::uint64_t(std::max(cus, 1)) * std::uint64_t(std::max(per_cu, 1));
}

template <int DX, int DY, int MODE>
std::uint64_t path_blocks() {
  static const std::uint64_t n = resident_blocks(k_path<DX, DY, MODE>);
  return n;
}

template <int DX, int DY, int MODE>
void path_launch(const PathArgs& a, hipStream_t s) {
  // Persistent waves: at most `slots` (scratch rows), at most one per group.
  const std::uint64_t waves = std::min(a.groups, a.slots);
  const std::uint64_t blocks = std::min((waves + kWaves - 1) / kWaves, path_blocks<DX, DY, MODE>());
  k_path<DX, DY, MODE><<<dim3(static_cast<unsigned>(blocks)), 64 * kWaves, 0, s>>>(
      a.jobs, a.tiles, a.gprefix, a.ntiles, a.groups, a.rowbase, a.pix, a.C, a.out, a.scratch, path_scratch_row(a.max_num),
      a.queue);
}

template <int DX, int DY>
void path_launch(const PathArgs& a, int mode, hipStream_t s) {
  if constexpr (DY == 0) {
    if (mode == kByteM) {
      path_launch<DX, DY, kByteM>(a, s);
      return;
    }
  }
  if (mode == kAddSum) {
    path_launch<DX, DY, kAddSum>(a, s);
  } else {
    path_launch<DX, DY, kFirstSum>(a, s);
  }
}

}  // namespace

void launch_tile_row_scan(const JobDesc* jobs, const TileDesc* tiles, const std::uint64_t* row_prefix, int ntiles,
                          std::uint64_t total_rows, std::uint64_t* pix, std::uint64_t* row_cells,
                          std::uint32_t* row_max, hipStream_t s) {
  if (total_rows == 0) return;
  k_tile_row_scan<<<dim3(static_cast<unsigned>((total_rows + 3) / 4)), 256, 0, s>>>(jobs, tiles, row_prefix, ntiles,
                                                                                    total_rows, pix, row_cells, row_max);
}

void launch_tile_cells(const TileDesc* tiles, int ntiles, const std::uint64_t* row_cells, const std::uint32_t* row_max,
                       std::uint32_t* rowbase, std::uint64_t* tile_cells, std::uint32_t* tile_max,
                       std::uint32_t* tile_row, hipStream_t s) {
  k_tile_cells<<<dim3(ntiles), kCellsThreads, 0, s>>>(tiles, row_cells, row_max, rowbase, tile_cells, tile_max, tile_row);
}

void launch_cost(const JobDesc* jobs, const TileDesc* tiles, const std::uint64_t* row_prefix, int ntiles,
                 std::uint64_t total_rows, const std::uint32_t* rowbase, const std::uint64_t* pix, std::uint8_t* C,
                 std::uint32_t* cmap, hipStream_t s) {
  if (total_rows == 0) return;
  k_cost<<<dim3(static_cast<unsigned>(total_rows)), kCostThreads, 0, s>>>(jobs, tiles, row_prefix, ntiles, rowbase, pix,
                                                                         C, cmap);
}

int path_scratch_row(int max_num) { return kPad + (max_num + 15) / 16 * 16 + kPad; }

std::uint64_t path_slots() {
  std::uint64_t b = path_blocks<1, 0, kAddSum>();
  b = std::max(b, path_blocks<1, 0, kFirstSum>());
  b = std::max(b, path_blocks<1, 0, kByteM>());
  b = std::max(b, path_blocks<0, 1, kAddSum>());
  b = std::max(b, path_blocks<1, 1, kAddSum>());
  b = std::max(b, path_blocks<-1, 1, kAddSum>());
  return b * kWaves;
}

std::size_t path_scratch_elems(std::uint64_t slots, int max_num) {
  return std::size_t(slots) * kScanPerWave * 2 * std::size_t(path_scratch_row(max_num));
}

void launch_sgm_path(int path, const PathArgs& a, int mode, hipStream_t s) {
  if (a.groups == 0) return;
  switch (path) {
    case 0: path_launch<1, 0>(a, mode, s); break;
    case 1: path_launch<-1, 0>(a, mode, s); break;
    case 2: path_launch<0, 1>(a, mode, s); break;
    case 3: path_launch<0, -1>(a, mode, s); break;
    case 4: path_launch<1, 1>(a, mode, s); break;
    case 5: path_launch<-1, -1>(a, mode, s); break;
    case 6: path_launch<-1, 1>(a, mode, s); break;
    default: path_launch<1, -1>(a, mode, s); break;
  }
}

// Four labels a lane where the launch then still has at most 1.5 waves per
// SIMD: there a step's chain is all that counts (384 x 288 with 64 labels: 75 us
// against 85 with eight, 127 with sixteen).  Eight otherwise: with more waves the
// shorter steps of four no longer pay for the instructions they repeat
// (640 x 480 with 64 labels: 172 us against 146, sixteen 176).
FullSplit full_split(int D, std::uint64_t scanlines) {
  auto lanes = [&](int labels) {
    int n = 2;
    while (n * labels < D) n *= 2;
    return n;
  };
  int dev = 0, cus = 0;
  (void)hipGetDevice(&dev);
  (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  const std::uint64_t waves = (scanlines * std::uint64_t(lanes(4)) + 63) / 64;
  if (lanes(4) <= 32 && waves <= std::uint64_t(6 * std::max(cus, 1))) return {4, lanes(4)};
  return {8, lanes(8)};
}

void launch_full(const FullArgs& a, FullSplit f, hipStream_t s) {
  if (a.groups == 0) return;
  const dim3 grid(static_cast<unsigned>((a.groups + kWaves - 1) / kWaves));
  switch (f.labels * 64 + f.lanes) {
    case 4 * 64 + 4: k_full<4, 4><<<grid, 64 * kWaves, 0, s>>>(a); break;
    case 4 * 64 + 8: k_full<8, 4><<<grid, 64 * kWaves, 0, s>>>(a); break;
    case 4 * 64 + 16: k_full<16, 4><<<grid, 64 * kWaves, 0, s>>>(a); break;
    case 4 * 64 + 32: k_full<32, 4><<<grid, 64 * kWaves, 0, s>>>(a); break;
    case 8 * 64 + 2: k_full<2, 8><<<grid, 64 * kWaves, 0, s>>>(a); break;
    case 8 * 64 + 4: k_full<4, 8><<<grid, 64 * kWaves, 0, s>>>(a); break;
    case 8 * 64 + 8: k_full<8, 8><<<grid, 64 * kWaves, 0, s>>>(a); break;
    case 8 * 64 + 16: k_full<16, 8><<<grid, 64 * kWaves, 0, s>>>(a); break;
    case 8 * 64 + 32: k_full<32, 8><<<grid, 64 * kWaves, 0, s>>>(a); break;
    default: k_full<64, 8><<<grid, 64 * kWaves, 0, s>>>(a); break;
  }
}

int compute_units() {
  int dev = 0, cus = 0;
  (void)hipGetDevice(&dev);
  (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  return cus;
}

SweepPlan sweep_plan(int np, int max_w, std::uint32_t max_chunks, std::uint64_t mean_chunks) {
  int dev = 0, lds = 0;
  (void)hipGetDevice(&dev);
  (void)hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev);
  return size_sweep(np, max_w, max_chunks, mean_chunks, compute_units(), lds);
}

namespace {
template <int NP, bool kByte, int H>
void sweep_launch(const SweepArgs& a, const SweepPlan& p, std::uint64_t blocks, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(std::min<std::uint64_t>(a.units, blocks)));
  // Dynamic LDS past 64 KB has to be asked for (a failure is the launch's).
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(&k_sweep<NP, kByte, H>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, p.lds_bytes) != hipSuccess)
    return;
  k_sweep<NP, kByte, H><<<grid, kSweepThreads, p.lds_bytes, s>>>(a);
}
}  // namespace

void launch_sweep(const SweepArgs& a, int np, bool bytes, const SweepPlan& p, std::uint64_t blocks, hipStream_t s) {
  if (a.units == 0) return;
  if (np == 3) {
    sweep_launch<3, false, 2>(a, p, blocks, s);
  } else if (bytes) {
    p.held == 2 ? sweep_launch<1, true, 2>(a, p, blocks, s) : sweep_launch<1, true, 4>(a, p, blocks, s);
  } else {
    p.held == 2 ? sweep_launch<1, false, 2>(a, p, blocks, s) : sweep_launch<1, false, 4>(a, p, blocks, s);
  }
}

void launch_select(const JobDesc* jobs, const TileDesc* tiles, const std::uint64_t* row_prefix, int ntiles,
                   std::uint64_t total_rows, const std::uint32_t* rowbase, const std::uint64_t* pix,
                   const std::uint32_t* cmap, const SumSrc& src, SelectParams p, int max_w, int max_D, float* tdisp, float* tconf, std::int16_t* tlab,
                   hipStream_t s) {
  if (total_rows == 0) return;
  const std::size_t lds = p.diagonal_lr ? std::size_t(max_w + max_D) * sizeof(std::uint32_t) : 0;
  const dim3 grid(static_cast<unsigned>(total_rows), static_cast<unsigned>((max_w + kSelPx - 1) / kSelPx));
  if (src.m != nullptr) {
    k_select<true><<<grid, kSelThreads, lds, s>>>(jobs, tiles, row_prefix, ntiles, rowbase, pix, cmap, src, p, tdisp,
                                                  tconf, tlab);
  } else {
    k_select<false><<<grid, kSelThreads, lds, s>>>(jobs, tiles, row_prefix, ntiles, rowbase, pix, cmap, src, p, tdisp,
                                                   tconf, tlab);
  }
}

void launch_sum_u16(std::uint16_t* dst, const SumSrc& src, std::uint64_t n, hipStream_t s) {
  const std::uint64_t n8 = (n + 7) / 8;
  if (n8 == 0 || src.n <= 0) return;
  k_sum_u16<<<dim3(static_cast<unsigned>((n8 + 255) / 256)), 256, 0, s>>>(dst, src, n8);
}

void launch_pack_rows(const std::int32_t* base, const std::int32_t* partner, int h, std::int32_t* rows4,
                      hipStream_t s) {
  k_pack_rows<<<dim3((h + 255) / 256), 256, 0, s>>>(base, partner, h, rows4);
}

void launch_blend(GridDesc g, const TileDesc* tiles, const float* tdisp, const float* tconf, const std::int16_t* tlab,
                  float* disp, float* conf, std::int16_t* lab, hipStream_t s) {
  k_blend<<<dim3((g.width + 255) / 256, g.height), 256, 0, s>>>(g, tiles, tdisp, tconf, tlab, disp, conf, lab);
}

}  // namespace r3dg
