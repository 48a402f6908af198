// Tile lists of a small scene without a sort of its intersections, without
// sizes read back by the host, in two launches:
//
//  1. rank: every Gaussian counts the depth keys before its own (ties by
//     index), so the packed rectangles are written in depth order.  n^2 / 64
//     wave comparisons of two VALU instructions: 17 us for 10k Gaussians, 45 us
//     for 20k, where the four passes of the depth sort take 33 and 40 and five
//     launches.
//  2. lists: a workgroup takes four neighbouring tiles of one tile row, tests
//     every rectangle in depth order against them (a ballot per 64 Gaussians
//     and tile) and writes each tile's hits at the tile's own n slots.
//
// The row/column bucketing of tile_bin.hip does the same in 15 launches of 2 to
// 17 us, each a short dependent chain at this size, and has the host wait for
// its totals in between; it reads every rectangle a few times where this one
// reads it once per four tiles, so this one is for few Gaussians on few tiles
// (small_fits).  Lists kernel: 12 us for 10k Gaussians on 256 or 1200 tiles.
// Frames of 10k Gaussians at 256 x 256 and 640 x 480: 178 -> 69 and 179 -> 79
// us; a step of 20k at 403 x 307: 510 -> 365 us.
//
// List t is gaussian_ids[ranges[t]) in [t n, (t + 1) n): lists do not touch one
// another, and follow one another in tile order as the compositing kernels'
// hit masks need.  Counts and order are those of the sort by (tile, depth
// bits, index) of intersections.py:10-88.
#include "block_scan.h"
#include "common.h"

namespace gs {
namespace {

constexpr int kStrip = 4;          // tiles per workgroup of the lists kernel
constexpr int kRankWaves = 16;
constexpr int kListWaves = 16;
// 16-bit ids and the strip's masks of this many Gaussians fill 63 KB of LDS.
constexpr int64_t kSmallMax = 24576;
// The lists' slots, n per tile: at most 64 MiB of ids.
constexpr int64_t kSmallSlots = int64_t(1) << 24;

bool small_fits(int64_t n, int64_t tiles) {
  return n > 0 && n <= kSmallMax && tiles > 0 && n * tiles <= kSmallSlots;
}

// Workgroup b ranks Gaussians [64 b, 64 b + 64), one per lane; its waves share
// the keys to compare with, 64 at a time, read as scalars.
__global__ __launch_bounds__(kRankWaves * 64) void rank_kernel(
    const uint32_t* __restrict__ keys, const uint32_t* __restrict__ rects, int n,
    uint32_t* __restrict__ sorted_rects, uint16_t* __restrict__ sorted_ids,
    float* __restrict__ clear, int clear_per_gaussian) {
  __shared__ uint32_t part[kRankWaves][64];
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const int b = blockIdx.x;
  const int i = b * 64 + lane;
  const int blocks = (n + 63) >> 6;
  const uint32_t mine = i < n ? keys[i] : 0xFFFFFFFFu;
  if (clear) {
    const int first = b * 64 * clear_per_gaussian;
    const int last = min(first + 64 * clear_per_gaussian, n * clear_per_gaussian);
    for (int k = first + int(threadIdx.x); k < last; k += kRankWaves * 64) clear[k] = 0.0f;
  }
  const int share = (blocks + kRankWaves - 1) / kRankWaves;
  const int j0 = wid * share, j1 = min(j0 + share, blocks);
  uint32_t before = 0;
  for (int jb = j0; jb < j1; ++jb) {  // wave-uniform
    if (jb == b || jb * 64 + 64 > n) {
      // The workgroup's own Gaussians (a tie comes before the lanes after it)
      // or the last, partial block: the lanes' keys in turn, past the end one
      // that is never before another.
      const int j = jb * 64 + lane;
      const uint32_t theirs = j < n ? keys[j] : 0xFFFFFFFFu;
#pragma unroll 8
      for (int k = 0; k < 64; ++k) {
        const uint32_t key = uint32_t(__builtin_amdgcn_readlane(int(theirs), k));
        const uint64_t ties = jb < b ? ~uint64_t(0) : jb > b ? 0 : ~uint64_t(1) << k;
        const uint64_t m = __builtin_amdgcn_ballot_w64(key < mine) |
                           (__builtin_amdgcn_ballot_w64(key == mine) & ties);
        before += __builtin_amdgcn_inverse_ballot_w64(m) ? 1u : 0u;
      }
      continue;
    }
    const uint32_t* __restrict__ block = keys + jb * 64;
    if (jb < b) {
#pragma unroll
      for (int k = 0; k < 64; ++k) before += block[k] <= mine ? 1u : 0u;
    } else {
#pragma unroll
      for (int k = 0; k < 64; ++k) before += block[k] < mine ? 1u : 0u;
    }
  }
  part[wid][lane] = before;
  __syncthreads();
  if (wid != 0 || i >= n) return;
  uint32_t rank = 0;
#pragma unroll
  for (int w = 0; w < kRankWaves; ++w) rank += part[w][lane];
  if (rank < uint32_t(n)) {  // always: the ranks are a permutation
    sorted_rects[rank] = rects[i];
    sorted_ids[rank] = uint16_t(i);
  }
}

// Workgroup (x, y): tiles x kStrip .. x kStrip + kStrip - 1 of tile row y.
// Dynamic LDS: the strip's masks [kStrip][blocks], then their prefixes
// [kStrip][blocks] (16 bits: below n), then the ids in depth order [n].
__global__ __launch_bounds__(kListWaves * 64) void lists_kernel(
    const uint32_t* __restrict__ sorted_rects, const uint16_t* __restrict__ sorted_ids, int n,
    int tw, int64_t* __restrict__ ranges, int32_t* __restrict__ gaussian_ids) {
  extern __shared__ uint64_t lds[];
  const int blocks = (n + 63) >> 6;
  uint64_t* masks = lds;
  uint16_t* prefix = reinterpret_cast<uint16_t*>(masks + kStrip * blocks);
  uint16_t* ids = prefix + kStrip * blocks;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const uint32_t tx0 = blockIdx.x * kStrip, ty = blockIdx.y;

  // 1. Hits of the strip's tiles, 64 Gaussians per wave and step; the loads of
  // four steps are in flight together.
  constexpr int kBatch = 4;
  for (int b0 = wid; b0 < blocks; b0 += kBatch * kListWaves) {
    uint32_t rect[kBatch];
    uint16_t id[kBatch];
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      const int g = (b0 + i * kListWaves) * 64 + lane;
      rect[i] = g < n ? sorted_rects[g] : kNoRect;
      id[i] = g < n ? sorted_ids[g] : uint16_t(0);
    }
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      const int b = b0 + i * kListWaves;
      if (b >= blocks) break;  // wave-uniform
      const uint32_t r = rect[i];
      const bool row = r != kNoRect && ty - ((r >> 16) & 0xFFu) <= (r >> 24);
      const uint32_t x0 = r & 0xFFu, w1 = (r >> 8) & 0xFFu;
      uint64_t mine = 0;
#pragma unroll
      for (int s = 0; s < kStrip; ++s) {
        const uint64_t m = __builtin_amdgcn_ballot_w64(row && tx0 + s - x0 <= w1);
        mine = lane == s ? m : mine;
      }
      if (lane < kStrip) masks[lane * blocks + b] = mine;
      if (b * 64 + lane < n) ids[b * 64 + lane] = id[i];
    }
  }
  __syncthreads();

  // 2. One wave per tile: the hits before each block, and the tile's range.
  if (wid < kStrip) {
    uint32_t carry = 0;
    for (int b0 = 0; b0 < blocks; b0 += 64) {
      const int b = b0 + lane;
      const uint32_t c = b < blocks ? uint32_t(__popcll(masks[wid * blocks + b])) : 0u;
      const uint32_t inc = carry + wave_inclusive_scan(c);
      if (b < blocks) prefix[wid * blocks + b] = uint16_t(inc - c);
      carry = uint32_t(__builtin_amdgcn_readlane(int(inc), 63));
    }
    const int tx = int(tx0) + wid;
    if (tx < tw && lane == 0) {
      const int64_t t = int64_t(ty) * tw + tx;
      reinterpret_cast<longlong2*>(ranges)[t] = make_longlong2(t * n, t * n + carry);
    }
  }
  __syncthreads();

  // 3. The lists: each tile's waves take chunks of 64 blocks, one block's mask
  // and prefix per lane, and visit the blocks with hits.
  constexpr int kTileWaves = kListWaves / kStrip;
  const int s = wid & (kStrip - 1);
  const int tx = int(tx0) + s;
  if (tx >= tw) return;  // wave-uniform, after the last barrier
  const int64_t t = int64_t(ty) * tw + tx;
  int32_t* list = gaussian_ids + t * n;
  for (int b0 = wid / kStrip * 64; b0 < blocks; b0 += kTileWaves * 64) {
    const int b = b0 + lane;
    const uint64_t m = b < blocks ? masks[s * blocks + b] : 0;
    const uint32_t first = b < blocks ? prefix[s * blocks + b] : 0u;
    uint64_t hits = __builtin_amdgcn_ballot_w64(m != 0);
    while (hits) {
      const int k = __builtin_ctzll(hits);
      hits &= hits - 1;
      const uint64_t mk = uint64_t(uint32_t(__builtin_amdgcn_readlane(int(uint32_t(m)), k))) |
                          uint64_t(uint32_t(__builtin_amdgcn_readlane(int(m >> 32), k))) << 32;
      const int at = __builtin_amdgcn_readlane(int(first), k) +
                     int(__builtin_amdgcn_mbcnt_hi(uint32_t(mk >> 32),
                                                   __builtin_amdgcn_mbcnt_lo(uint32_t(mk), 0u)));
      if (__builtin_amdgcn_inverse_ballot_w64(mk)) list[at] = ids[(b0 + k) * 64 + lane];
    }
  }
}

size_t lists_lds(int64_t n) {
  const int64_t blocks = (n + 63) / 64;
  return size_t(kStrip * blocks * 10 + blocks * 64 * 2);
}

}  // namespace
}  // namespace gs

using namespace gs;

extern "C" {

GS_API size_t gs_small_lists_bytes(int64_t n, int32_t tiles_w, int32_t tiles_h) {
  if (tiles_w <= 0 || tiles_h <= 0 || tiles_w > kMaxAxisTiles || tiles_h > kMaxAxisTiles) return 0;
  if (!small_fits(n, int64_t(tiles_w) * tiles_h)) return 0;
  return align_up(size_t(n) * 4) + align_up(size_t(n) * 2);
}

GS_API int gs_small_lists(const uint32_t* depth_keys, const uint32_t* tile_rects, int64_t n,
                          int32_t tiles_w, int32_t tiles_h, int64_t* ranges,
                          int32_t* gaussian_ids, int64_t num_ids, void* workspace,
                          size_t workspace_bytes, float* clear, int32_t clear_per_gaussian,
                          void* stream) {
  clear_error();
  const size_t need = gs_small_lists_bytes(n, tiles_w, tiles_h);
  GS_REQUIRE(need > 0, GS_ERR_UNSUPPORTED,
             "small lists need at most %lld Gaussians and %lld list slots (got %lld on %d x %d "
             "tiles)",
             (long long)kSmallMax, (long long)kSmallSlots, (long long)n, tiles_w, tiles_h);
  GS_REQUIRE(depth_keys && tile_rects && ranges && gaussian_ids && workspace,
             GS_ERR_INVALID_ARGUMENT, "null pointer argument");
  GS_REQUIRE((reinterpret_cast<uintptr_t>(ranges) & 15u) == 0 &&
                 (reinterpret_cast<uintptr_t>(workspace) & 15u) == 0,
             GS_ERR_INVALID_ARGUMENT, "ranges and workspace must be 16-byte aligned");
  GS_REQUIRE(workspace_bytes >= need, GS_ERR_WORKSPACE,
             "workspace too small (%zu bytes, need %zu)", workspace_bytes, need);
  GS_REQUIRE(num_ids >= n * tiles_w * tiles_h, GS_ERR_WORKSPACE,
             "list buffer too small (%lld ids, need %lld)", (long long)num_ids,
             (long long)(n * tiles_w * tiles_h));
  GS_REQUIRE(clear_per_gaussian >= 0 && clear_per_gaussian <= 64, GS_ERR_INVALID_ARGUMENT,
             "invalid clear size %d", clear_per_gaussian);
  hipStream_t s = as_stream(stream);
  uint32_t* rects = static_cast<uint32_t*>(workspace);
  uint16_t* ids =
      reinterpret_cast<uint16_t*>(static_cast<char*>(workspace) + align_up(size_t(n) * 4));
  rank_kernel<<<unsigned(ceil_div(n, 64)), kRankWaves * 64, 0, s>>>(
      depth_keys, tile_rects, int(n), rects, ids, clear, clear_per_gaussian);
  GS_TRY(check_launch("small_lists rank"));
  const dim3 grid(unsigned(ceil_div(tiles_w, kStrip)), unsigned(tiles_h));
  lists_kernel<<<grid, kListWaves * 64, unsigned(lists_lds(n)), s>>>(rects, ids, int(n), tiles_w,
                                                                     ranges, gaussian_ids);
  return check_launch("small_lists");
}

}  // extern "C"
