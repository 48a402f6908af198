// Tile lists of a small scene without a sort of its intersections, without
// sizes read back by the host, in three launches:
//
//  1. order: chunks of 256 depth keys are sorted (each key counts those of its
//     chunk before it), then every Gaussian's rank is its place in its chunk
//     plus a binary search in each other chunk (ties by index), and the packed
//     rectangles are written in depth order.  Two launches whose chains are a
//     few LDS reads long: 4.4 + 4.5 us for 10k Gaussians, 4.4 + 8.3 for 20k.
//     Counting all n keys for each Gaussian took 17.4 and 46.9 us (n^2 / 64
//     wave comparisons of two VALU instructions), the four passes of the depth
//     sort take 33 and 40 us and five launches.
//  2. lists: a workgroup takes up to four neighbouring tiles of one tile row,
//     tests every rectangle in depth order against them (a ballot per 64 Gaussians
//     and tile) and writes each tile's hits at the tile's own n slots.
//
// The row/column bucketing of tile_bin.hip does the same in 15 launches of 2 to
// 17 us, each a short dependent chain at this size, and has the host wait for
// its totals in between; it reads every rectangle a few times where this one
// reads it once per one to four tiles, so this one is for few Gaussians on few
// tiles (small_fits).
// Frames of 10k Gaussians at 256 x 256 and 640 x 480: 178 -> 46 and 179 -> 61
// us.
//
// List t is gaussian_ids[ranges[t]) in [t n, (t + 1) n): lists do not touch one
// another, and follow one another in tile order as the compositing kernels'
// hit masks need.  Counts and order are those of the sort by (tile, depth
// bits, index) of intersections.py:10-88.
#include "block_scan.h"
#include "common.h"

namespace gs {
namespace {

// Tiles per workgroup of the lists kernel (its strip): 1, 2 or 4, the least whose
// workgroups are all resident at once, two per CU.  More of them share the
// chip's loads and each tile's list is written by more waves; past that they
// wait for one another and read the rectangles again.  10k Gaussians on 256
// tiles 12.4 us with strips of 4, 6.7 of 1; 20k on 520 tiles 15.5 of 4, 12.0 of
// 2; 10k on 1200 tiles 12.0 of 4.
constexpr int64_t kListGroups = 512;
constexpr int kChunk = 256;        // keys sorted by one workgroup
constexpr int kBlocks = kChunk / 64;
constexpr int kRankWaves = 16;
static_assert(kRankWaves == kBlocks * kBlocks, "chunk_kernel: a wave per pair of blocks");
// Chunks searched from LDS at a time (48 KB, so that two workgroups share a CU).
constexpr int kRoundChunks = 48;
constexpr int kWaveChunks = kRoundChunks / kRankWaves;
constexpr int kListWaves = 16;
// 16-bit ids and the strip's masks of this many Gaussians fill 63 KB of LDS.
constexpr int64_t kSmallMax = 24576;
// The lists' slots, n per tile: at most 64 MiB of ids.
constexpr int64_t kSmallSlots = int64_t(1) << 24;

bool small_fits(int64_t n, int64_t tiles) {
  return n > 0 && n <= kSmallMax && tiles > 0 && n * tiles <= kSmallSlots;
}

// Workgroup c sorts keys [256 c, 256 c + 256) by (key, index), past the end of
// the array by ~0u, which come after all others of the last chunk.  Wave (i, j)
// counts for the 64 keys of block i those of block j before them.
__global__ __launch_bounds__(kRankWaves * 64) void chunk_kernel(
    const uint32_t* __restrict__ keys, int n, uint32_t* __restrict__ chunk_keys,
    uint16_t* __restrict__ chunk_ids) {
  __shared__ __align__(16) uint32_t own[kChunk];
  __shared__ uint32_t part[kBlocks][kChunk];
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const int first = blockIdx.x * kChunk;
  if (threadIdx.x < kChunk) {
    const int g = first + int(threadIdx.x);
    own[threadIdx.x] = g < n ? keys[g] : 0xFFFFFFFFu;
  }
  __syncthreads();
  const int i = wid & (kBlocks - 1), j = wid / kBlocks;
  const uint32_t mine = own[i * 64 + lane];
  const uint4* block = reinterpret_cast<const uint4*>(own + j * 64);
  uint32_t before = 0;
  if (j < i) {
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const uint4 k = block[q];
      before += (k.x <= mine) + (k.y <= mine) + (k.z <= mine) + (k.w <= mine);
    }
  } else if (j > i) {
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const uint4 k = block[q];
      before += (k.x < mine) + (k.y < mine) + (k.z < mine) + (k.w < mine);
    }
  } else {
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const uint4 k = block[q];
      before += (k.x < mine || (k.x == mine && 4 * q + 0 < lane)) +
                (k.y < mine || (k.y == mine && 4 * q + 1 < lane)) +
                (k.z < mine || (k.z == mine && 4 * q + 2 < lane)) +
                (k.w < mine || (k.w == mine && 4 * q + 3 < lane));
    }
  }
  part[j][i * 64 + lane] = before;
  __syncthreads();
  if (threadIdx.x >= kChunk) return;
  uint32_t place = 0;
#pragma unroll
  for (int b = 0; b < kBlocks; ++b) place += part[b][threadIdx.x];
  if (place < uint32_t(kChunk)) {  // always: the places are a permutation
    chunk_keys[first + place] = own[threadIdx.x];
    chunk_ids[first + place] = uint16_t(first + int(threadIdx.x));
  }
}

// Workgroup b ranks the 64 sorted keys [64 b, 64 b + 64) of chunk b / 4, one
// per lane: neighbours in value, so a wave's searches read few different LDS
// words.  Its waves share the chunks to search.
__global__ __launch_bounds__(kRankWaves * 64) void rank_kernel(
    const uint32_t* __restrict__ chunk_keys, const uint16_t* __restrict__ chunk_ids, int chunks,
    const uint32_t* __restrict__ rects, int n, uint32_t* __restrict__ sorted_rects,
    uint16_t* __restrict__ sorted_ids, float* __restrict__ clear, int clear_per_gaussian) {
  __shared__ __align__(16) uint32_t staged[kRoundChunks * kChunk];
  __shared__ uint32_t part[kRankWaves][64];
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const int b = blockIdx.x;
  const int own = b / kBlocks;
  const uint32_t mine = chunk_keys[b * 64 + lane];
  const int id = chunk_ids[b * 64 + lane];
  if (clear) {
    const int first = min(b * 64, n) * clear_per_gaussian;
    const int last = min(b * 64 + 64, n) * clear_per_gaussian;
    for (int k = first + int(threadIdx.x); k < last; k += kRankWaves * 64) clear[k] = 0.0f;
  }
  uint32_t before = 0;
  for (int c0 = 0; c0 < chunks; c0 += kRoundChunks) {  // workgroup-uniform
    if (c0) __syncthreads();  // the previous round's searches are done
    const int quads = min(chunks - c0, kRoundChunks) * (kChunk / 4);
    const uint4* from = reinterpret_cast<const uint4*>(chunk_keys + c0 * kChunk);
    uint4* to = reinterpret_cast<uint4*>(staged);
#pragma unroll
    for (int i = 0; i < kRoundChunks * kChunk / 4 / (kRankWaves * 64); ++i) {
      const int q = int(threadIdx.x) + i * kRankWaves * 64;
      if (q < quads) to[q] = from[q];
    }
    __syncthreads();
    // Keys of chunk c before mine: those of a chunk with lower indices also
    // where they are equal.  The chunks' searches run side by side; one that
    // is not there searches the first chunk, for nothing.
    int at[kWaveChunks];
    uint32_t place[kWaveChunks], below[kWaveChunks];
#pragma unroll
    for (int t = 0; t < kWaveChunks; ++t) {
      const int c = c0 + wid + t * kRankWaves;
      at[t] = c < chunks ? (c - c0) * kChunk : 0;
      place[t] = 0;
      // Counted: keys < below.  ~0u + 1 stays ~0u; see the end.
      below[t] = c < own && mine != 0xFFFFFFFFu ? mine + 1 : mine;
    }
#pragma unroll
    for (int step = kChunk / 2; step > 0; step >>= 1) {
#pragma unroll
      for (int t = 0; t < kWaveChunks; ++t)
        place[t] += staged[at[t] + place[t] + step - 1] < below[t] ? step : 0;
    }
#pragma unroll
    for (int t = 0; t < kWaveChunks; ++t) {
      const int c = c0 + wid + t * kRankWaves;
      place[t] += staged[at[t] + place[t]] < below[t] ? 1 : 0;  // place <= 255 before
      if (c < own && mine == 0xFFFFFFFFu) place[t] = kChunk;     // <= ~0u: all of them
      if (c < chunks && c != own) before += place[t];
    }
  }
  part[wid][lane] = before;
  __syncthreads();
  if (wid != 0 || id >= n) return;
  uint32_t rank = uint32_t(b % kBlocks * 64 + lane);
#pragma unroll
  for (int w = 0; w < kRankWaves; ++w) rank += part[w][lane];
  if (rank < uint32_t(n)) {  // always: the ranks are a permutation
    sorted_rects[rank] = rects[id];
    sorted_ids[rank] = uint16_t(id);
  }
}

// Workgroup (x, y): tiles x STRIP .. x STRIP + STRIP - 1 of tile row y.
// Dynamic LDS: the strip's masks [STRIP][blocks], then their prefixes
// [STRIP][blocks] (16 bits: below n), then the ids in depth order [n].
template <int STRIP>
__global__ __launch_bounds__(kListWaves * 64) void lists_kernel(
    const uint32_t* __restrict__ sorted_rects, const uint16_t* __restrict__ sorted_ids, int n,
    int tw, int64_t* __restrict__ ranges, int32_t* __restrict__ gaussian_ids) {
  extern __shared__ uint64_t lds[];
  const int blocks = (n + 63) >> 6;
  uint64_t* masks = lds;
  uint16_t* prefix = reinterpret_cast<uint16_t*>(masks + STRIP * blocks);
  uint16_t* ids = prefix + STRIP * blocks;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const uint32_t tx0 = blockIdx.x * STRIP, ty = blockIdx.y;

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
      for (int s = 0; s < STRIP; ++s) {
        const uint64_t m = __builtin_amdgcn_ballot_w64(row && tx0 + s - x0 <= w1);
        mine = lane == s ? m : mine;
      }
      if (lane < STRIP) masks[lane * blocks + b] = mine;
      if (b * 64 + lane < n) ids[b * 64 + lane] = id[i];
    }
  }
  __syncthreads();

  // 2. One wave per tile: the hits before each block, and the tile's range.
  if (wid < STRIP) {
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

  // 3. The lists: each tile's waves take equal chunks of up to 64 blocks,
  // one block's mask and prefix per lane, and visit the blocks with hits.
  constexpr int kTileWaves = kListWaves / STRIP;
  const int s = wid & (STRIP - 1);
  const int tx = int(tx0) + s;
  if (tx >= tw) return;  // wave-uniform, after the last barrier
  const int64_t t = int64_t(ty) * tw + tx;
  int32_t* list = gaussian_ids + t * n;
  const int share = min(64, (blocks + kTileWaves - 1) / kTileWaves);
  for (int b0 = wid / STRIP * share; b0 < blocks; b0 += kTileWaves * share) {
    const int b = lane < share ? b0 + lane : blocks;
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

template <int STRIP>
void launch_lists(const uint32_t* rects, const uint16_t* ids, int n, int tw, int th,
                  int64_t* ranges, int32_t* gaussian_ids, hipStream_t s) {
  const int64_t blocks = ceil_div(n, 64);
  const size_t lds = size_t(STRIP * blocks * 10 + blocks * 64 * 2);
  lists_kernel<STRIP><<<dim3(unsigned(ceil_div(tw, STRIP)), unsigned(th)), kListWaves * 64, lds,
                        s>>>(rects, ids, n, tw, ranges, gaussian_ids);
}

}  // namespace
}  // namespace gs

using namespace gs;

extern "C" {

GS_API size_t gs_small_lists_bytes(int64_t n, int32_t tiles_w, int32_t tiles_h) {
  if (tiles_w <= 0 || tiles_h <= 0 || tiles_w > kMaxAxisTiles || tiles_h > kMaxAxisTiles) return 0;
  if (!small_fits(n, int64_t(tiles_w) * tiles_h)) return 0;
  const size_t padded = size_t(ceil_div(n, kChunk)) * kChunk;
  return align_up(size_t(n) * 4) + align_up(size_t(n) * 2) + align_up(padded * 4) +
         align_up(padded * 2);
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
  const int chunks = int(ceil_div(n, kChunk));
  char* at = static_cast<char*>(workspace);
  uint32_t* rects = reinterpret_cast<uint32_t*>(at);
  at += align_up(size_t(n) * 4);
  uint16_t* ids = reinterpret_cast<uint16_t*>(at);
  at += align_up(size_t(n) * 2);
  uint32_t* chunk_keys = reinterpret_cast<uint32_t*>(at);
  at += align_up(size_t(chunks) * kChunk * 4);
  uint16_t* chunk_ids = reinterpret_cast<uint16_t*>(at);
  chunk_kernel<<<unsigned(chunks), kRankWaves * 64, 0, s>>>(depth_keys, int(n), chunk_keys,
                                                            chunk_ids);
  GS_TRY(check_launch("small_lists chunks"));
  rank_kernel<<<unsigned(chunks * kBlocks), kRankWaves * 64, 0, s>>>(
      chunk_keys, chunk_ids, chunks, tile_rects, int(n), rects, ids, clear, clear_per_gaussian);
  GS_TRY(check_launch("small_lists rank"));
  auto groups = [&](int strip) { return ceil_div(tiles_w, strip) * tiles_h; };
  auto lists = groups(1) <= kListGroups   ? launch_lists<1>
               : groups(2) <= kListGroups ? launch_lists<2>
                                          : launch_lists<4>;
  lists(rects, ids, int(n), tiles_w, tiles_h, ranges, gaussian_ids, s);
  return check_launch("small_lists");
}

}  // extern "C"
