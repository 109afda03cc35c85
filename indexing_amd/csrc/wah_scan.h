// wah_scan.h -- building blocks of the single-pass scans (the scan and
// compaction primitives, the staged kernels, WAH decode and encode): row
// loads, the look-back over two-field statuses, and the scan state that
// cleans up after itself.
#pragma once

#include "wah_device.h"
#include "wah_kernels.h"

namespace wah {

// Four consecutive 32-bit words.  Loads and stores of W4 ask for 4-byte
// alignment only (gfx950 global accesses of any width need no more), so every
// caller's pointer takes the same path.
typedef uint32_t W4 __attribute__((ext_vector_type(4)));
typedef W4 W4u __attribute__((aligned(4)));

// A tile is THREADS x 4 x ROWS elements.  A wave owns 256 x ROWS consecutive
// ones and loads them as ROWS rows of 256: lane l holds elements 4l .. 4l + 3
// of each row, one 16-byte load, so a wave's load covers 1 KiB without gaps.
// (A lane owning all its elements consecutively makes every load stride over
// the whole wave's range: 4 ROWS cache lines per wave instruction instead of
// 8, which held the earlier kernels under 1 TB/s.)
constexpr int kScanThreads = 512;
constexpr int kScanWaves = kScanThreads / kWave;
constexpr int kRowElems = 4 * kWave;
template <int ROWS>
constexpr uint32_t kScanTileOf = kScanThreads * 4 * ROWS;

// Element 4l of row r of wave w's part of a tile, relative to the tile.
template <int ROWS>
__device__ __forceinline__ uint32_t row_at(int w, int l, int r) {
  return (uint32_t)(w * ROWS * kRowElems + r * kRowElems + 4 * l);
}

// p[i .. i + 3], 0 at and past n.
template <bool FULL>
__device__ __forceinline__ W4 load4(const uint32_t* __restrict__ p, uint64_t i, uint64_t n) {
  if (FULL) return *reinterpret_cast<const W4u*>(p + i);
  W4 x = {0u, 0u, 0u, 0u};
  if (i < n) x.x = p[i];
  if (i + 1 < n) x.y = p[i + 1];
  if (i + 2 < n) x.z = p[i + 2];
  if (i + 3 < n) x.w = p[i + 3];
  return x;
}
template <bool FULL>
__device__ __forceinline__ void store4(uint32_t* __restrict__ p, uint64_t i, uint64_t n, W4 x) {
  if (FULL) {
    *reinterpret_cast<W4u*>(p + i) = x;
    return;
  }
  if (i < n) p[i] = x.x;
  if (i + 1 < n) p[i + 1] = x.y;
  if (i + 2 < n) p[i + 2] = x.z;
  if (i + 3 < n) p[i + 3] = x.w;
}

__device__ __forceinline__ uint32_t wave_max(uint32_t x) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) {
    const uint32_t o = __shfl_xor(x, d, kWave);
    x = o > x ? o : x;
  }
  return x;
}
__device__ __forceinline__ uint32_t wave_sum(uint32_t x) {
  return readlane(wave_incl_add(x), kWave - 1);
}
// Sums that stop at 2^32 - 1 instead of wrapping.
__device__ __forceinline__ uint32_t add_sat(uint32_t a, uint32_t b) {
  return __builtin_elementwise_add_sat(a, b);
}
__device__ __forceinline__ uint32_t wave_incl_add_sat(uint32_t x) {
  x = add_sat(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xF, 0xF, true));   // row_shr:1
  x = add_sat(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xF, 0xF, true));   // row_shr:2
  x = add_sat(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xF, 0xF, true));   // row_shr:4
  x = add_sat(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xF, 0xF, true));   // row_shr:8
  x = add_sat(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xA, 0xF, false));  // row_bcast:15
  x = add_sat(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xC, 0xF, false));  // row_bcast:31
  return x;
}
// Lane l - 1's x (lane 0: first), lane l + 1's x (lane 63: last).
__device__ __forceinline__ uint32_t lane_before(uint32_t x, uint32_t first) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)first, (int)x, 0x138, 0xF, 0xF, false);
}
__device__ __forceinline__ uint32_t lane_after(uint32_t x, uint32_t last) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)last, (int)x, 0x130, 0xF, 0xF, false);
}

// ---- look-back over status words flag << 62 | hi << 32 | lo --------------
// hi (30 bits) and lo (32 bits) combine separately over the earlier tiles:
constexpr int kOpNone = 0;
constexpr int kOpSum = 1;
constexpr int kOpMax = 2;
constexpr int kOpOrSinceHi = 3;  // lo: OR from the last tile with hi != 0 on
constexpr int kOpSumSat = 4;     // lo: sum, 2^32 - 1 at most

// Run by a whole wave: publishes the tile's (hi, lo) and returns the
// combination over tiles first .. tile - 1, reading 64 predecessors per round
// trip.  closed: the tile's own values already are the inclusive prefix
// (tile `first`; a segmented sum whose tile starts a segment), so later tiles
// stop there at once; else the inclusive prefix is published at the end.
template <int HI, int LO>
__device__ __forceinline__ void lookback2(uint64_t* status, uint32_t tile, uint32_t hi,
                                          uint32_t lo, bool closed, uint32_t* fault,
                                          uint32_t& pre_hi, uint32_t& pre_lo,
                                          uint32_t first = 0) {
  constexpr uint64_t kHiMask = (1ull << 30) - 1;
  const uint32_t lane = lane_id();
  const uint64_t own = ((hi & kHiMask) << 32) | lo;
  closed |= tile == first;
  if (lane == 0)
    st_agent(&status[tile], ((uint64_t)(closed ? kFlagPrefix : kFlagAgg) << 62) | own);
  uint32_t ah = 0, al = 0;
  bool or_open = true;  // kOpOrSinceHi: no tile with hi != 0 met yet
  int64_t base = (int64_t)tile - 1;
  ScanWait wait;
  while (base >= (int64_t)first) {
    const int64_t idx = base - (int64_t)lane;
    const uint64_t s = idx >= (int64_t)first ? ld_agent(&status[idx]) : ((uint64_t)kFlagPrefix << 62);
    const uint32_t f = (uint32_t)(s >> 62);
    const uint64_t pmask = ballot(f == kFlagPrefix);
    const uint64_t empty = ballot(f == 0);
    // lanes up to the nearest prefix, all of which have to be there
    const uint64_t need = pmask ? (pmask ^ (pmask - 1)) : ~0ull;
    if (empty & need) {
      if (wait.poll(empty & need)) {
        if (lane == 0) atomicOr(fault, 1u);
        break;
      }
      if ((wait.polls & 1023u) == 0 && ld_agent(fault)) break;
      __builtin_amdgcn_s_sleep(1);
      continue;
    }
    const bool take = (need >> lane) & 1u;
    const uint32_t h = take ? (uint32_t)((s >> 32) & kHiMask) : 0u;
    const uint32_t v = take ? (uint32_t)s : 0u;
    if (LO == kOpSum) al += wave_sum(v);
    if (LO == kOpSumSat) al = add_sat(al, readlane(wave_incl_add_sat(v), kWave - 1));
    if (LO == kOpOrSinceHi && or_open) {
      const uint64_t hm = ballot(h != 0u);
      const uint64_t upto = hm ? (hm ^ (hm - 1)) : ~0ull;
      al |= wave_or((upto >> lane) & 1u ? v : 0u);
      or_open = hm == 0;
    }
    if (HI == kOpSum) ah += wave_sum(h);
    if (HI == kOpMax) {
      const uint32_t m = wave_max(h);
      ah = m > ah ? m : ah;
    }
    if (pmask) break;
    base -= kWave;
    wait.next_window();
  }
  if (!closed && lane == 0) {
    uint32_t ih = 0, il = 0;
    if (HI == kOpSum) ih = ah + hi;
    if (HI == kOpMax) ih = hi > ah ? hi : ah;
    if (LO == kOpSum) il = al + lo;
    if (LO == kOpSumSat) il = add_sat(al, lo);
    if (LO == kOpOrSinceHi) il = hi ? lo : al | lo;
    st_agent(&status[tile], ((uint64_t)kFlagPrefix << 62) | ((ih & kHiMask) << 32) | il);
  }
  pre_hi = ah;
  pre_lo = al;
}

// ---- tiles and the state of a launch ---------------------------------------
// The block's next tile (`tiles` or more: none), by the rules of wah_tiles.h.  A
// launch with a block for every tile draws nothing: its blocks know their tile
// and that there is no other.
__device__ __forceinline__ uint32_t scan_next_tile(ScanState* st, uint32_t* s_tile, uint32_t tiles,
                                                   bool first) {
  if (!scan_draws(tiles, gridDim.x)) return first ? blockIdx.x : tiles;
  // (opaque: the draw's address is formed here, not kept in registers across a tile)
  uint32_t b = blockIdx.x;
  asm volatile("" : "+s"(b));
  if (threadIdx.x == 0) {
    const uint32_t lanes = tile_lanes(gridDim.x), lane = b % lanes;
    *s_tile = drawn_tile(atomicAdd(&st->tiles[lane * kLaneStride], 1u), lanes, lane);
  }
  __syncthreads();
  const uint32_t tile = __builtin_amdgcn_readfirstlane(*s_tile);
  __syncthreads();
  return tile;
}

// End of a block.  The last block of the launch hands the fault word and the
// result to the host (host: page-locked memory; where it is null nobody waits
// for the launch, and a fault goes to *kept) and zeroes the state
// for the next launch, so no launch needs a fill before it.  Every wave first
// waits for its own stores and atomics: a status published late would
// otherwise land on the zeroed state.  The blocks count themselves per lane
// and the lanes' last blocks count the lanes, since atomics on one address
// take about 11 ns each.
__device__ __forceinline__ void scan_finish(ScanState* st, uint64_t* status, uint32_t tiles,
                                            uint64_t* host, uint64_t* kept = nullptr) {
  __shared__ uint32_t s_last;
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) {
    const uint32_t lanes = tile_lanes(gridDim.x);
    const uint32_t lane = blockIdx.x % lanes;
    const uint32_t own = (gridDim.x - lane + lanes - 1) / lanes;
    bool last = atomicAdd(&st->tiles[lane * kLaneStride + 1], 1u) == own - 1;
    if (last) last = atomicAdd(&st->done, 1u) == lanes - 1;
    s_last = last;
  }
  __syncthreads();
  if (!s_last) return;
  for (uint32_t i = threadIdx.x; i < tiles; i += blockDim.x) st_agent(&status[i], (uint64_t)0);
  if (threadIdx.x == 0) {
    const uint64_t f = ld_agent(&st->fault);
    uint64_t r = ld_agent(&st->result);
    for (uint32_t i = 0; i < kTileLanes; ++i) {  // the lanes' maxima
      const uint64_t m = ld_agent(reinterpret_cast<uint64_t*>(&st->tiles[i * kLaneStride + 2]));
      r = m > r ? m : r;
    }
    if (host) {
      __hip_atomic_store(&host[0], f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      __hip_atomic_store(&host[1], r, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    } else if (f) {
      __hip_atomic_store(kept, f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    st_agent(&st->fault, 0u);
    st_agent(&st->done, 0u);
    st_agent(&st->result, (uint64_t)0);
    for (uint32_t i = 0; i < kTileLanes; ++i)
      for (uint32_t j = 0; j < 4; ++j) st_agent(&st->tiles[i * kLaneStride + j], 0u);
  }
}

// Stores the tile's `count` words staged in LDS (word i at stage[i]) to
// out[0 .. count): single words up to the first 16-byte boundary, then 16
// bytes per store, then the rest.
__device__ __forceinline__ void store_staged(const uint32_t* stage, uint32_t* __restrict__ out,
                                             uint32_t count) {
  const uint32_t t = threadIdx.x;
  const uint32_t head0 = (4u - (uint32_t)(((uintptr_t)out >> 2) & 3u)) & 3u;
  const uint32_t head = head0 < count ? head0 : count;
  const uint32_t quads = (count - head) / 4u;
  if (t < head) out[t] = stage[t];
  for (uint32_t q = t; q < quads; q += blockDim.x) {
    const uint32_t j = head + 4u * q;
    const W4 v = {stage[j], stage[j + 1], stage[j + 2], stage[j + 3]};
    *reinterpret_cast<W4*>(out + j) = v;
  }
  const uint32_t j = head + 4u * quads + t;
  if (j < count) out[j] = stage[j];
}

}  // namespace wah
