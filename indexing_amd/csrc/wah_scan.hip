// wah_scan.hip -- gfx950 kernels of the scan and compaction primitives and of
// the stages that are scans (merge, fuse, column length).  Each is one launch:
// a tile's elements are read once into registers, combined across lanes (DPP),
// waves (LDS) and tiles (look-back), and written once; wah_scan.h holds the
// parts.  What bounds them is HBM.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "wah_scan.h"

namespace wah {

namespace {

// Rows per tile and blocks per CU of each kernel. A launch has no more blocks
// than the registers and LDS of a block let the device hold at once. What a tile
// costs besides its bytes is one look-back (its wait is for the tiles just
// before it), so the largest tiles that leave two blocks per CU are the fastest:
// 2^24 elements, 16384-element tiles at two blocks per CU against 8192 at four
// and 4096 at four: scan 31.7 / 35.8 / 46.9 us, compaction 40.2 / 42.6 / 51.4
// us, fuse (half the elements) 20.6 / 22.7 / 28.9 us on 2^22 (timed with blocks
// that took their first tile by index). The segmented scan and the column
// lengths hold more registers per row and gain nothing from a larger tile.
constexpr int kScanRows = 8, kCompactRows = 8, kFuseRows = 4, kSegRows = 4, kMergeRows = 4,
              kColenRows = 4;
constexpr int kScanBlocks = 2;
// Under kSmallScan elements the chip is not filled and a tile's own latency
// counts: three calls on 30,011 elements take 48 us with tiles of 8192 and 56
// with 16384; at 2^20 the larger ones are ahead (46.7 against 47.8 us).
constexpr int kSmallRows = 2;
constexpr uint64_t kSmallScan = 1ull << 19;
constexpr int waves_per_eu(int blocks) { return blocks * kScanWaves / 4; }

// Sum of the waves' values before wave w, and of all (s_tot: one per wave).
__device__ __forceinline__ uint32_t waves_before(const uint32_t* s_tot, int w, uint32_t* all) {
  const uint32_t l = lane_id();
  const uint32_t x = l < (uint32_t)kScanWaves ? s_tot[l] : 0u;
  const uint32_t inc = wave_incl_add(x);
  *all = readlane(inc, kScanWaves - 1);
  return readlane(inc - x, w);
}

}  // namespace

// Exclusive uint32 sum scan (include/scan.cl), wrapping mod 2^32.  2^24
// elements: 34.5 us (3.9 TB/s); 184 us as one look-back thread per tile of
// 2048 elements and lanes that load 8 consecutive ones.
template <int ROWS>
__global__ __launch_bounds__(kScanThreads, waves_per_eu(kScanBlocks)) void k_scan(
    const uint32_t* in, uint64_t n, uint32_t* out, ScanState* st, uint64_t* status,
    uint32_t tiles, uint64_t* kept) {
  constexpr uint32_t TILE = kScanTileOf<ROWS>;
  __shared__ uint32_t s_tot[kScanWaves];
  __shared__ uint32_t s_prefix, s_tile;
  const int l = threadIdx.x % kWave;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  for (uint32_t tile = scan_next_tile(st, &s_tile, tiles, true); tile < tiles;
       tile = scan_next_tile(st, &s_tile, tiles, false)) {
    const uint64_t base = (uint64_t)tile * TILE;
    auto body = [&](auto full_tag) {
      constexpr bool FULL = decltype(full_tag)::value;
      W4 x[ROWS];
      uint32_t ex[ROWS], run = 0;
#pragma unroll
      for (int r = 0; r < ROWS; ++r) x[r] = load4<FULL>(in, base + row_at<ROWS>(w, l, r), n);
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        const uint32_t s = x[r].x + x[r].y + x[r].z + x[r].w;
        const uint32_t inc = wave_incl_add(s);
        ex[r] = run + inc - s;
        run += readlane(inc, kWave - 1);
      }
      if (l == 0) s_tot[w] = run;
      __syncthreads();
      uint32_t all;
      const uint32_t before = waves_before(s_tot, w, &all);
      if (w == 0) {
        uint32_t h, p;
        lookback2<kOpNone, kOpSum>(status, tile, 0u, all, false, &st->fault, h, p);
        if (l == 0) s_prefix = p;
      }
      __syncthreads();
      const uint32_t add = s_prefix + before;
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        W4 o;
        o.x = ex[r] + add;
        o.y = o.x + x[r].x;
        o.z = o.y + x[r].y;
        o.w = o.z + x[r].z;
        store4<FULL>(out, base + row_at<ROWS>(w, l, r), n, o);
      }
    };
    if (base + TILE <= n) body(std::true_type{});
    else body(std::false_type{});
  }
  scan_finish(st, status, tiles, nullptr, kept);
}

// Segmented inclusive sum scan (include/segmented_scan.cl): restarts where
// heads != 0.  Inside a wave it is the plain scan minus the plain scan's value
// at the segment's head (both wrap mod 2^32, so the difference is exact):
// one DPP scan per row and one shuffle that fetches the head's value, instead
// of a scan whose every step selects.  Elements of a segment that began before
// the wave are "open" and take the carry once it is known.  A tile with a head
// publishes its last segment's sum as a prefix at once: later tiles need
// nothing from before it.  2^24 elements: 41.6 us (4.8 TB/s; was 230 us).
__global__ __launch_bounds__(kScanThreads, waves_per_eu(kScanBlocks)) void k_segscan(
    const uint32_t* in, const uint32_t* heads, uint64_t n, uint32_t* out, ScanState* st,
    uint64_t* status, uint32_t tiles, uint64_t* kept) {
  constexpr int ROWS = kSegRows;
  constexpr uint32_t TILE = kScanTileOf<ROWS>;
  __shared__ uint32_t s_sum[kScanWaves], s_head[kScanWaves];
  __shared__ uint32_t s_prefix, s_tile;
  const int l = threadIdx.x % kWave;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  for (uint32_t tile = scan_next_tile(st, &s_tile, tiles, true); tile < tiles;
       tile = scan_next_tile(st, &s_tile, tiles, false)) {
    const uint64_t base = (uint64_t)tile * TILE;
    auto body = [&](auto full_tag) {
      constexpr bool FULL = decltype(full_tag)::value;
      W4 x[ROWS];
      uint32_t hb = 0;  // head flags of the lane's elements: bit 4r + k
#pragma unroll
      for (int r = 0; r < ROWS; ++r) x[r] = load4<FULL>(in, base + row_at<ROWS>(w, l, r), n);
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        const W4 h = load4<FULL>(heads, base + row_at<ROWS>(w, l, r), n);
        hb |= ((h.x ? 1u : 0u) | (h.y ? 2u : 0u) | (h.z ? 4u : 0u) | (h.w ? 8u : 0u)) << (4 * r);
      }
      if (tile == 0 && threadIdx.x == 0) hb |= 1u;  // element 0 starts a segment
      uint32_t run = 0;    // plain sum of the wave's earlier rows
      uint32_t start = 0;  // plain sum before the open segment's head
      uint32_t openm = 0;  // elements whose segment began before the wave
      bool open = true;    // no head in the wave's earlier rows
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        const uint32_t h4 = (hb >> (4 * r)) & 15u;
        const uint32_t p1 = x[r].x, p2 = p1 + x[r].y, p3 = p2 + x[r].z, s = p3 + x[r].w;
        const uint32_t inc = wave_incl_add(s);
        const uint32_t ex = run + inc - s;
        // plain sum before the lane's last head
        const uint32_t b = ex + (h4 & 8u ? p3 : h4 & 4u ? p2 : h4 & 2u ? p1 : 0u);
        const uint64_t hm = ballot(h4 != 0u);
        const uint64_t below = hm & ((1ull << l) - 1ull);
        const int src = below ? 63 - __builtin_clzll(below) : 0;
        const uint32_t got = __shfl(b, src, kWave);
        uint32_t cur = below ? got : start;
        bool o = !below && open;
        W4 y;
        if (h4 & 1u) { cur = ex; o = false; }
        y.x = ex + p1 - cur;
        openm |= o ? 1u << (4 * r) : 0u;
        if (h4 & 2u) { cur = ex + p1; o = false; }
        y.y = ex + p2 - cur;
        openm |= o ? 2u << (4 * r) : 0u;
        if (h4 & 4u) { cur = ex + p2; o = false; }
        y.z = ex + p3 - cur;
        openm |= o ? 4u << (4 * r) : 0u;
        if (h4 & 8u) { cur = ex + p3; o = false; }
        y.w = ex + s - cur;
        openm |= o ? 8u << (4 * r) : 0u;
        x[r] = y;
        run += readlane(inc, kWave - 1);
        if (hm) {  // wave-uniform
          start = readlane(b, 63 - __builtin_clzll(hm));
          open = false;
        }
      }
      if (l == 0) {
        s_sum[w] = open ? run : run - start;
        s_head[w] = open ? 0u : 1u;
      }
      __syncthreads();
      // carry into the wave from the tile's earlier waves; the tile's own
      uint32_t carry = 0, agg = 0;
      bool closed = false, tile_closed = false;
#pragma unroll
      for (int i = 0; i < kScanWaves; ++i) {
        if (i == w) {
          carry = agg;
          closed = tile_closed;
        }
        const bool h = s_head[i] != 0u;
        agg = h ? s_sum[i] : agg + s_sum[i];
        tile_closed |= h;
      }
      if (w == 0) {
        uint32_t hi, p;
        lookback2<kOpNone, kOpSum>(status, tile, 0u, agg, tile_closed, &st->fault, hi, p);
        if (l == 0) s_prefix = p;
      }
      __syncthreads();
      if (!closed) carry += s_prefix;
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        const uint32_t o4 = openm >> (4 * r);
        W4 y = x[r];
        y.x += o4 & 1u ? carry : 0u;
        y.y += o4 & 2u ? carry : 0u;
        y.z += o4 & 4u ? carry : 0u;
        y.w += o4 & 8u ? carry : 0u;
        store4<FULL>(out, base + row_at<ROWS>(w, l, r), n, y);
      }
    };
    if (base + TILE <= n) body(std::true_type{});
    else body(std::false_type{});
  }
  scan_finish(st, status, tiles, nullptr, kept);
}

// Order-preserving compaction.  FUSE false: keep a[i] where b[i] != 0
// (include/stream_compaction.cl:124-160).  FUSE true: the interleaved words
// (a[i], b[i]) with zero words dropped (fuse_fill_literals); half the
// elements per tile, since each may leave two words.  The kept words are
// placed in LDS by a scan of the lanes' counts and stored contiguously.  2^24
// elements, half kept: 42 us (4.0 TB/s; was 204 us); 2^22 entries fused: 21 us
// (3.2 TB/s; was 85 us).
template <int ROWS, bool FUSE>
__global__ __launch_bounds__(kScanThreads, waves_per_eu(kScanBlocks)) void k_compact(
    const uint32_t* __restrict__ a, const uint32_t* __restrict__ b, uint64_t n,
    uint32_t* __restrict__ out, ScanState* st, uint64_t* status, uint32_t tiles, uint64_t* host) {
  constexpr uint32_t TILE = kScanTileOf<ROWS>;
  const uint64_t cap = FUSE ? 2 * n : n;
  __shared__ uint32_t s_stage[FUSE ? 2 * TILE : TILE];
  __shared__ uint32_t s_tot[kScanWaves];
  __shared__ uint32_t s_prefix, s_tile;
  const int l = threadIdx.x % kWave;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  for (uint32_t tile = scan_next_tile(st, &s_tile, tiles, true); tile < tiles;
       tile = scan_next_tile(st, &s_tile, tiles, false)) {
    const uint64_t base = (uint64_t)tile * TILE;
    uint32_t all;
    auto body = [&](auto full_tag) {
      constexpr bool FULL = decltype(full_tag)::value;
      W4 x[ROWS], y[ROWS];
      uint32_t pos[ROWS], run = 0;
#pragma unroll
      for (int r = 0; r < ROWS; ++r) y[r] = load4<FULL>(b, base + row_at<ROWS>(w, l, r), n);
#pragma unroll
      for (int r = 0; r < ROWS; ++r) x[r] = load4<FULL>(a, base + row_at<ROWS>(w, l, r), n);
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        uint32_t c = (y[r].x != 0u) + (y[r].y != 0u) + (y[r].z != 0u) + (y[r].w != 0u);
        if (FUSE) c += (x[r].x != 0u) + (x[r].y != 0u) + (x[r].z != 0u) + (x[r].w != 0u);
        const uint32_t inc = wave_incl_add(c);
        pos[r] = run + inc - c;
        run += readlane(inc, kWave - 1);
      }
      if (l == 0) s_tot[w] = run;
      __syncthreads();
      const uint32_t before = waves_before(s_tot, w, &all);
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        uint32_t p = before + pos[r];
        const uint32_t xv[4] = {x[r].x, x[r].y, x[r].z, x[r].w};
        const uint32_t yv[4] = {y[r].x, y[r].y, y[r].z, y[r].w};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          if (FUSE) {
            if (xv[k]) s_stage[p++] = xv[k];
            if (yv[k]) s_stage[p++] = yv[k];
          } else {
            if (yv[k]) s_stage[p++] = xv[k];
          }
        }
      }
    };
    if (base + TILE <= n) body(std::true_type{});
    else body(std::false_type{});
    if (w == 0) {
      uint32_t h, p;
      lookback2<kOpNone, kOpSum>(status, tile, 0u, all, false, &st->fault, h, p);
      if (l == 0) {
        s_prefix = p;
        if (tile == tiles - 1) st_agent(&st->result, (uint64_t)p + all);
      }
    }
    __syncthreads();
    const uint32_t pre = s_prefix;
    if ((uint64_t)pre + all <= cap) store_staged(s_stage, out + pre, all);
    else if (threadIdx.x == 0) atomicOr(&st->fault, 2u);  // never for a consistent scan
  }
  scan_finish(st, status, tiles, host);
}

// Reduce-by-key OR over runs of equal (value, chid), any run length
// (include/merge_lit_by_val_chids.cl).  An element is a head when it differs
// from its predecessor and a last when its successor is a head; a run's last
// element emits (value, chid, OR of the run) at index heads - 1.  The OR runs
// along the lane's four elements, then across lanes with DPP steps that stop
// at the lane of the nearest head, then across waves and tiles by carries.
// The three output arrays leave through one LDS buffer, one after another.
// 2^22 pairs: 32 us (3.2 TB/s; was 124 us with a 64-bit scan operator over
// shuffles, three reads of the inputs and one look-back thread).
__global__ __launch_bounds__(kScanThreads, waves_per_eu(kScanBlocks)) void k_merge(
    const uint32_t* __restrict__ vals, const uint32_t* __restrict__ chids,
    const uint32_t* __restrict__ lits, uint64_t n, uint32_t* __restrict__ out_v,
    uint32_t* __restrict__ out_c, uint32_t* __restrict__ out_l, ScanState* st, uint64_t* status,
    uint32_t tiles, uint64_t* host) {
  constexpr int ROWS = kMergeRows;
  constexpr uint32_t TILE = kScanTileOf<ROWS>;
  __shared__ uint32_t s_stage[TILE];
  __shared__ uint32_t s_heads[kScanWaves], s_lasts[kScanWaves], s_or[kScanWaves];
  __shared__ uint32_t s_pre_heads, s_pre_or, s_tile;
  const int l = threadIdx.x % kWave;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  for (uint32_t tile = scan_next_tile(st, &s_tile, tiles, true); tile < tiles;
       tile = scan_next_tile(st, &s_tile, tiles, false)) {
    const uint64_t base = (uint64_t)tile * TILE;
    auto body = [&](auto full_tag) {
      constexpr bool FULL = decltype(full_tag)::value;
      const uint64_t wb = base + row_at<ROWS>(w, 0, 0);  // the wave's first element
      W4 v[ROWS], c[ROWS], o[ROWS];
#pragma unroll
      for (int r = 0; r < ROWS; ++r) v[r] = load4<FULL>(vals, wb + row_at<ROWS>(0, l, r), n);
#pragma unroll
      for (int r = 0; r < ROWS; ++r) c[r] = load4<FULL>(chids, wb + row_at<ROWS>(0, l, r), n);
#pragma unroll
      for (int r = 0; r < ROWS; ++r) o[r] = load4<FULL>(lits, wb + row_at<ROWS>(0, l, r), n);
      // the elements before and after the wave's (uniform loads)
      const uint64_t wn = wb + (uint64_t)ROWS * kRowElems;
      uint32_t pv = 0, pc = 0, nv = 0, nc = 0;
      const bool have_prev = wb > 0 && wb <= n, have_next = wn < n;
      if (have_prev) { pv = vals[wb - 1]; pc = chids[wb - 1]; }
      if (have_next) { nv = vals[wn]; nc = chids[wn]; }
      uint32_t hb = 0;     // head flags, bit 4r + k
      uint32_t valid = 0;  // elements below n
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        const uint32_t qv = lane_before(v[r].w, r ? readlane(v[r ? r - 1 : 0].w, kWave - 1) : pv);
        const uint32_t qc = lane_before(c[r].w, r ? readlane(c[r ? r - 1 : 0].w, kWave - 1) : pc);
        uint32_t h = (v[r].x != qv || c[r].x != qc ? 1u : 0u) |
                     (v[r].y != v[r].x || c[r].y != c[r].x ? 2u : 0u) |
                     (v[r].z != v[r].y || c[r].z != c[r].y ? 4u : 0u) |
                     (v[r].w != v[r].z || c[r].w != c[r].z ? 8u : 0u);
        uint32_t ok = 15u;
        if (!FULL) {
          const uint64_t g = wb + row_at<ROWS>(0, l, r);
          ok = g + 4 <= n ? 15u : g < n ? (1u << (uint32_t)(n - g)) - 1u : 0u;
        }
        hb |= (h & ok) << (4 * r);
        valid |= ok << (4 * r);
      }
      if (tile == 0 && threadIdx.x == 0 && n) hb |= 1u;
      // last flags: the next element is a head, or there is none
      const bool next_head = !have_next || nv != readlane(v[ROWS - 1].w, kWave - 1) ||
                             nc != readlane(c[ROWS - 1].w, kWave - 1);
      uint32_t lb = 0;
      {
        // heads and ends of the following element, bit 4r + k
        const uint32_t stop = hb | ~valid;
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
          const uint32_t s4 = (stop >> (4 * r)) & 15u;
          const uint32_t after = r + 1 < ROWS
                                     ? readlane(stop, 0) >> (4 * (r + 1 < ROWS ? r + 1 : r)) & 1u
                                     : (next_head ? 1u : 0u);
          const uint32_t nx = lane_after(s4 & 1u, after);
          lb |= ((s4 >> 1) | nx << 3) << (4 * r);
        }
        lb &= valid;
      }
      // OR since the nearest head, within the wave
      uint32_t openm = 0;      // elements whose run began before the wave
      uint32_t carry_or = 0;   // OR since the last head of the wave's earlier rows
      bool open = true;
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        const uint32_t h4 = (hb >> (4 * r)) & 15u;
        // along the lane
        W4 y = o[r];
        y.y |= h4 & 2u ? 0u : y.x;
        y.z |= h4 & 4u ? 0u : y.y;
        y.w |= h4 & 8u ? 0u : y.z;
        // across lanes: x = OR over lanes max(hl, l - d + 1) .. l, hl the
        // nearest lane at or below with a head (its part after that head)
        const uint64_t hm = ballot(h4 != 0u);
        const uint64_t upto = hm & (l == kWave - 1 ? ~0ull : (2ull << l) - 1ull);
        const int hl = upto ? 63 - __builtin_clzll(upto) : 0;
        uint32_t x = y.w;
        const int in_row = l % 16;
        uint32_t s;
        s = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xF, 0xF, true);
        x |= l - hl >= 1 && in_row >= 1 ? s : 0u;
        s = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xF, 0xF, true);
        x |= l - hl >= 2 && in_row >= 2 ? s : 0u;
        s = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xF, 0xF, true);
        x |= l - hl >= 4 && in_row >= 4 ? s : 0u;
        s = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xF, 0xF, true);
        x |= l - hl >= 8 && in_row >= 8 ? s : 0u;
        // lane 15 of the row before, for rows 1 and 3, then lane 31 for rows 2, 3
        s = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xA, 0xF, false);
        x |= hl < (l & ~15) ? s : 0u;
        s = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xC, 0xF, false);
        x |= hl < 32 ? s : 0u;
        const uint32_t prev = lane_before(x, 0u);  // OR since the nearest head below the lane
        const uint64_t below = hm & ((1ull << l) - 1ull);
        uint32_t in = prev | (below ? 0u : carry_or);
        const bool op = !below && open;
        // into the lane's elements before its first head
        const uint32_t lead = h4 ? (h4 & (~h4 + 1u)) - 1u : 15u;
        y.x |= lead & 1u ? in : 0u;
        y.y |= lead & 2u ? in : 0u;
        y.z |= lead & 4u ? in : 0u;
        y.w |= lead & 8u ? in : 0u;
        openm |= op ? lead << (4 * r) : 0u;
        o[r] = y;
        carry_or = readlane(y.w, kWave - 1);
        open = open && hm == 0;
      }
      // wave totals: heads, lasts and the OR since the last head
      const uint32_t hsum = wave_sum((uint32_t)__builtin_popcount(hb));
      // lasts before each row's lane: rows' counts are at most 256
      uint32_t pos[ROWS], run = 0;
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        const uint32_t k = (uint32_t)__builtin_popcount((lb >> (4 * r)) & 15u);
        const uint32_t inc = wave_incl_add(k);
        pos[r] = run + inc - k;
        run += readlane(inc, kWave - 1);
      }
      if (l == 0) {
        s_heads[w] = hsum;
        s_lasts[w] = run;
        s_or[w] = carry_or;
      }
      __syncthreads();
      uint32_t heads_all = 0, lasts_all = 0, lasts_before = 0, agg = 0, carry = 0;
      bool closed = false, any = false;  // a head in the earlier waves of the tile / in the tile
#pragma unroll
      for (int i = 0; i < kScanWaves; ++i) {
        if (i == w) {
          lasts_before = lasts_all;
          carry = agg;
          closed = any;
        }
        const uint32_t h = s_heads[i];
        agg = h ? s_or[i] : agg | s_or[i];
        any |= h != 0u;
        heads_all += h;
        lasts_all += s_lasts[i];
      }
      if (w == 0) {
        uint32_t ph, po;
        lookback2<kOpSum, kOpOrSinceHi>(status, tile, heads_all, agg, false, &st->fault, ph, po);
        if (l == 0) {
          s_pre_heads = ph;
          s_pre_or = po;
          if (tile == tiles - 1) st_agent(&st->result, (uint64_t)ph + heads_all);
        }
      }
      // the first emitted run has index (heads before the tile) - 1 when it
      // began before the tile, else (heads before the tile)
      const bool cont = tile > 0 && readlane(hb & 1u, 0) == 0u;  // wave 0's is the tile's
      if (threadIdx.x == 0) s_tile = cont ? 1u : 0u;             // free between draws
      auto put = [&](const W4* x) {
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
          uint32_t p = lasts_before + pos[r];
          const uint32_t e[4] = {x[r].x, x[r].y, x[r].z, x[r].w};
#pragma unroll
          for (int k = 0; k < 4; ++k)
            if ((lb >> (4 * r + k)) & 1u) s_stage[p++] = e[k];
        }
      };
      put(v);
      __syncthreads();
      const uint64_t at = (uint64_t)s_pre_heads - s_tile;
      const bool fits = at + lasts_all <= n;
      if (!fits && threadIdx.x == 0) atomicOr(&st->fault, 2u);
      if (fits) store_staged(s_stage, out_v + at, lasts_all);
      if (!closed) carry |= s_pre_or;
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        const uint32_t o4 = openm >> (4 * r);
        o[r].x |= o4 & 1u ? carry : 0u;
        o[r].y |= o4 & 2u ? carry : 0u;
        o[r].z |= o4 & 4u ? carry : 0u;
        o[r].w |= o4 & 8u ? carry : 0u;
      }
      __syncthreads();
      put(c);
      __syncthreads();
      if (fits) store_staged(s_stage, out_c + at, lasts_all);
      __syncthreads();
      put(o);
      __syncthreads();
      if (fits) store_staged(s_stage, out_l + at, lasts_all);
      __syncthreads();
    };
    if (base + TILE <= n) body(std::true_type{});
    else body(std::false_type{});
  }
  scan_finish(st, status, tiles, host);
}

// compute_column_length over merged entries (values, fills): keys at value
// changes, offsets = exclusive scan of (1 + (fill != 0)).  Keys and words of a
// tile fit 16 bits each, so one scan per row carries both.  2^22 entries: 17 us
// (was 59 us).
__global__ __launch_bounds__(kScanThreads, waves_per_eu(kScanBlocks)) void k_colen(
    const uint32_t* __restrict__ vals, const uint32_t* __restrict__ fills, uint64_t k,
    uint32_t* __restrict__ out_keys, uint32_t* __restrict__ out_offsets,
    wahgpu_counts_dev* __restrict__ counts, ScanState* st, uint64_t* status, uint32_t tiles,
    uint64_t* host) {
  constexpr int ROWS = kColenRows;
  constexpr uint32_t TILE = kScanTileOf<ROWS>;
  static_assert(2 * TILE < 65536, "a tile's words fit 16 bits");
  __shared__ uint32_t s_tot[kScanWaves];
  __shared__ uint32_t s_keys, s_words, s_tile;
  const int l = threadIdx.x % kWave;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  for (uint32_t tile = scan_next_tile(st, &s_tile, tiles, true); tile < tiles;
       tile = scan_next_tile(st, &s_tile, tiles, false)) {
    const uint64_t base = (uint64_t)tile * TILE;
    auto body = [&](auto full_tag) {
      constexpr bool FULL = decltype(full_tag)::value;
      const uint64_t wb = base + row_at<ROWS>(w, 0, 0);
      W4 v[ROWS];
      uint32_t hb = 0, fb = 0;  // key starts and nonzero fills, bit 4r + k
#pragma unroll
      for (int r = 0; r < ROWS; ++r) v[r] = load4<FULL>(vals, wb + row_at<ROWS>(0, l, r), k);
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        const W4 f = load4<FULL>(fills, wb + row_at<ROWS>(0, l, r), k);
        fb |= ((f.x ? 1u : 0u) | (f.y ? 2u : 0u) | (f.z ? 4u : 0u) | (f.w ? 8u : 0u)) << (4 * r);
      }
      uint32_t pv = 0;
      if (wb > 0 && wb <= k) pv = vals[wb - 1];
      uint32_t ex[ROWS], run = 0;
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        const uint32_t qv = lane_before(v[r].w, r ? readlane(v[r ? r - 1 : 0].w, kWave - 1) : pv);
        uint32_t ok = 15u;
        if (!FULL) {
          const uint64_t g = wb + row_at<ROWS>(0, l, r);
          ok = g + 4 <= k ? 15u : g < k ? (1u << (uint32_t)(k - g)) - 1u : 0u;
        }
        uint32_t h = (v[r].x != qv ? 1u : 0u) | (v[r].y != v[r].x ? 2u : 0u) |
                     (v[r].z != v[r].y ? 4u : 0u) | (v[r].w != v[r].z ? 8u : 0u);
        if (r == 0 && tile == 0 && threadIdx.x == 0) h |= 1u;
        h &= ok;
        hb |= h << (4 * r);
        const uint32_t words = (uint32_t)(__builtin_popcount(ok) + __builtin_popcount((fb >> (4 * r)) & ok));
        const uint32_t s = ((uint32_t)__builtin_popcount(h) << 16) | words;
        const uint32_t inc = wave_incl_add(s);
        ex[r] = run + inc - s;
        run += readlane(inc, kWave - 1);
      }
      if (l == 0) s_tot[w] = run;
      __syncthreads();
      uint32_t all;
      const uint32_t before = waves_before(s_tot, w, &all);
      if (w == 0) {
        uint32_t ph, pw;
        lookback2<kOpSum, kOpSum>(status, tile, all >> 16, all & 0xFFFFu, false, &st->fault, ph, pw);
        if (l == 0) {
          s_keys = ph;
          s_words = pw;
          if (tile == tiles - 1) {
            counts->length = (uint64_t)pw + (all & 0xFFFFu);
            counts->keycnt = (uint64_t)ph + (all >> 16);
            st_agent(&st->result, (uint64_t)ph + (all >> 16));
          }
        }
      }
      __syncthreads();
      const uint32_t kb = s_keys, wp = s_words;
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        const uint32_t h4 = (hb >> (4 * r)) & 15u;
        if (!h4) continue;
        const uint32_t at = before + ex[r];
        uint32_t ki = kb + (at >> 16);
        const uint32_t w0 = wp + (at & 0xFFFFu);
        const uint32_t e[4] = {v[r].x, v[r].y, v[r].z, v[r].w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if ((h4 >> i) & 1u) {
            const uint32_t below = (1u << i) - 1u;
            if (ki < k) {
              out_keys[ki] = e[i];
              out_offsets[ki] = w0 + i + (uint32_t)__builtin_popcount((fb >> (4 * r)) & below);
            } else {
              atomicOr(&st->fault, 2u);
            }
            ++ki;
          }
        }
      }
    };
    if (base + TILE <= k) body(std::true_type{});
    else body(std::false_type{});
  }
  scan_finish(st, status, tiles, host);
}

// lengths[i] = offsets[i+1] - offsets[i]; the last key runs to L.
__global__ __launch_bounds__(kBlock) void k_lengths(const uint32_t* __restrict__ offsets,
                                                    uint32_t* __restrict__ lengths,
                                                    const wahgpu_counts_dev* __restrict__ counts,
                                                    uint64_t cap) {
  const uint64_t K = counts->keycnt < cap ? counts->keycnt : cap, L = counts->length;
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < K;
       i += (uint64_t)gridDim.x * kBlock) {
    const uint32_t end = (i + 1 < K) ? offsets[i + 1] : (uint32_t)L;
    lengths[i] = end - offsets[i];
  }
}

// ---- launchers ---------------------------------------------------------------

namespace {
constexpr int least(int a, int b) { return a < b ? a : b; }
static_assert(WAHGPU_MAX_VALUES <=
                      kScanStatusWords *
                          kScanTileOf<least(least(kScanRows, kCompactRows),
                                            least(least(kFuseRows, kSegRows),
                                                  least(kMergeRows, kColenRows)))> &&
                  kSmallScan / kScanTileOf<kSmallRows> <= kScanStatusWords,
              "a status word per tile of every scan");
struct Tiles {
  uint32_t count, grid;
};
Tiles tiles_of(uint64_t n, int rows, const ScanRun& a) {
  const uint64_t tile = kScanThreads * 4 * rows;
  const uint32_t count = (uint32_t)((n + tile - 1) / tile), most = a.cus * (uint32_t)kScanBlocks;
  return {count, count < most ? count : most};
}
}  // namespace

void launch_scan(const ScanRun& a, const uint32_t* in, const uint32_t* heads, uint64_t n,
                 uint32_t* out, bool segmented, hipStream_t s) {
  if (!n) return;
  const bool small = n < kSmallScan;
  const Tiles t = tiles_of(n, segmented ? kSegRows : small ? kSmallRows : kScanRows, a);
  if (a.captured)  // the status words follow the state
    launch_fill32(reinterpret_cast<uint32_t*>(a.state), sizeof(ScanState) / 4 + 2ull * t.count, 0, s);
  if (segmented)
    hipLaunchKernelGGL(k_segscan, dim3(t.grid), dim3(kScanThreads), 0, s, in, heads, n, out,
                       a.state, a.status, t.count, a.kept);
  else if (small)
    hipLaunchKernelGGL(k_scan<kSmallRows>, dim3(t.grid), dim3(kScanThreads), 0, s, in, n, out,
                       a.state, a.status, t.count, a.kept);
  else
    hipLaunchKernelGGL(k_scan<kScanRows>, dim3(t.grid), dim3(kScanThreads), 0, s, in, n, out,
                       a.state, a.status, t.count, a.kept);
}

void launch_compact(const ScanRun& a, const uint32_t* data, const uint32_t* valid, uint64_t n,
                    int mode, uint32_t* out, hipStream_t s) {
  if (!n) return;
  const bool small = n < kSmallScan;
  const Tiles t = tiles_of(n, small ? kSmallRows : mode == 0 ? kCompactRows : kFuseRows, a);
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(t.grid), dim3(kScanThreads), 0, s, data, valid, n, out,
                       a.state, a.status, t.count, a.host);
  };
  if (mode == 0) go(small ? k_compact<kSmallRows, false> : k_compact<kCompactRows, false>);
  else go(small ? k_compact<kSmallRows, true> : k_compact<kFuseRows, true>);
}

void launch_merge(const ScanRun& a, const uint32_t* vals, const uint32_t* chids,
                  const uint32_t* lits, uint64_t n, uint32_t* ov, uint32_t* oc, uint32_t* ol,
                  hipStream_t s) {
  if (!n) return;
  const Tiles t = tiles_of(n, kMergeRows, a);
  hipLaunchKernelGGL(k_merge, dim3(t.grid), dim3(kScanThreads), 0, s, vals, chids, lits, n, ov,
                     oc, ol, a.state, a.status, t.count, a.host);
}

void launch_colen(const ScanRun& a, const uint32_t* vals, const uint32_t* fills, uint64_t k,
                  uint32_t* keys, uint32_t* offsets, uint32_t* lengths,
                  wahgpu_counts_dev* counts, hipStream_t s) {
  if (!k) return;
  const Tiles t = tiles_of(k, kColenRows, a);
  hipLaunchKernelGGL(k_colen, dim3(t.grid), dim3(kScanThreads), 0, s, vals, fills, k, keys,
                     offsets, counts, a.state, a.status, t.count, a.host);
  const uint64_t lg = (k + kBlock - 1) / kBlock;
  hipLaunchKernelGGL(k_lengths, dim3(lg < 1024 ? (uint32_t)lg : 1024u), dim3(kBlock), 0, s,
                     offsets, lengths, counts, k);
}

}  // namespace wah
