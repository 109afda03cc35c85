// wah_kernels.hip -- gfx950 kernels of the WAH bitmap-index build.
//
// Fused build (what wahgpu_build and the batched builds run), for columns of
// uint32 values:
//   k_begin       zeroes the header and per-column state (and writes a single
//                 column's descriptor)
//   k_histogram   one read of the values: histograms of all four 8-bit
//                 digits, repeat rows, run counts per radix tile, the maximum;
//                 zeroing of look-back state
//   k_plan        per column: sort mode (pairs or runs), key width, digit
//                 offsets; passes whose digit is the same for every value are
//                 switched off (on the device, no host sync)
//   k_runcut      run mode: rows -> one (value, rid, literal bits) item per run
//   k_onesweep x4 stable LSD radix pass per active digit: LDS fetch-add (or
//                 ballot) ranking, LDS staging, decoupled look-back over tiles
//   k_tail        sorted items -> chunk ids, OR-merged literals, fills,
//                 zero-fill removal, word positions, keys and offsets
//   k_finish      per column: k, lengths[i] = offsets[i+1] - offsets[i], fault
// The staged kernels (what `phases` runs, one per reference stage) that are
// scans, and the scan / compaction primitives, are in wah_scan.hip.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "wah_scan.h"

namespace wah {

__global__ __launch_bounds__(kBlock) void k_fill32(uint32_t* __restrict__ p, uint64_t words,
                                                   uint32_t v) {
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < words;
       i += (uint64_t)gridDim.x * kBlock)
    p[i] = v;
}

// Zeroes the build header and the per-column histograms; a single-column
// build also gets its descriptor written here (no host-to-device copy).
__global__ __launch_bounds__(kBlock) void k_begin(Header* __restrict__ hdr,
                                                  ColState* __restrict__ cs, uint32_t cols_cap,
                                                  uint32_t* __restrict__ tile_runs,
                                                  uint32_t tiles_cap, DescHead* __restrict__ desc,
                                                  int inline_desc, Dims one_dims, Column one) {
  const uint64_t gt = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
  const uint64_t gs = (uint64_t)gridDim.x * kBlock;
  for (uint64_t i = gt; i < tiles_cap; i += gs) tile_runs[i] = 0;
  uint32_t* h = reinterpret_cast<uint32_t*>(hdr);
  for (uint64_t i = gt; i < sizeof(Header) / 4; i += gs) h[i] = 0;
  const uint64_t zw = (uint64_t)cols_cap * kColZeroWords;
  for (uint64_t i = gt; i < zw; i += gs) {
    const uint64_t c = i / kColZeroWords, w = i % kColZeroWords;
    reinterpret_cast<uint32_t*>(&cs[c])[w] = 0;
  }
  if (inline_desc && gt == 0) {
    desc->dims = one_dims;
    desc_cols(desc)[0] = one;
  }
}

// ---------------------------------------------------------------------------
// Histogram of all four 8-bit digits per column (reads the values once).
// Block b takes a contiguous range of 4096-value chunks, accumulates in LDS
// and folds into the column's histogram when the column changes.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void hist_flush(uint32_t* h, uint32_t* hr, uint32_t* s_max,
                                           uint32_t& vmax, ColState* col) {
  const int t = threadIdx.x;
  for (int d = 32; d >= 1; d >>= 1) {
    const uint32_t o = __shfl_xor(vmax, d, kWave);
    vmax = o > vmax ? o : vmax;
  }
  if ((t % kWave) == 0) s_max[t / kWave] = vmax;
  __syncthreads();
  for (int i = t; i < 1024; i += kBlock) {
    if (h[i]) atomicAdd(&col->hist[0][i], h[i]);
    if (hr[i]) atomicAdd(&col->rep[0][i], hr[i]);
    h[i] = 0;
    hr[i] = 0;
  }
  if (t == 0) {
    uint32_t m = 0;
    for (int i = 0; i < kWaves; ++i) m = s_max[i] > m ? s_max[i] : m;
    atomicMax(&col->maxval, m);
  }
  vmax = 0;
  __syncthreads();
}

// 8 waves per SIMD: the grid is sized for 8 resident blocks per CU
__global__ __launch_bounds__(kBlock, 8) void k_histogram(
    const uint32_t* __restrict__ values, const DescHead* __restrict__ desc,
    ColState* __restrict__ cs, uint32_t* __restrict__ status0,
    uint64_t* __restrict__ tail_status, uint32_t* __restrict__ tile_entries,
    uint32_t* __restrict__ tile_runs, uint32_t sort_tile, uint32_t* __restrict__ chunk_runs) {
  __shared__ uint32_t h[4 * 256];
  __shared__ uint32_t hr[4 * 256];
  __shared__ uint32_t s_max[kWaves];
  const int t = threadIdx.x;
  const Dims dims = desc->dims;
  const Column* cols = desc_cols(desc);
  for (int i = t; i < 1024; i += kBlock) h[i] = hr[i] = 0;
  // zero the look-back state the later kernels of the same index build use
  const uint64_t gthreads = (uint64_t)gridDim.x * kBlock;
  const uint64_t gt = (uint64_t)blockIdx.x * kBlock + t;
  const uint64_t s0 = (uint64_t)dims.sort_tiles * 256;
  for (uint64_t i = gt; i < s0; i += gthreads) status0[i] = 0;
  for (uint64_t i = gt; i < dims.tail_tiles; i += gthreads) {
    tail_status[i] = 0;
    tile_entries[i] = 0;
  }
  __syncthreads();

  const uint32_t per = (dims.hist_chunks + gridDim.x - 1) / gridDim.x;
  uint32_t c0 = blockIdx.x * per;
  const uint32_t c1 = c0 + per < dims.hist_chunks ? c0 + per : dims.hist_chunks;
  if (c0 >= c1) return;
  uint32_t col = find_segment(&cols[0].hist_chunk0, sizeof(Column) / 4, dims.ncols, c0);
  uint32_t col_end = col + 1 < dims.ncols ? cols[col + 1].hist_chunk0 : dims.hist_chunks;
  uint32_t vmax = 0;
  for (uint32_t c = c0; c < c1; ++c) {
    if (c >= col_end) {  // next column (block-uniform)
      hist_flush(h, hr, s_max, vmax, &cs[col]);
      col = find_segment(&cols[0].hist_chunk0, sizeof(Column) / 4, dims.ncols, c);
      col_end = col + 1 < dims.ncols ? cols[col + 1].hist_chunk0 : dims.hist_chunks;
    }
    const Column cd = cols[col];
    const uint64_t lo = (uint64_t)(c - cd.hist_chunk0) * kHistChunk;
    // as a 32-bit minimum (a column holds fewer than 2^30 rows): written as a
    // 64-bit compare and a select beside the branch on it, hipcc 7.2 selects
    // on a stale condition bit
    const uint32_t left = (uint32_t)(cd.n - lo);
    const uint32_t cnt = __builtin_elementwise_min(left, kHistChunk);
    const uint32_t* src = values + cd.off + lo;
    // row of src[i] is rid_base + lo + i; a row repeats its predecessor when
    // it is not the first of the column or of a chunk and has its value
    const uint32_t row0 = cd.rid_base + (uint32_t)lo;
    const uint32_t wv = __builtin_amdgcn_readfirstlane(t / kWave);
    const uint32_t w0 = wv * kWave * 4;  // the wave's first row of the chunk
    // Whole chunks and a column's last, partial one run the same code: rows
    // past the column take the value of the wave's first row (so they vary no
    // digit) and are left out of the counts.  A wave with no row does nothing.
    auto chunk = [&](auto full_tag) {
      constexpr bool FULL = decltype(full_tag)::value;
      // four 16-byte loads per thread (4-byte aligned ones do), and per wave
      // the value before each of its four 256-value spans, all issued before
      // any is used: one memory latency per chunk
      W4 q[4];
      if (FULL) {
#pragma unroll
        for (int u = 0; u < 4; ++u) q[u] = reinterpret_cast<const W4u*>(src)[u * kBlock + t];
      } else {  // one row at a time, past the end the last one: no branches
        // (opaque: the indices are formed here, not kept across whole chunks)
        const uint32_t end = cnt - 1u, t4 = 4u * opaque((uint32_t)t);
        auto at = [&](uint32_t i) -> uint32_t { return src[i < end ? i : end]; };
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const uint32_t i0 = t4 + (uint32_t)(u * kBlock * 4);
          q[u] = W4{at(i0), at(i0 + 1u), at(i0 + 2u), at(i0 + 3u)};
        }
      }
      // lane u < 4: the value before span u of the wave (one vector load)
      uint32_t wprev;
      {
        const uint32_t lu = lane_id();
        const uint32_t s0 = (lu * kBlock + wv * kWave) * 4;  // span's first index
        wprev = lu < 4u && lo + s0 > 0 && (FULL || s0 < cnt) ? src[(int64_t)s0 - 1] : 0u;
      }
      __builtin_amdgcn_sched_barrier(0);
      // The wave's 1024 rows of the chunk (4 spans of 256).  A digit the same
      // in all 1024 rows adds once (the high digits of small values); a digit
      // that varies adds once per span that holds a single value (inside a
      // run), and otherwise one LDS atomic per row.  Lane 0 adds from its own
      // values, so no per-span scalars stay live.  The repeat histograms are
      // added only when some row of the wave repeats its predecessor (a
      // wave-uniform branch), so columns without repeats carry no per-row
      // conditions on their atomics.
      const uint32_t f0 = __builtin_amdgcn_readfirstlane(q[0].x);
      uint32_t vm = 0xFFFFu;  // rows of the lane below the column's end: bit 4u + j
      if (!FULL) {
        vm = 0;
        const uint32_t t4 = 4u * opaque((uint32_t)t);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const uint32_t i0 = t4 + (uint32_t)(u * kBlock * 4);
          const uint32_t ok = i0 + 4 <= cnt ? 15u : i0 < cnt ? (1u << (cnt - i0)) - 1u : 0u;
          vm |= ok << (4 * u);
          q[u].x = ok & 1u ? q[u].x : f0;
          q[u].y = ok & 2u ? q[u].y : f0;
          q[u].z = ok & 4u ? q[u].z : f0;
          q[u].w = ok & 8u ? q[u].w : f0;
        }
      }
      // rows of span u of the wave, and of the wave
      auto span_rows = [&](int u) -> uint32_t {
        const uint32_t s0 = (uint32_t)(u * kBlock * 4) + w0;
        return FULL || cnt >= s0 + 4u * kWave ? 4u * kWave : cnt > s0 ? cnt - s0 : 0u;
      };
      const uint32_t rows = span_rows(0) + span_rows(1) + span_rows(2) + span_rows(3);
      uint32_t x = 0;    // bits in which a value of the lane differs from its span's first
      uint32_t fx = 0;   // bits in which a span's first value differs from f0
      uint32_t one = 0;  // bit u: span u holds a single value
      uint32_t rm = 0;   // repeat rows of the lane: bit 4u + j
      // row % 31 of q[u].x; spans are 1024 rows apart and 1024 = 33 * 31 + 1
      uint32_t m = (row0 + (uint32_t)t * 4u) % 31u;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        // lane l-1's last value (DPP wave shift); lane 0 the value before the span
        const uint32_t prev = lane_before(q[u].w, readlane(wprev, u));
        const uint32_t e[4] = {q[u].x, q[u].y, q[u].z, q[u].w};
        uint32_t mj = m;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          vmax = e[j] > vmax ? e[j] : vmax;
          const uint32_t pv = j == 0 ? prev : e[j - 1];
          const bool rep = lo + (uint32_t)(u * kBlock + t) * 4 + j > 0 && mj != 0u && e[j] == pv;
          rm |= rep ? 1u << (4 * u + j) : 0u;
          mj = mj == 30u ? 0u : mj + 1u;
        }
        m = m == 30u ? 0u : m + 1u;
        const uint32_t fu = __builtin_amdgcn_readfirstlane(e[0]);
        const uint32_t xu = (e[0] ^ fu) | (e[1] ^ fu) | (e[2] ^ fu) | (e[3] ^ fu);
        one |= ballot(xu != 0u) == 0 ? 1u << u : 0u;
        x |= xu;
        fx |= fu ^ f0;
      }
      if (!FULL) rm &= vm;
      // a bit varies over the 1024 rows iff it varies inside a span or
      // between the spans' first values
      const uint32_t vary = wave_or(x) | fx;
      // runs of the wave's rows, added to their radix tile and, where the cut
      // goes by chunks (see k_runcut), kept in the wave's word of the chunk's
      // four: a run-mode column's cut places its items from them.  The words
      // are the column's part of a literal buffer that nothing holds yet; a
      // wave without rows has none, so they end before the column's.  No
      // block barrier, so the waves of a block stream their chunks
      // independently.
      const uint32_t reps = readlane(wave_incl_add((uint32_t)__builtin_popcount(rm)), kWave - 1);
      if (lane_id() == 0) {
        if (dims.sort_tiles < kCutTiles)
          chunk_runs[cd.off + lo / (kHistChunk / 4) + wv] = rows - reps;
        if (rows != reps)
          atomicAdd(&tile_runs[cd.sort_tile0 + (uint32_t)(lo / sort_tile)], rows - reps);
      }
      if (vary == 0u) {
        // every row of the chunk holds f0 (inside a run): lane p adds the
        // wave's rows, and its repeat rows, to digit p's bin of f0
        const uint32_t lp = lane_id();
        if (lp < 4u) {
          const uint32_t bin = lp * 256u + ((f0 >> (8u * lp)) & 255u);
          atomicAdd(&h[bin], rows);
          if (reps) atomicAdd(&hr[bin], reps);
        }
        return;
      }
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        if (((vary >> (8 * p)) & 255u) == 0u) {
          if (lane_id() == 0) atomicAdd(&h[p * 256 + ((q[0].x >> (8 * p)) & 255u)], rows);
          continue;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const uint32_t e[4] = {q[u].x, q[u].y, q[u].z, q[u].w};
          if ((one >> u) & 1u) {
            if (lane_id() == 0) atomicAdd(&h[p * 256 + ((e[0] >> (8 * p)) & 255u)], span_rows(u));
          } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
              if (FULL || ((vm >> (4 * u + j)) & 1u))
                atomicAdd(&h[p * 256 + ((e[j] >> (8 * p)) & 255u)], 1u);
          }
        }
      }
      if (reps) {
        uint32_t rcu[4];  // repeats of each span
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          rcu[u] = 0;
#pragma unroll
          for (int j = 0; j < 4; ++j) rcu[u] += (uint32_t)__popcll(ballot((rm >> (4 * u + j)) & 1u));
        }
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          if (((vary >> (8 * p)) & 255u) == 0u) {
            if (lane_id() == 0) atomicAdd(&hr[p * 256 + ((q[0].x >> (8 * p)) & 255u)], reps);
            continue;
          }
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const uint32_t e[4] = {q[u].x, q[u].y, q[u].z, q[u].w};
            if ((one >> u) & 1u) {
              if (lane_id() == 0 && rcu[u]) atomicAdd(&hr[p * 256 + ((e[0] >> (8 * p)) & 255u)], rcu[u]);
            } else {
#pragma unroll
              for (int j = 0; j < 4; ++j)
                if ((rm >> (4 * u + j)) & 1u) atomicAdd(&hr[p * 256 + ((e[j] >> (8 * p)) & 255u)], 1u);
            }
          }
        }
      }
    };
    if (cnt == kHistChunk) chunk(std::true_type{});
    else if (w0 < cnt) chunk(std::false_type{});
  }
  hist_flush(h, hr, s_max, vmax, &cs[col]);
}

// After the histogram, per column: digit offsets and the pass plan (digits
// that are the same for every value of the column are skipped).  A kernel of
// its own so the histogram blocks need no device-scope fences (on gfx950
// each one writes back and invalidates the L2).
__global__ __launch_bounds__(kBlock) void k_plan(const DescHead* __restrict__ desc,
                                                 ColState* __restrict__ cs, Header* __restrict__ hdr,
                                                 uint32_t* __restrict__ tile_runs,
                                                 wahgpu_counts_dev* __restrict__ counts,
                                                 int force_pair, uint32_t sort_tile,
                                                 WideState* __restrict__ wide) {
  __shared__ uint64_t s_scan[kWaves];
  __shared__ int s_trivial[4];
  __shared__ uint32_t s_wide;  // 1 + wide slot of a column that takes wide digits
  const int t = threadIdx.x, l = t % kWave;
  const int w = __builtin_amdgcn_readfirstlane(t / kWave);
  const uint32_t ncols = desc->dims.ncols;
  for (uint32_t c = blockIdx.x; c < ncols; c += gridDim.x) {
    const uint64_t n = desc_cols(desc)[c].n;
    ColState* col = &cs[c];
    // Wave p takes digit p, lane l its bins 4l .. 4l + 3: the digits' scans
    // run side by side, with one barrier after them (one after another over
    // the block, with two barriers each, they made the kernel 7 us of a
    // build of 2^20 rows).
    const uint4 hq = reinterpret_cast<const uint4*>(col->hist[w])[l];
    const uint4 rq = reinterpret_cast<const uint4*>(col->rep[w])[l];
    // every digit counts every repeat row once
    const uint32_t reps = readlane(wave_incl_add(rq.x + rq.y + rq.z + rq.w), kWave - 1);
    // Run mode when it sorts under 2/3 of the rows (an item moves 12 bytes
    // per pass, a pair 8).
    const uint64_t runs = n - reps;
    const bool run_mode = !force_pair && n > 0 && 3 * runs < 2 * n;
    const uint64_t items = run_mode ? runs : n;
    {
      const uint32_t h[4] = {hq.x - (run_mode ? rq.x : 0u), hq.y - (run_mode ? rq.y : 0u),
                             hq.z - (run_mode ? rq.z : 0u), hq.w - (run_mode ? rq.w : 0u)};
      const uint32_t sum = h[0] + h[1] + h[2] + h[3];
      uint4 ex;
      ex.x = wave_incl_add(sum) - sum;
      ex.y = ex.x + h[0];
      ex.z = ex.y + h[1];
      ex.w = ex.z + h[2];
      reinterpret_cast<uint4*>(col->digit_offset[w])[l] = ex;
      bool all = false;  // one digit holds every item
#pragma unroll
      for (int i = 0; i < 4; ++i) all |= (uint64_t)h[i] == items;
      const bool trivial = ballot(all) != 0;
      if (l == 0) s_trivial[w] = trivial;
    }
    if (run_mode) {
      // where each radix tile's runs go: exclusive prefix of the runs per tile
      const Column cd = desc_cols(desc)[c];
      uint32_t* tr = tile_runs + cd.sort_tile0;
      const uint32_t tiles = sort_tiles_of(n, sort_tile);
      // thread t scans a strip of consecutive tiles; a strip of up to 64
      // tiles (2^28 rows in 16384-row tiles) stays in registers between the
      // sum and the prefix, longer ones are read twice in batches of 16
      const uint32_t per = (tiles + kBlock - 1) / kBlock;
      const uint32_t s0 = t * per < tiles ? t * per : tiles;
      const uint32_t s1 = s0 + per < tiles ? s0 + per : tiles;
      constexpr uint32_t kStrip = 64;
      if (per <= kStrip) {  // block-uniform
        uint32_t x[kStrip];
        uint64_t sum = 0;
#pragma unroll
        for (uint32_t i = 0; i < kStrip; ++i) x[i] = s0 + i < s1 ? tr[s0 + i] : 0u;
#pragma unroll
        for (uint32_t i = 0; i < kStrip; ++i) sum += x[i];
        uint64_t tot;
        uint64_t run = block_exclusive<OpAdd>(sum, s_scan, &tot);
#pragma unroll
        for (uint32_t i = 0; i < kStrip; ++i) {
          if (s0 + i < s1) tr[s0 + i] = (uint32_t)run;
          run += x[i];
        }
      } else {
        uint64_t sum = 0;
        for (uint32_t b = s0; b < s1; b += 16) {
          uint32_t x[16];
#pragma unroll
          for (int i = 0; i < 16; ++i) x[i] = b + i < s1 ? tr[b + i] : 0u;
#pragma unroll
          for (int i = 0; i < 16; ++i) sum += x[i];
        }
        uint64_t tot;
        uint64_t run = block_exclusive<OpAdd>(sum, s_scan, &tot);
        for (uint32_t b = s0; b < s1; b += 16) {
          uint32_t x[16];
#pragma unroll
          for (int i = 0; i < 16; ++i) x[i] = b + i < s1 ? tr[b + i] : 0u;
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            if (b + i < s1) tr[b + i] = (uint32_t)run;
            run += x[i];
          }
        }
      }
    }
    __syncthreads();
    if (t == 0) {
      uint32_t a = 0;
      for (int p = 0; p < 4; ++p)
        if (n > 0 && !s_trivial[p]) col->shift[a++] = 8u * p;
      for (uint32_t q = a; q < 4; ++q) col->shift[q] = 0;
      // Wide digits when they take fewer passes: the key's significant bits
      // split as evenly as possible into passes of at most kWideBits.
      const Column cw = desc_cols(desc)[c];
      const uint32_t bits = col->maxval ? 32u - (uint32_t)__clz(col->maxval) : 0u;
      const uint32_t aw = (bits + kWideBits - 1) / kWideBits;
      const bool wide = cw.wide_slot != 0u && !run_mode && !force_pair && n >= kWideMinValues &&
                        aw < a;
      col->wide = wide ? 1u : 0u;
      col->wide_slot = wide ? cw.wide_slot - 1u : 0u;
      s_wide = wide ? cw.wide_slot : 0u;
      if (wide) {
        uint32_t at = 0;
        for (uint32_t i = 0; i < (uint32_t)kWidePasses; ++i) {
          const uint32_t b = i < aw ? bits / aw + (i < bits % aw ? 1u : 0u) : 0u;
          col->wbits[i] = b;
          col->wshift[i] = at;
          at += b;
        }
        a = aw;
      }
      col->num_active = a;
      col->mode = run_mode ? kModeRun : kModePair;
      // keys below 2^16 travel as 16-bit words from the first pass's output
      // on (the stage API reads 32-bit keys)
      col->narrow = !force_pair && a > 0 && col->maxval < 65536u;
      col->items = (uint32_t)items;
      // pair mode: values, then A, B, A, B; run mode: the cut writes B
      if (run_mode) col->final_buf = (a % 2) ? kBufA : kBufB;
      else col->final_buf = (a == 0) ? kBufValues : ((a - 1) % 2 == 0 ? kBufA : kBufB);
      if (a) atomicMax(wide ? &hdr->max_wide : &hdr->max_active[run_mode ? 1 : 0], a);
      if (n) atomicAdd(&hdr->mode_cols[run_mode ? 1 : 0], 1u);
      wahgpu_counts_dev z;
      z.k = 0; z.length = 0; z.keycnt = 0;
      z.bound = col->maxval; z.passes = a; z.fault = 0;
      z.mode = run_mode ? kModeRun : wide ? kModeWideReport : kModePair;
      counts[desc_cols(desc)[c].index] = z;
    }
    __syncthreads();
    if (s_wide) {  // the wide histograms start at zero (k_whist adds to them)
      uint32_t* hw = wide[s_wide - 1u].hist[0];
      for (uint32_t i = t; i < (uint32_t)kWidePasses * kWideBins; i += kBlock) hw[i] = 0;
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Run mode, before the radix launches: cuts each run-mode column into runs
// (a row starts one unless it repeats its predecessor's value inside the
// same 31-row chunk) and writes one item per run, in row order, to buffer B:
// value, rid of its first row, literal bits of its rows.  An ordered stream
// compaction without look-back: the histogram counted the runs of each radix
// tile, k_plan turned the counts into offsets, and a block takes whole units
// (static grid stride) and walks a unit in steps of one chunk of the
// histogram with a running offset.  A unit is a radix tile where there are
// kCutTiles or more: one for every block that runs.  With fewer, blocks that
// walk a 16384-row tile in four steps leave the chip idle (the cut of 128
// columns of 2^17 rows, and of one of 2^20, took 30 us); there a unit is one
// chunk, placed by its tile's offset and the runs that the histogram kept for
// the tile's earlier chunks (15 us; 128 columns of 2^17 rows build in 481 us,
// 492 before).  Chunks everywhere cost a column of 2^28 rows 10 us more.
// Lane t owns 16 consecutive rows
// (16-byte loads); a run is at most 31 rows, so the run of a lane's last
// start ends within the next two lanes (or the next wave's first two, or
// the rows past the step, exchanged in LDS).  Items are staged in LDS and
// stored contiguously, one array at a time.
// ---------------------------------------------------------------------------
constexpr int kCutRows = 16;                    // rows per lane
constexpr int kCutStep = kBlock * kCutRows;     // rows per block step
static_assert(kCutStep == (int)kHistChunk, "a chunk of the histogram per block step");
__global__ __launch_bounds__(kBlock, 8) void k_runcut(
    const uint32_t* __restrict__ values, uint32_t* __restrict__ keysB,
    uint32_t* __restrict__ ridsB, uint32_t* __restrict__ litsB,
    const DescHead* __restrict__ desc, const ColState* __restrict__ cs,
    Header* __restrict__ hdr, const uint32_t* __restrict__ tile_runs, uint32_t sort_tile,
    const uint32_t* __restrict__ chunk_runs) {
  constexpr int R = kCutRows;
  constexpr uint32_t kAll = (1u << R) - 1u;
  __shared__ uint32_t s_stage[kCutStep];
  __shared__ uint32_t s_wsum[kWaves];
  __shared__ uint32_t s_wlead[kWaves + 1];  // rows before the first stop of wave w; [kWaves]: past the step
  const Dims dims = desc->dims;
  const Column* cols = desc_cols(desc);
  const int t = threadIdx.x, l = t % kWave;
  const int w = __builtin_amdgcn_readfirstlane(t / kWave);  // scalar: per-wave LDS addresses
  if (hdr->mode_cols[1] == 0) return;  // no run-mode column
  const bool whole = dims.sort_tiles >= kCutTiles;
  const uint32_t units = whole ? dims.sort_tiles : dims.hist_chunks;
  const uint32_t unit_rows = whole ? sort_tile : kHistChunk;
  const uint32_t* unit0 = whole ? &cols[0].sort_tile0 : &cols[0].hist_chunk0;
  for (uint32_t u = blockIdx.x; u < units; u += gridDim.x) {
    const uint32_t c = find_segment(unit0, sizeof(Column) / 4, dims.ncols, u);
    const ColState* col = &cs[c];
    if (col->mode != kModeRun) continue;  // block-uniform, no LDS touched
    const Column cd = cols[c];
    // column-local rows fit 32 bits (a column holds fewer than 2^30)
    const uint32_t n = (uint32_t)cd.n;
    const uint32_t t0 = (u - (whole ? cd.sort_tile0 : cd.hist_chunk0)) * unit_rows;
    const uint32_t t1 = t0 + unit_rows < n ? t0 + unit_rows : n;
    const uint32_t* vp = values + cd.off;
    const uint32_t items = col->items;
    // runs of the column's earlier rows: those before the radix tile, and the
    // words of the tile's earlier chunks (a lane a word: no tile has more
    // than 64)
    const uint32_t tlo = t0 - t0 % sort_tile;
    uint32_t off = tile_runs[cd.sort_tile0 + t0 / sort_tile];
    if (tlo != t0) {  // block-uniform
      const bool in = (uint32_t)l < (t0 - tlo) / (kHistChunk / 4);
      const uint32_t x = in ? chunk_runs[cd.off + tlo / (kHistChunk / 4) + l] : 0u;
      off += readlane(wave_incl_add(x), kWave - 1);
    }
    for (uint32_t lo = t0; lo < t1; lo += kCutStep) {
      const uint32_t j0 = lo + (uint32_t)t * R;  // the lane's first row
      const uint32_t nv = t1 > j0 ? (t1 - j0 < (uint32_t)R ? t1 - j0 : (uint32_t)R) : 0u;
      uint32_t v[R];
      if (lo + kCutStep <= t1) {
#pragma unroll
        for (int q = 0; q < R / 4; ++q) {
          const W4 x = reinterpret_cast<const W4u*>(vp + j0)[q];
          v[4 * q] = x.x; v[4 * q + 1] = x.y; v[4 * q + 2] = x.z; v[4 * q + 3] = x.w;
        }
      } else {
#pragma unroll
        for (int i = 0; i < R; ++i) v[i] = (uint32_t)i < nv ? vp[j0 + i] : 0u;
      }
      // predecessor of the lane's first row: lane l-1's last, or for lane 0
      // the row before the wave (one load per wave)
      uint32_t pv;
      {
        const uint32_t gw = lo + (uint32_t)(w * kWave * R);
        const uint32_t p0 = gw > 0 && gw <= n ? vp[gw - 1] : 0u;
        pv = (uint32_t)__builtin_amdgcn_update_dpp((int)p0, (int)v[R - 1], 0x138, 0xF, 0xF, false);
      }
      const uint32_t m0 = (cd.rid_base + j0) % 31u;  // row % 31 of the lane's first row
      // Run starts, without branches: a row starts a run when it differs
      // from its predecessor, begins a chunk (row % 31 == 0: at most one of
      // the lane's R < 31 rows, the (31 - m0) % 31-th) or is the column's
      // first row; rows past the column's end start nothing.
      uint32_t sm;
      {
        const uint32_t ci = m0 == 0u ? 0u : 31u - m0;
        sm = (ci < (uint32_t)R ? 1u << ci : 0u) | (j0 == 0u ? 1u : 0u);
#pragma unroll
        for (int i = 0; i < R; ++i) {
          const uint32_t prev = i ? v[i - 1] : pv;
          sm |= (v[i] != prev ? 1u : 0u) << i;
        }
        sm &= nv >= (uint32_t)R ? kAll : (1u << nv) - 1u;
      }
      const uint32_t stops = sm | (~0u << nv & kAll);
      const uint32_t lead = stops ? (uint32_t)__builtin_ctz(stops) : (uint32_t)R;
      const uint32_t cnt = (uint32_t)__builtin_popcount(sm);
      const uint32_t inc = wave_incl_add(cnt);
      if (l == kWave - 1) s_wsum[w] = inc;
      const uint64_t hsm = ballot(stops != 0u);
      const uint32_t L1 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)lead, 0x130, 0xF, 0xF, false);
      const uint32_t L2 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)L1, 0x130, 0xF, 0xF, false);
      {
        // rows before the wave's first stop (within its first two lanes)
        const uint32_t l0 = readlane(lead, 0), l1 = readlane(lead, 1);
        if (l == 0) s_wlead[w] = (hsm & 1ull) ? l0 : (uint32_t)R + l1;
      }
      if (w == kWaves - 1) {  // rows past the step: where its last run ends
        const uint32_t g = lo + (uint32_t)kCutStep + l;
        const bool valid = l < 32 && g < n;
        const uint32_t x = valid ? vp[g] : 0u;
        const uint32_t last = readlane(v[R - 1], kWave - 1);
        const uint32_t px = (uint32_t)__builtin_amdgcn_update_dpp((int)last, (int)x, 0x138, 0xF, 0xF, false);
        const bool st = !valid | ((cd.rid_base + g) % 31u == 0u) | (x != px);  // no branches
        const uint64_t sb = ballot(st);  // lanes 32.. always stop
        if (l == 0) s_wlead[kWaves] = (uint32_t)__builtin_ctzll(sb);
      }
      __syncthreads();
      uint32_t woff, tot;
      {
        const uint32_t x = l < kWaves ? s_wsum[l] : 0u;
        const uint32_t xi = wave_incl_add(x);
        woff = readlane(xi - x, __builtin_amdgcn_readfirstlane(w));
        tot = readlane(xi, kWaves - 1);
      }
      // rows after the lane that the run of its last start covers
      const uint32_t nw = s_wlead[w + 1];
      uint32_t cont;
      if (l == kWave - 1) cont = nw;
      else if ((hsm >> (l + 1)) & 1ull) cont = L1;
      else if (l == kWave - 2) cont = (uint32_t)R + nw;
      else cont = (uint32_t)R + L2;
      if (nv < (uint32_t)R) cont = 0;  // the run ends with the rows
      const uint32_t k0 = woff + inc - cnt;  // items of the step before the lane
      if (off + tot > items) {
        if (t == 0) atomicOr(&hdr->fault, 2u);
        return;  // block-uniform: the chunks' runs disagree with the items
      }
      // the item of start i: round 0 its value, 1 its rid, 2 its literal bits
      auto item = [&](int round, int i) -> uint32_t {
        if (round == 0) return v[i];
        if (round == 1) return cd.rid_base + j0 + i;
        const uint32_t rest = stops >> (i + 1);
        const uint32_t len = rest ? (uint32_t)__builtin_ctz(rest) + 1u : (uint32_t)(R - i) + cont;
        const uint32_t mi = m0 + i >= 31u ? m0 + i - 31u : m0 + i;
        return ((len >= 32u ? 0u : (1u << len)) - 1u) << mi;
      };
      if (3 * tot <= (uint32_t)kCutStep) {
        // few runs: the three arrays staged together, one round
        uint32_t k = k0;
#pragma unroll
        for (int i = 0; i < R; ++i) {
          if ((sm >> i) & 1u) {
            s_stage[k] = item(0, i);
            s_stage[tot + k] = item(1, i);
            s_stage[2 * tot + k] = item(2, i);
            ++k;
          }
        }
        __syncthreads();
        for (uint32_t j = t; j < 3 * tot; j += kBlock) {
          const uint32_t r = j / tot, q = j - r * tot;  // tot > 0 here
          uint32_t* dst = (r == 0 ? keysB : r == 1 ? ridsB : litsB) + cd.off + off;
          dst[q] = s_stage[j];
        }
        __syncthreads();
      } else {
        // three rounds through LDS: values, rids, literal bits
#pragma unroll 1
        for (int round = 0; round < 3; ++round) {
          uint32_t k = k0;
#pragma unroll
          for (int i = 0; i < R; ++i)
            if ((sm >> i) & 1u) s_stage[k++] = item(round, i);
          __syncthreads();
          uint32_t* dst = (round == 0 ? keysB : round == 1 ? ridsB : litsB) + cd.off + off;
          for (uint32_t j = t; j < tot; j += kBlock) dst[j] = s_stage[j];
          __syncthreads();
        }
      }
      off += tot;
    }
  }
}

// Ranking of a radix pass.  kRankMatch: peers = lanes with the same digit
// from 8 ballots, rank = peers below + earlier count (stable by
// construction, ~50 VALU per key).  kRankAtomic: one LDS fetch-add per key on
// the wave's digit counter; the returned counts are a stable rank because the
// LDS serializes the lanes of one instruction that hit one address in lane
// order -- not a documented guarantee, so a context takes this path only
// after k_rank_selftest has checked it on the device.
constexpr int kRankMatch = 0;
constexpr int kRankAtomic = 1;

// Checks on this device that LDS fetch-adds of one wave instruction return,
// for lanes on the same address, counts in increasing lane order: many
// address patterns (1 to 64 lanes per address, every lane order), repeated.
// *ok = 1 if every check held.
__global__ __launch_bounds__(256) void k_rank_selftest(uint32_t* ok) {
  __shared__ uint32_t cnt[4][256];
  const int t = threadIdx.x, w = t / kWave, l = t % kWave;
  uint32_t good = 1;
  for (uint32_t round = 0; round < 512; ++round) {
    for (int i = t; i < 4 * 256; i += 256) (&cnt[0][0])[i] = 0;
    __syncthreads();
    // address pattern of this round: few to many distinct digits
    const uint32_t h = (uint32_t)l * 2654435761u ^ (round * 40503u + (uint32_t)w * 977u);
    const uint32_t span = 1u + (round % 64u);
    const uint32_t d = (h >> 7) % span;
    uint32_t prev = 0;
    for (int rep = 0; rep < 4; ++rep) {
      const uint32_t r = atomicAdd(&cnt[w][d], 1u);
      uint64_t peers = ballot(true);
#pragma unroll
      for (int b = 0; b < 8; ++b) {
        const bool bit = (d >> b) & 1u;
        const uint64_t bb = ballot(bit);
        peers &= bit ? bb : ~bb;
      }
      const uint32_t expect = (uint32_t)rep * (uint32_t)__popcll(peers) + mbcnt(peers);
      if (r != expect || (rep > 0 && r <= prev)) good = 0;
      prev = r;
    }
    __syncthreads();
  }
  if (!good) atomicAnd(ok, 0u);
}

// ---------------------------------------------------------------------------
// Launch `a` of the stable LSD radix sort runs each column's a-th active pass
// (Onesweep-style): launch 0 reads the values (rids implicit) into buffer A,
// then A -> B, B -> A, A -> B.  Tile = THREADS x ITEMS keys of one column;
// wave w ranks keys [w*64*ITEMS, +64*ITEMS) of the tile in (item, lane)
// order, which is the input order, so equal digits keep their relative order
// (stability).  Keys and then rids are staged in one LDS buffer in digit
// order and written out in runs per digit.  Run mode moves (key, rid,
// literal bits) items the run cut wrote to B: launch 0 reads B.
// ---------------------------------------------------------------------------
// MODES 0: the tiles of the pair-mode columns; 1: of the run-mode columns; 2:
// of the former and then of the latter in one launch, where a mode without an
// a-th pass costs a scalar load.  A launch per mode leaves half the radix
// launches of a single column with nothing to do, 4 to 5 us each (2^20 rows
// 77 us, in one launch 70); with both bodies in one kernel fewer scalar
// registers are left per body, and from 2^24 rows on that costs more (2^28
// rows: 2835 us, in one launch 2863).
template <int THREADS, int ITEMS, int RANK, int MODES>
__global__ __launch_bounds__(THREADS, sort_waves_per_eu(ITEMS)) void k_onesweep(
    uint32_t a, const uint32_t* __restrict__ values, uint32_t* keysA, uint32_t* ridsA,
    uint32_t* keysB, uint32_t* ridsB, uint32_t* litsA, uint32_t* litsB,
    const DescHead* __restrict__ desc, const ColState* __restrict__ cs, Header* __restrict__ hdr,
    uint32_t* status_base, uint64_t status_stride, uint32_t lanes) {
  constexpr int TILE = THREADS * ITEMS;
  constexpr int WAVES = THREADS / kWave;
  static_assert(THREADS >= 256 && THREADS % 256 == 0, "one thread per digit");
  static_assert(TILE <= 65536, "LDS slots packed in 16 bits");
  __shared__ uint32_t s_stage[TILE];
  __shared__ uint32_t s_wcnt[WAVES][256];
  __shared__ uint32_t s_excl[256];
  __shared__ uint32_t s_glob[256];
  __shared__ uint32_t s_dsum[4];
  __shared__ uint32_t s_tile;
  if constexpr (MODES != 1) {
    constexpr bool RUN = false;
#include "radix_tiles.inl"
  }
  if constexpr (MODES == 2) __syncthreads();  // the last draw is read before the next mode's first
  if constexpr (MODES != 0) {
    constexpr bool RUN = true;
#include "radix_tiles.inl"
  }
}

#ifndef WAH_WIDE_LOOKAHEAD  // predecessors per look-back round trip of the wide passes
#define WAH_WIDE_LOOKAHEAD 8
#endif

// ---------------------------------------------------------------------------
// Wide digits (pair-mode columns that k_plan marked wide).
//
// k_whist: histograms of the column's wide digits over its values (the
// 8-bit ones of k_histogram do not give them), in LDS per block, added to
// the column's WideState; and zero look-back state for the first wide pass.
// Blocks take contiguous ranges of the 4096-value histogram chunks, as in
// k_histogram, and skip the chunks of other columns.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_whist(const uint32_t* __restrict__ values,
                                                  const DescHead* __restrict__ desc,
                                                  const ColState* __restrict__ cs,
                                                  WideState* __restrict__ ws,
                                                  uint32_t* __restrict__ wstatus0) {
  __shared__ uint32_t h[kWidePasses * kWideBins];
  const int t = threadIdx.x;
  const Dims dims = desc->dims;
  const Column* cols = desc_cols(desc);
  for (uint32_t tile = blockIdx.x; tile < dims.wide_tiles; tile += gridDim.x) {
    const uint32_t c = find_segment(&cols[0].wide_tile0, sizeof(Column) / 4, dims.ncols, tile);
    if (!cs[c].wide) continue;  // block-uniform
    uint32_t* st = wstatus0 + (uint64_t)tile * kWideBins;
    for (uint32_t i = t; i < kWideBins; i += kBlock) st[i] = 0;
  }
  for (uint32_t i = t; i < (uint32_t)kWidePasses * kWideBins; i += kBlock) h[i] = 0;
  __syncthreads();
  const uint32_t per = (dims.hist_chunks + gridDim.x - 1) / gridDim.x;
  const uint32_t c0 = blockIdx.x * per;
  const uint32_t c1 = c0 + per < dims.hist_chunks ? c0 + per : dims.hist_chunks;
  uint32_t col = c0 < c1 ? find_segment(&cols[0].hist_chunk0, sizeof(Column) / 4, dims.ncols, c0)
                         : 0u;
  bool counted = false;  // h holds counts of column `col`
  auto flush = [&]() {
    __syncthreads();
    uint32_t* dst = ws[cs[col].wide_slot].hist[0];
    for (uint32_t i = t; i < (uint32_t)kWidePasses * kWideBins; i += kBlock) {
      if (h[i]) atomicAdd(&dst[i], h[i]);
      h[i] = 0;
    }
    __syncthreads();
    counted = false;
  };
  for (uint32_t c = c0; c < c1;) {
    const uint32_t col_end = col + 1 < dims.ncols ? cols[col + 1].hist_chunk0 : dims.hist_chunks;
    if (c >= col_end) {  // next column (block-uniform)
      if (counted) flush();
      col = find_segment(&cols[0].hist_chunk0, sizeof(Column) / 4, dims.ncols, c);
      continue;
    }
    const ColState* st = &cs[col];
    if (!st->wide) {  // skip the rest of this column's chunks
      c = col_end;
      continue;
    }
    counted = true;
    const Column cd = cols[col];
    const uint64_t lo = (uint64_t)(c - cd.hist_chunk0) * kHistChunk;
    const uint32_t cnt = cd.n - lo < kHistChunk ? (uint32_t)(cd.n - lo) : kHistChunk;
    const uint32_t* src = values + cd.off + lo;
    const uint32_t np = st->num_active;
    const uint32_t sh0 = st->wshift[0], sh1 = st->wshift[1], sh2 = st->wshift[2];
    const uint32_t m0 = (1u << st->wbits[0]) - 1u, m1 = (1u << st->wbits[1]) - 1u,
                   m2 = (1u << st->wbits[2]) - 1u;
    auto add = [&](uint32_t v) {
      atomicAdd(&h[(v >> sh0) & m0], 1u);
      if (np > 1) atomicAdd(&h[kWideBins + ((v >> sh1) & m1)], 1u);
      if (np > 2) atomicAdd(&h[2 * kWideBins + ((v >> sh2) & m2)], 1u);
    };
    if (cnt == kHistChunk && ((uintptr_t)src % 16) == 0) {
      // four 16-byte loads per thread, issued before any is counted
      const uint4* v4 = reinterpret_cast<const uint4*>(src);
      uint4 q[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) q[u] = v4[u * kBlock + t];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        add(q[u].x);
        add(q[u].y);
        add(q[u].z);
        add(q[u].w);
      }
    } else {
      for (uint32_t i = t; i < cnt; i += kBlock) add(src[i]);
    }
    ++c;
  }
  if (counted) flush();
}

// k_wplan: each wide column's digit histograms -> exclusive prefixes (the
// first row of each digit's keys in the column), in place.
__global__ __launch_bounds__(kBlock) void k_wplan(const DescHead* __restrict__ desc,
                                                  const ColState* __restrict__ cs,
                                                  WideState* __restrict__ ws) {
  __shared__ uint64_t s_scan[kWaves];
  constexpr uint32_t kPer = kWideBins / kBlock;
  const int t = threadIdx.x;
  const uint32_t ncols = desc->dims.ncols;
  for (uint32_t c = blockIdx.x; c < ncols; c += gridDim.x) {
    const ColState* col = &cs[c];
    if (!col->wide) continue;  // block-uniform
    for (uint32_t p = 0; p < col->num_active; ++p) {
      uint32_t* hp = ws[col->wide_slot].hist[p] + (uint32_t)t * kPer;
      uint32_t x[kPer];
      uint64_t sum = 0;
#pragma unroll
      for (uint32_t k = 0; k < kPer; ++k) {
        x[k] = hp[k];
        sum += x[k];
      }
      uint64_t total;
      uint64_t ex = block_exclusive<OpAdd>(sum, s_scan, &total);
#pragma unroll
      for (uint32_t k = 0; k < kPer; ++k) {
        hp[k] = (uint32_t)ex;
        ex += x[k];
      }
    }
  }
}

// k_wsweep: launch `a` sorts the a-th wide digit of every wide column, one
// tile of kWideTile pairs at a time, as k_onesweep does with 8-bit digits:
// rank in LDS, publish the tile's digit counts, look back for the counts of
// the tiles before it, scatter through LDS.  The 2048 digits take two 16-bit
// counters per LDS word (a wave ranks at most 64 x kWideItems keys and a
// tile holds 8192), and thread t owns digits 4t .. 4t + 3.
template <int RANK>
__global__ __launch_bounds__(kWideThreads, sort_waves_per_eu(kWideItems)) void k_wsweep(
    uint32_t a, const uint32_t* __restrict__ values, uint32_t* keysA, uint32_t* ridsA,
    uint32_t* keysB, uint32_t* ridsB, const DescHead* __restrict__ desc,
    const ColState* __restrict__ cs, const WideState* __restrict__ ws, Header* __restrict__ hdr,
    uint32_t* status_base, uint64_t status_stride, uint32_t lanes) {
  constexpr int THREADS = kWideThreads, ITEMS = kWideItems, TILE = (int)kWideTile;
  constexpr int WAVES = THREADS / kWave;
  constexpr int DPT = (int)kWideBins / THREADS;  // digits per thread
  static_assert(DPT == 4, "two counter words per thread and wave");
  static_assert(TILE <= 65535, "16-bit counters and slots");
  __shared__ uint32_t s_stage[TILE];
  __shared__ uint32_t s_cnt[WAVES][kWideBins / 2];
  __shared__ uint32_t s_glob[kWideBins];
  __shared__ uint32_t s_wsum[WAVES];
  __shared__ uint32_t s_tilen;
  __shared__ uint32_t s_tile;

  const bool implicit = a == 0;
  const uint32_t* src_keys = implicit ? values : ((a % 2) ? keysA : keysB);
  const uint32_t* src_rids = (a % 2) ? ridsA : ridsB;
  uint32_t* dst_keys = (a % 2) ? keysB : keysA;
  uint32_t* dst_rids = (a % 2) ? ridsB : ridsA;
  uint32_t* status = status_base + (uint64_t)(a % 2) * status_stride;
  uint32_t* status_next = status_base + (uint64_t)(1u - a % 2) * status_stride;
  uint32_t* fault = &hdr->fault;
  const Dims dims = desc->dims;
  const Column* cols = desc_cols(desc);
  const int t = threadIdx.x, l = t % kWave;
  const int w = __builtin_amdgcn_readfirstlane(t / kWave);
  if (hdr->max_wide <= a) return;  // no column has an a-th wide pass
  uint32_t* counter = hdr->tiles[kCounterWide + a];

  uint32_t iter = 0;
  for (;;) {
    for (int i = t; i < WAVES * (int)kWideBins / 2; i += THREADS) (&s_cnt[0][0])[i] = 0;
    const uint32_t tile = __builtin_amdgcn_readfirstlane(
        next_tile(counter, lanes, &s_tile, iter, tile_group(dims.wide_tiles, gridDim.x, lanes, WAH_SORT_TILE_GROUP)));
    if (tile >= dims.wide_tiles) break;
    const uint32_t c = find_segment(&cols[0].wide_tile0, sizeof(Column) / 4, dims.ncols, tile);
    const ColState* col = &cs[c];
    const Column cd = cols[c];
    const uint32_t first = cd.wide_tile0;
    const uint64_t base = (uint64_t)(tile - first) * TILE;  // column-local
    const uint64_t n = cd.n;
    if (!col->wide || col->num_active <= a || base >= n) {
      __syncthreads();  // s_tile is read by every wave before it is rewritten
      continue;
    }
    const uint32_t shift = col->wshift[a];
    const uint32_t dmask = (1u << col->wbits[a]) - 1u;
    const uint32_t* goff = ws[col->wide_slot].hist[a];
    const bool narrow = col->narrow != 0u, src_narrow = narrow && !implicit;
#pragma unroll
    for (int k = 0; k < DPT; ++k) status_next[(uint64_t)tile * kWideBins + DPT * t + k] = 0;
    const uint64_t wbase = base + (uint64_t)w * kWave * ITEMS + l;
    auto sweep = [&](auto full_tag) {
      constexpr bool FULL = decltype(full_tag)::value;
      uint32_t key[ITEMS], rank[ITEMS];
      const uint32_t nvalid =
          FULL ? (uint32_t)ITEMS * kWave : (uint32_t)(n > wbase ? n - wbase : 0);
      if (src_narrow) {
        const uint16_t* kp = reinterpret_cast<const uint16_t*>(src_keys + cd.off) + wbase;
#pragma unroll
        for (int i = 0; i < ITEMS; ++i)
          key[i] = FULL || (uint32_t)(i * kWave) < nvalid ? (uint32_t)kp[i * kWave] : 0u;
      } else {
        const uint32_t* kp = src_keys + cd.off + wbase;
#pragma unroll
        for (int i = 0; i < ITEMS; ++i)
          key[i] = FULL || (uint32_t)(i * kWave) < nvalid ? kp[i * kWave] : 0u;
      }
      uint32_t part = 0;
#pragma unroll
      for (int i = 0; i < ITEMS; ++i)
        part |= (FULL || (uint32_t)(i * kWave) < nvalid ? 1u : 0u) << i;
#pragma unroll
      for (int i = 0; i < ITEMS; ++i) {
        if (FULL || ((part >> i) & 1u)) {
          const uint32_t d = (key[i] >> shift) & dmask;
          const uint32_t hs = 16u * (d & 1u);
          if (RANK == kRankAtomic) {
            rank[i] = (atomicAdd(&s_cnt[w][d >> 1], 1u << hs) >> hs) & 0xFFFFu;
          } else {
            uint64_t peers = ballot(true);
#pragma unroll
            for (int b = 0; b < kWideBits; ++b) {
              const bool bit = (d >> b) & 1u;
              const uint64_t bb = ballot(bit);
              peers &= bit ? bb : ~bb;
            }
            const uint32_t cnt = (uint32_t)__popcll(peers);
            const uint32_t below = mbcnt(peers);
            const uint32_t prior = (s_cnt[w][d >> 1] >> hs) & 0xFFFFu;
            rank[i] = prior + below;
            // two digits share a word: add, do not store
            if (below == cnt - 1) atomicAdd(&s_cnt[w][d >> 1], cnt << hs);
          }
        }
      }
      __syncthreads();
      // digits 4t .. 4t + 3: wave prefixes and tile totals
      uint32_t tot[DPT] = {0u, 0u, 0u, 0u};
#pragma unroll
      for (int i = 0; i < WAVES; ++i) {
        const uint32_t w0 = s_cnt[i][2 * t], w1 = s_cnt[i][2 * t + 1];
        s_cnt[i][2 * t] = tot[0] | (tot[1] << 16);
        s_cnt[i][2 * t + 1] = tot[2] | (tot[3] << 16);
        tot[0] += w0 & 0xFFFFu;
        tot[1] += w0 >> 16;
        tot[2] += w1 & 0xFFFFu;
        tot[3] += w1 >> 16;
      }
      uint32_t* my = &status[(uint64_t)tile * kWideBins + DPT * t];
#pragma unroll
      for (int k = 0; k < DPT; ++k)
        st_agent(&my[k], ((tile == first ? kFlagPrefix : kFlagAgg) << 30) | tot[k]);
      const uint32_t sum4 = tot[0] + tot[1] + tot[2] + tot[3];
      const uint32_t inc = wave_incl_add(sum4);
      if (l == kWave - 1) s_wsum[w] = inc;
      __syncthreads();
      uint32_t ex = inc - sum4;  // tile-local first slot of digit 4t
#pragma unroll
      for (int i = 0; i < WAVES; ++i) ex += i < w ? s_wsum[i] : 0u;
      uint32_t exk[DPT];
#pragma unroll
      for (int k = 0; k < DPT; ++k) {
        exk[k] = ex;
        ex += tot[k];
      }
      if (t == THREADS - 1) s_tilen = ex;
#pragma unroll
      for (int i = 0; i < WAVES; ++i) {
        s_cnt[i][2 * t] += exk[0] | (exk[1] << 16);
        s_cnt[i][2 * t + 1] += exk[2] | (exk[3] << 16);
      }
      __syncthreads();
      // Stage the keys in digit order before the look-back, which then
      // holds few registers (the tile-local slots do not depend on it).
#pragma unroll
      for (int i = 0; i < ITEMS; ++i) {
        if (FULL || ((part >> i) & 1u)) {
          const uint32_t d = (key[i] >> shift) & dmask;
          const uint32_t pos = ((s_cnt[w][d >> 1] >> (16u * (d & 1u))) & 0xFFFFu) + rank[i];
          s_stage[pos] = key[i];
          rank[i] = pos;  // keep the LDS slot for the rids
        }
      }
      uint32_t slot2[(ITEMS + 1) / 2];
#pragma unroll
      for (int i = 0; i < ITEMS; i += 2)
        slot2[i / 2] = (rank[i] & 0xFFFFu) | (i + 1 < ITEMS ? rank[i + 1 < ITEMS ? i + 1 : i] << 16 : 0u);
      uint32_t prev[DPT] = {0u, 0u, 0u, 0u};
      if (tile > first) {
        lookback_digits4<WAH_WIDE_LOOKAHEAD>(status + DPT * t, tile, first, kWideBins, fault, prev);
#pragma unroll
        for (int k = 0; k < DPT; ++k) st_agent(&my[k], (kFlagPrefix << 30) | (prev[k] + tot[k]));
      }
#pragma unroll
      for (int k = 0; k < DPT; ++k)
        s_glob[DPT * t + k] = goff[DPT * t + k] + prev[k] - exk[k];  // + slot = column index
      uint32_t rid[ITEMS];
      if (implicit) {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) rid[i] = cd.rid_base + (uint32_t)wbase + (uint32_t)(i * kWave);
      } else {
        const uint32_t* rp = src_rids + cd.off + wbase;
#pragma unroll
        for (int i = 0; i < ITEMS; ++i)
          rid[i] = FULL || (uint32_t)(i * kWave) < nvalid ? rp[i * kWave] : 0u;
      }
      __syncthreads();
      const uint32_t tile_n = FULL ? (uint32_t)TILE : s_tilen;
      uint32_t* dk = dst_keys + cd.off;
      uint32_t* dr = dst_rids + cd.off;
      uint16_t* dk16 = reinterpret_cast<uint16_t*>(dk);
      const uint32_t last = (uint32_t)(n - 1);  // stores stay in the column
      bool bad = false;
      uint32_t gq[ITEMS];
#pragma unroll
      for (int j = 0; j < ITEMS; ++j) {
        const uint32_t q = (uint32_t)j * THREADS + t;
        gq[j] = last;
        if (FULL || q < tile_n) {
          const uint32_t k = s_stage[q];
          const uint32_t g = s_glob[(k >> shift) & dmask] + q;
          bad |= g > last;
          gq[j] = g < last ? g : last;
          if (narrow) dk16[gq[j]] = (uint16_t)k;
          else dk[gq[j]] = k;
        }
      }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < ITEMS; ++i)
        if (FULL || ((part >> i) & 1u)) s_stage[(slot2[i / 2] >> (16 * (i % 2))) & 0xFFFFu] = rid[i];
      __syncthreads();
#pragma unroll
      for (int j = 0; j < ITEMS; ++j) {
        const uint32_t q = (uint32_t)j * THREADS + t;
        if (FULL || q < tile_n) dr[gq[j]] = s_stage[q];
      }
      if (ballot(bad) && l == 0) atomicOr(fault, 2u);  // a scatter index past the column
    };
    if (base + TILE <= n) sweep(std::true_type{});
    else sweep(std::false_type{});
    __syncthreads();
  }
}

// Selects the sorted arrays of one column (after its active passes); the
// pointers address the column's first pair.
struct SortedView {
  const uint32_t* keys;  // 32-bit keys, or 16-bit ones at the same start (narrow)
  const uint32_t* rids;
  const uint32_t* lits;  // run mode
  bool implicit;
  bool narrow;
  __device__ __forceinline__ uint32_t key(uint32_t i) const {
    return narrow ? (uint32_t)reinterpret_cast<const uint16_t*>(keys)[i] : keys[i];
  }
};
__device__ __forceinline__ SortedView sorted_view(const ColState* col, const Column& cd,
                                                  const uint32_t* values,
                                                  const uint32_t* keysA, const uint32_t* ridsA,
                                                  const uint32_t* keysB, const uint32_t* ridsB,
                                                  const uint32_t* litsA = nullptr,
                                                  const uint32_t* litsB = nullptr) {
  SortedView v;
  const uint32_t f = col->final_buf;
  v.implicit = f == kBufValues;
  v.narrow = col->narrow != 0u && f != kBufValues;
  v.keys = (f == kBufValues ? values : (f == kBufA ? keysA : keysB)) + cd.off;
  v.rids = (f == kBufA ? ridsA : ridsB) + cd.off;
  v.lits = (f == kBufA ? litsA : litsB) + cd.off;
  return v;
}

// ---------------------------------------------------------------------------
// Fused tail over the sorted items: (value, rid) pairs, or in run mode
// (value, rid, literal bits) runs.  Per item: chid = rid/31; an entry starts
// where (value, chid) changes and ORs the literal bits of the items up to the
// next entry start (at most 31 rows, one chunk); a key starts where value
// changes.  fill = chid for a key start, else chid - chid_prev - 1; an entry
// emits [fill if nonzero, literal].
//
// Blocked layout: thread t owns the ITEMS consecutive items [t*ITEMS, +ITEMS)
// of a tile, loaded from HBM straight into registers with 16-byte loads.  An
// item's predecessor is the lane's previous register, lane l-1's last item
// (DPP wave shift) or, for lane 0, one load per wave.  Word and key counts
// are summed along the lane, then one DPP wave scan and the wave totals give
// each lane its tile-local offsets; a wave-parallel look-back across tiles
// gives the tile's.  The run of a lane's last entry start continues into at
// most four following lanes (31 items, ITEMS >= 8 per lane): their lead bits
// (before their first entry start) arrive by DPP lane shifts; a run crossing
// into the next wave or tile takes that wave's or tile's lead bits, which
// are exchanged in LDS.  Words are staged in LDS at tile-local positions and
// stored contiguously.
// ---------------------------------------------------------------------------
// MODES as in k_onesweep: one mode's tiles per launch for long columns, both in
// one launch for the others.
template <int THREADS, int ITEMS, int MODES>
__global__ __launch_bounds__(THREADS, tail_waves_per_eu(ITEMS)) void k_tail(
    const DescHead* __restrict__ desc, const ColState* __restrict__ cs, Header* __restrict__ hdr,
    const uint32_t* values, const uint32_t* keysA, const uint32_t* ridsA,
    const uint32_t* keysB, const uint32_t* ridsB, const uint32_t* litsA, const uint32_t* litsB,
    uint32_t* __restrict__ keys_out, uint32_t* __restrict__ offsets_out,
    uint32_t* __restrict__ words_out, uint64_t* status, uint32_t* __restrict__ tile_entries,
    uint32_t lanes, wahgpu_counts_dev* __restrict__ counts) {
  constexpr int TILE = THREADS * ITEMS;
  constexpr int WAVES = THREADS / kWave;
  static_assert(ITEMS % 8 == 0 && ITEMS <= 16, "16-byte loads (8 narrow keys); runs span <= 4 lanes");
  static_assert(2 * TILE < 65536, "tile word and key counts fit 16 bits");
  constexpr uint32_t kAll = (1u << ITEMS) - 1u;
  // staged words, one pad word per 16: lanes that write ~16 words apart
  // (two per item) land in different banks
  __shared__ uint32_t s_words[2 * TILE + 2 * TILE / 16];
  __shared__ uint32_t s_wtot[WAVES];
  __shared__ uint32_t s_went[WAVES];
  __shared__ uint32_t s_wlead[WAVES + 1];  // [w]: lead bits of wave w; [WAVES]: of the next tile
  __shared__ uint64_t s_prefix;
  __shared__ uint32_t s_tile;
  if constexpr (MODES != 1) {
    constexpr bool RUN = false;
#include "tail_tiles.inl"
  }
  if constexpr (MODES == 2) __syncthreads();  // the last draw is read before the next mode's first
  if constexpr (MODES != 0) {
    constexpr bool RUN = true;
#include "tail_tiles.inl"
  }
}

// Per column: k = the sum of its tail tiles' entry counts; lengths[i] =
// offsets[i+1] - offsets[i], the last key running to L; the build's fault
// word is copied into every column's counts.
__global__ __launch_bounds__(kBlock) void k_finish(const DescHead* __restrict__ desc,
                                                   const Header* __restrict__ hdr,
                                                   const uint32_t* __restrict__ tile_entries,
                                                   const uint32_t* __restrict__ offsets,
                                                   uint32_t* __restrict__ lengths,
                                                   wahgpu_counts_dev* __restrict__ counts) {
  const uint32_t ncols = desc->dims.ncols;
  const Column* cols = desc_cols(desc);
  const uint32_t fault = hdr->fault;
  const uint64_t gt = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
  const uint64_t gs = (uint64_t)gridDim.x * kBlock;
  {
    // k per column = the entry counts of its tail tiles (zeroed by the
    // histogram, written by the tiles that held items).  Each wave takes 64
    // consecutive tiles, sums them per column (segmented wave scan) and adds
    // each column's part once.
    const uint32_t lane = threadIdx.x % kWave;
    const uint32_t ntiles = desc->dims.tail_tiles;
    for (uint64_t w0 = gt - lane; w0 < ntiles; w0 += gs) {
      const uint32_t tile = (uint32_t)w0 + lane;
      uint32_t c = find_segment(&cols[0].tail_tile0, sizeof(Column) / 4, ncols, (uint32_t)w0);
      uint32_t v = 0;
      if (tile < ntiles) {
        while (c + 1 < ncols && cols[c + 1].tail_tile0 <= tile) ++c;
        v = tile_entries[tile];
      }
      const uint32_t cp = (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)c, 0x138, 0xF, 0xF, false);
      const uint64_t hm = ballot(c != cp);  // first lane of each column
      const uint32_t inc = wave_incl_add(v);
      const uint64_t upto = lane == kWave - 1 ? ~0ull : ((2ull << lane) - 1ull);
      const int h = 63 - __builtin_clzll(hm & upto);  // this lane's first lane of its column
      const uint32_t seg = inc - (uint32_t)__shfl((int)(inc - v), h, kWave);
      const bool last = lane == kWave - 1 || ((hm >> (lane + 1)) & 1ull);
      if (last && seg) atomicAdd((unsigned long long*)&counts[cols[c].index].k, (unsigned long long)seg);
    }
  }
  // The blocks are dealt to the columns, `parts` of them to each; with more
  // columns than blocks a block takes every gridDim-th.  (All blocks walking
  // all columns cost a batch of 128 columns 90 us.)
  if (ncols == 0) return;
  const uint32_t parts = gridDim.x > ncols ? gridDim.x / ncols : 1u;
  const uint32_t part = blockIdx.x / ncols;
  if (part >= parts) return;
  for (uint32_t c = blockIdx.x % ncols; c < ncols; c += gridDim.x) {
    const Column cd = cols[c];
    const uint64_t kc = counts[cd.index].keycnt;
    const uint64_t K = kc < cd.n ? kc : cd.n, L = counts[cd.index].length;
    const uint32_t* o = offsets + cd.off;
    uint32_t* len = lengths + cd.off;
    const uint32_t step = parts * kBlock;
    for (uint32_t i = part * kBlock + threadIdx.x; i < K; i += step) {
      const uint32_t end = (i + 1 < K) ? o[i + 1] : (uint32_t)L;
      len[i] = end - o[i];
    }
    if (part == 0 && threadIdx.x == 0 && fault) counts[cd.index].fault = fault;
  }
}

// ---------------------------------------------------------------------------
// Staged kernels that are no scan (one per reference stage); wah_scan.hip holds
// the others.
// ---------------------------------------------------------------------------
// Copy the sorted result of column 0 out of the pass buffers (stage API).
__global__ __launch_bounds__(kBlock) void k_sort_finalize(
    const DescHead* __restrict__ desc, const ColState* __restrict__ cs, const uint32_t* values,
    const uint32_t* keysA, const uint32_t* ridsA, const uint32_t* keysB, const uint32_t* ridsB,
    uint32_t* out_keys, uint32_t* out_rids) {
  const Column cd = desc_cols(desc)[0];
  const SortedView sv = sorted_view(&cs[0], cd, values, keysA, ridsA, keysB, ridsB);
  if (sv.keys == out_keys && !sv.implicit) return;
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < cd.n;
       i += (uint64_t)gridDim.x * kBlock) {
    out_keys[i] = sv.key((uint32_t)i);
    out_rids[i] = sv.implicit ? cd.rid_base + (uint32_t)i : sv.rids[i];
  }
}

// include/produce_chunk_id_literals.cl:17-24
__global__ __launch_bounds__(kBlock) void k_chunks(const uint32_t* __restrict__ rids, uint64_t n,
                                                   uint32_t* __restrict__ chids,
                                                   uint32_t* __restrict__ lits) {
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * kBlock) {
    uint32_t r = rids[i];
    lits[i] = 0x80000000u | (1u << (r % 31u));
    chids[i] = r / 31u;
  }
}

// include/produce_fills.cl:24-43
__global__ __launch_bounds__(kBlock) void k_fills(const uint32_t* __restrict__ vals,
                                                  const uint32_t* __restrict__ chids, uint64_t k,
                                                  uint32_t* __restrict__ fills) {
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < k;
       i += (uint64_t)gridDim.x * kBlock) {
    uint32_t c = chids[i];
    fills[i] = (i > 0 && vals[i] == vals[i - 1]) ? c - chids[i - 1] - 1u : c;
  }
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
static uint32_t cap_grid(uint32_t work, uint32_t cap) {
  const uint32_t g = work < cap ? work : cap;
  return g ? g : 1u;
}
// Grid of a kernel that draws tiles: a whole number of blocks per counter lane
// (see tile_group).
static uint32_t tile_grid(uint32_t tiles, uint32_t cap) {
  const uint32_t whole = tiles > kTileLanes ? (tiles + kTileLanes - 1) / kTileLanes * kTileLanes : tiles;
  return cap_grid(whole, cap);
}

// Radix blocks resident per CU: the waves the register budget allows
// (sort_waves_per_eu per SIMD) and the LDS of k_onesweep (staged keys,
// per-wave digit counts, digit tables; 160 KiB per CU).
template <int T, int I>
constexpr uint32_t sort_blocks_per_cu() {
  constexpr uint32_t by_waves = sort_waves_per_eu(I) * 4 / (T / kWave);
  constexpr uint32_t lds = T * I * 4 + (T / kWave) * 1024 + 2 * 1024 + 64;
  constexpr uint32_t by_lds = 160u * 1024u / lds;
  constexpr uint32_t b = by_waves < by_lds ? by_waves : by_lds;
  return b ? b : 1u;
}

// Wide-digit blocks per CU: two 512-thread blocks (4 waves per SIMD) with
// ~72 KiB of LDS each (staged keys, 16-bit counters, digit offsets).
constexpr uint32_t kWideBlocksPerCU = 2;

// The run cut and the four radix launches for one tile shape (with the
// wide-digit launches when a column may take them).
template <int T, int I>
static void launch_radix(const BuildArgs& a, hipStream_t s, LaunchHook* hook) {
  const uint32_t grid = tile_grid(a.sort_tiles_cap, WAH_STATIC_TILES
                                                       ? a.sort_tiles_cap
                                                       : a.max_resident / 4 * sort_blocks_per_cu<T, I>());
  if (!a.force_pair)
    hipLaunchKernelGGL(k_runcut, dim3(cap_grid(a.hist_chunks_cap, 2 * a.max_resident)),
                       dim3(kBlock), 0, s, a.values, a.keysB, a.ridsB, a.litsB, a.desc, a.cs,
                       a.hdr, a.tile_runs, (uint32_t)(T * I), a.litsA);
  // wide digits: the histograms of the wide columns' digits and their offsets
  const uint32_t wgrid = tile_grid(a.wide_tiles_cap, WAH_STATIC_TILES ? a.wide_tiles_cap
                                                                    : a.max_resident / 4 * kWideBlocksPerCU);
  if (a.wide_tiles_cap) {
    uint64_t hb = (a.n_cap + 4 * kHistChunk - 1) / (4 * kHistChunk);
    if (hb > a.hist_chunks_cap) hb = a.hist_chunks_cap;
    hipLaunchKernelGGL(k_whist, dim3(cap_grid((uint32_t)hb, kHistMaxBlocks)), dim3(kBlock), 0, s,
                       a.values, a.desc, a.cs, a.wide, a.wide_status);
    hipLaunchKernelGGL(k_wplan, dim3(cap_grid(a.cols_cap, 1024)), dim3(kBlock), 0, s, a.desc,
                       a.cs, a.wide);
  }
  if (hook) hook->mark(s);
  // each launch runs the a-th pass of pair-mode columns, then of run-mode
  // columns
  for (uint32_t p = 0; p < 4; ++p) {
    auto sweep = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(grid), dim3(T), 0, s, p, a.values, a.keysA, a.ridsA, a.keysB,
                         a.ridsB, a.litsA, a.litsB, a.desc, a.cs, a.hdr, a.sort_status,
                         a.sort_status_stride, tile_lanes(grid));
    };
    if (!a.long_tail && !a.force_pair) {
      sweep(a.atomic_rank ? k_onesweep<T, I, kRankAtomic, 2> : k_onesweep<T, I, kRankMatch, 2>);
    } else {
      sweep(a.atomic_rank ? k_onesweep<T, I, kRankAtomic, 0> : k_onesweep<T, I, kRankMatch, 0>);
      if (!a.force_pair)
        sweep(a.atomic_rank ? k_onesweep<T, I, kRankAtomic, 1> : k_onesweep<T, I, kRankMatch, 1>);
    }
    if (a.wide_tiles_cap && p < (uint32_t)kWidePasses) {
      if (a.atomic_rank)
        hipLaunchKernelGGL((k_wsweep<kRankAtomic>), dim3(wgrid), dim3(kWideThreads), 0, s, p,
                           a.values, a.keysA, a.ridsA, a.keysB, a.ridsB, a.desc, a.cs, a.wide,
                           a.hdr, a.wide_status, a.wide_status_stride, tile_lanes(wgrid));
      else
        hipLaunchKernelGGL((k_wsweep<kRankMatch>), dim3(wgrid), dim3(kWideThreads), 0, s, p,
                           a.values, a.keysA, a.ridsA, a.keysB, a.ridsB, a.desc, a.cs, a.wide,
                           a.hdr, a.wide_status, a.wide_status_stride, tile_lanes(wgrid));
    }
    if (hook) hook->mark(s);
  }
}

void launch_sort(const BuildArgs& a, hipStream_t s, LaunchHook* hook) {
  hipLaunchKernelGGL(k_begin, dim3(64), dim3(kBlock), 0, s, a.hdr, a.cs, a.cols_cap,
                     a.tile_runs, a.sort_tiles_cap, a.desc, (int)a.inline_desc, a.one_dims, a.one);
  // Two chunks per block: 2^20 values 64.2 us, with four 67.0 and with one 65.3;
  // 2^18 zipf values 63.9, with four 71.4; 128 columns of 2^12 to 2^20 values
  // 449, 465 and 450.  Longer single columns take four: there the adds of each
  // block's bins to the column's count (5 million ids 201.7 us, with two 203.4).
  // (At most 1024 blocks: 2^25 uniform values 442 -> 431 us, but 2^26 in runs
  // 248 -> 260 and 2^25 zipf ones 491 -> 495.)
  const uint64_t hist_rows = (!a.inline_desc || a.n_cap <= (1u << 21) ? 2 : 4) * kHistChunk;
  uint64_t hb = (a.n_cap + hist_rows - 1) / hist_rows;
  if (hb > a.hist_chunks_cap) hb = a.hist_chunks_cap;
  hipLaunchKernelGGL(k_histogram, dim3(cap_grid((uint32_t)hb, kHistMaxBlocks)), dim3(kBlock), 0,
                     s, a.values, a.desc, a.cs, a.sort_status, a.tail_status, a.tile_entries,
                     a.tile_runs, radix_tile(a.shape), a.litsA);
  hipLaunchKernelGGL(k_plan, dim3(cap_grid(a.cols_cap, 1024)), dim3(kBlock), 0, s, a.desc, a.cs,
                     a.hdr, a.tile_runs, a.counts, (int)a.force_pair, radix_tile(a.shape), a.wide);
  switch (a.shape) {
#define WAH_SHAPE_CASE(sh) \
  case sh: launch_radix<radix_threads(sh), radix_items(sh)>(a, s, hook); break;
    WAH_SHAPE_CASE(1)
    WAH_SHAPE_CASE(2)
    WAH_SHAPE_CASE(3)
    WAH_SHAPE_CASE(4)
    WAH_SHAPE_CASE(5)
#undef WAH_SHAPE_CASE
    default: launch_radix<radix_threads(0), radix_items(0)>(a, s, hook); break;
  }
  static_assert(kRadixShapes == 6, "a case per compiled shape");
}

// The tails of a long column, on 16384-item tiles, or of other columns and of
// batches, on 8192-item tiles.
template <int T, int I, int MODES>
static void launch_tail_tiles(const BuildArgs& a, uint32_t blocks_per_cu, hipStream_t s) {
  const uint32_t grid = tile_grid(
      a.tail_tiles_cap, WAH_STATIC_TILES ? a.tail_tiles_cap : a.max_resident / 4 * blocks_per_cu);
  hipLaunchKernelGGL((k_tail<T, I, MODES>), dim3(grid), dim3(T), 0, s, a.desc, a.cs, a.hdr,
                     a.values, a.keysA, a.ridsA, a.keysB, a.ridsB, a.litsA, a.litsB, a.out_keys,
                     a.out_offsets, a.out_words, a.tail_status, a.tile_entries,
                     WAH_TAIL_LANES ? WAH_TAIL_LANES : tile_lanes(grid), a.counts);
}

void launch_tail(const BuildArgs& a, hipStream_t s, LaunchHook* hook) {
  if (a.long_tail) {
    launch_tail_tiles<kLongTailThreads, kLongTailItems, 0>(a, kLongTailBlocksPerCU, s);
    launch_tail_tiles<kLongTailThreads, kLongTailItems, 1>(a, kLongTailBlocksPerCU, s);
  } else {
    launch_tail_tiles<kTailThreads, kTailItems, 2>(a, kTailBlocksPerCU, s);
  }
  if (hook) hook->mark(s);
  // blocks for up to 8 x 256 keys per column of a batch at a time
  const uint64_t lg = (a.n_cap + kBlock - 1) / kBlock, most = a.cols_cap > 128u ? 8ull * a.cols_cap : 1024u;
  hipLaunchKernelGGL(k_finish, dim3(cap_grid((uint32_t)(lg < most ? lg : most), 8192)),
                     dim3(kBlock), 0, s, a.desc, a.hdr, a.tile_entries, a.out_offsets,
                     a.out_lengths, a.counts);
}

void launch_sort_finalize(const BuildArgs& a, hipStream_t s) {
  uint64_t g = (a.n_cap + kBlock - 1) / kBlock;
  if (g > 4096) g = 4096;
  if (g == 0) return;
  hipLaunchKernelGGL(k_sort_finalize, dim3((uint32_t)g), dim3(kBlock), 0, s, a.desc, a.cs,
                     a.values, a.keysA, a.ridsA, a.keysB, a.ridsB, a.sorted_keys, a.sorted_rids);
}

void launch_rank_selftest(uint32_t* ok, hipStream_t s) {
  hipLaunchKernelGGL(k_rank_selftest, dim3(64), dim3(256), 0, s, ok);
}

static uint32_t grid_for(uint64_t n) {
  uint64_t g = (n + kBlock - 1) / kBlock;
  if (g > 8192) g = 8192;
  return g ? (uint32_t)g : 1u;
}

void launch_fill32(uint32_t* p, uint64_t words, uint32_t v, hipStream_t s) {
  if (!words) return;
  hipLaunchKernelGGL(k_fill32, dim3(grid_for(words)), dim3(kBlock), 0, s, p, words, v);
}

void launch_chunks(const uint32_t* rids, uint64_t n, uint32_t* chids, uint32_t* lits,
                   hipStream_t s) {
  if (!n) return;
  hipLaunchKernelGGL(k_chunks, dim3(grid_for(n)), dim3(kBlock), 0, s, rids, n, chids, lits);
}

void launch_fills(const uint32_t* vals, const uint32_t* chids, uint64_t k, uint32_t* fills,
                  hipStream_t s) {
  if (!k) return;
  hipLaunchKernelGGL(k_fills, dim3(grid_for(k)), dim3(kBlock), 0, s, vals, chids, k, fills);
}

}  // namespace wah
