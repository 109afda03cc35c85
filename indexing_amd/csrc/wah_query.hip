// wah_query.hip -- gfx950 kernels of the query side of a WAH index: decoding
// WAH word streams into row bitmaps, and encoding row bitmaps (or a bitwise
// combination of two) back into WAH words in the build's canonical form.
//
// Word format (src/cpu.cpp:47-74): bit 31 set = literal, whose payload bits
// 0..30 are the rows 31 c + b of its chunk c; bit 31 clear = fill of
// (bits 0..29) chunks, all of value bit 30.  Each key's stream starts at
// chunk 0, so a word's first chunk is the sum of the chunk counts of the
// words before it in its key's stream.
//
// Row bitmap: row r is bit r % 32 of 32-bit word r / 32.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "wah_scan.h"
#include "wah_slices.h"

namespace wah {

namespace {

// Decode tiles of 4096 words at two blocks per CU: two million words (2^27 rows
// at density 0.01) take 18.9 us, 2048-word tiles 21.5, 8192-word ones 19.6, and
// two streams of 6000 words 9.3, 10.1 and 14.8 us (a lane writes its words one
// after another, so a short stream wants more lanes).
constexpr int kDecRows = 2;
constexpr uint32_t kDecTile = kScanTileOf<kDecRows>;  // words per decode tile
// Resident blocks per CU.
constexpr int kDecBlocks = 2;
// 20.2 us for 2^27 rows, with 2 and 3 blocks 24.5 and 23.1 (timed with blocks that
// took their first tile by index; 21.3 with all tiles drawn)
constexpr int kEncBlocks = 4;
static_assert(kDecTile == kDecodeTileWords, "what the host counts status words by");
constexpr int query_waves_per_eu(int blocks) { return blocks * kScanWaves / 4; }

__device__ __forceinline__ uint32_t word_chunks(uint32_t w) {
  return (w & 0x80000000u) ? 1u : (w & 0x3FFFFFFFu);
}

// ORs the payload of a literal at chunk c into the bitmap, dropping rows at or
// past nrows (chunks = chunks of nrows rows; rows are below 2^32).
__device__ __forceinline__ void or_literal(uint32_t* bitmap, uint64_t nrows, uint32_t chunks,
                                           uint32_t c, uint32_t bits) {
  if (c >= chunks) return;
  const uint32_t row0 = 31u * c;
  if (nrows - row0 < 31) bits &= (1u << (uint32_t)(nrows - row0)) - 1u;
  const uint32_t wi = row0 >> 5, sh = row0 & 31u;
  const uint32_t lo = bits << sh;
  if (lo) atomicOr(&bitmap[wi], lo);
  if (sh > 1) {
    const uint32_t hi = bits >> (32u - sh);
    if (hi) atomicOr(&bitmap[wi + 1], hi);
  }
}

// How a word beside a literal's bears on the bitmap words they may share: a
// literal (its payload is in those words), a 0-fill (nothing is), or a word
// that says nothing about the neighbouring chunk (a fill of no chunks, the end
// of the stream) or sets rows by itself (a 1-fill).
__device__ __forceinline__ bool beside_literal(uint32_t v) { return v & 0x80000000u; }
__device__ __forceinline__ bool beside_open(uint32_t v) {
  return !(v & 0x80000000u) && ((v & 0x40000000u) || !(v & 0x3FFFFFFFu));
}

// Writes the payload of a literal at chunk c of a single stream, between the
// words before and after it.  A bitmap word holds rows of two chunks at most,
// c and c + 1: where both are literals the later one writes the word with the
// earlier one's rows, else the one that has rows there does, so every word is
// stored once and no atomics are needed (device-scope ORs ran at 37 G/s, which
// held a decode of 2^27 rows at 59 us).  Beside an open word the ORs stay.
__device__ __forceinline__ void put_literal(uint32_t* bitmap, uint64_t nrows, uint32_t chunks,
                                            uint32_t c, uint32_t bits, uint32_t before,
                                            uint32_t after) {
  if (c >= chunks) return;
  const uint32_t row0 = 31u * c;
  if (nrows - row0 < 31) bits &= (1u << (uint32_t)(nrows - row0)) - 1u;
  const uint32_t wi = row0 >> 5, sh = row0 & 31u;
  // rows shared with chunk c - 1: word wi (sh = 0: that chunk ends with a word)
  uint32_t lo = 0;
  if (sh) {
    lo = bits << sh;
    if (beside_literal(before)) lo |= (before & 0x7FFFFFFFu) >> (31u - sh);
  }
  // rows shared with chunk c + 1: word wi + 1, or wi when c starts it
  const uint32_t hi = sh ? (sh > 1 ? bits >> (32u - sh) : 0u) : bits;
  const uint32_t hw = sh ? wi + 1u : wi;
  const bool take_hi = hi && !(beside_literal(after) && c + 1u < chunks);
  if (beside_open(before) || beside_open(after)) {
    if (lo) atomicOr(&bitmap[wi], lo);
    if (take_hi) atomicOr(&bitmap[hw], hi);
  } else {
    if (lo) bitmap[wi] = lo;
    if (take_hi) bitmap[hw] = hi;
  }
}

// Sets rows [row0, row0 + count) (a 1-fill; the build never writes one, the
// decoder of src/cpu.cpp:60-66 accepts it).
__device__ void set_rows(uint32_t* bitmap, uint64_t nrows, uint64_t row0, uint64_t count) {
  uint64_t end = row0 + count < nrows ? row0 + count : nrows;
  for (uint64_t r = row0; r < end;) {
    const uint32_t sh = (uint32_t)(r & 31u);
    const uint64_t take = (32u - sh) < end - r ? (32u - sh) : end - r;
    const uint32_t m = take == 32 ? 0xFFFFFFFFu : ((1u << (uint32_t)take) - 1u) << sh;
    atomicOr(&bitmap[r >> 5], m);
    r += take;
  }
}

// Number of the ascending x[0 .. n) below v, by a whole wave: 64 probes per
// round trip.
__device__ __forceinline__ uint64_t wave_lower_bound(const uint32_t* __restrict__ x, uint64_t n,
                                                     uint64_t v) {
  const uint32_t l = lane_id();
  uint64_t a = 0, e = n;  // answer in [a, e]
  while (e > a) {
    const uint64_t step = (e - a + kWave - 1) / kWave;
    const uint64_t p = a + (l + 1) * step - 1;  // last element of the lane's strip
    const bool below = p < e && x[p] < v;
    const uint64_t whole = (uint64_t)__builtin_popcountll(ballot(below));  // strips all below v
    a += whole * step;
    if (step == 1) break;
    e = a + step - 1 < e ? a + step - 1 : e;
  }
  return a;
}

}  // namespace

namespace {

constexpr int kSliceThreads = 1024;
constexpr int kEnterRows = 4;  // tiles of 8192 words
constexpr uint32_t kEnterTile = kScanTileOf<kEnterRows>;
static_assert(kEnterTile >= kDecTile, "a range has no more of these");

// A range that decodes by slices: one pass over its words, as k_q_decode<true>
// makes it (per key a scan of chunk counts, with look-back), that writes where
// each key's words enter each slice: table[slice * keys + key] = first chunk <<
// 32 | word + 1 of the word whose chunks hold the slice's first.  A lane needs
// the first chunk of its four words only, and looks for a slice's start among
// all of their chunks at once; a tile in which no key starts, which is most of
// them, skips everything about keys.
// (54 MB of words take 31 us, 35 as profiled.)
__device__ __forceinline__ void enter_slices(const uint32_t* __restrict__ words,
                                             const uint32_t* __restrict__ offsets, uint32_t span,
                                             uint32_t slices, uint64_t* __restrict__ table,
                                             ScanState* st, uint64_t* status, uint64_t* host) {
  __shared__ uint32_t s_sum[kScanWaves], s_head[kScanWaves];
  __shared__ uint32_t s_mark[kEnterTile / 32];
  __shared__ uint64_t s_key0, s_key1;
  __shared__ uint32_t s_prefix, s_tile;
  const uint32_t recip = 0xFFFFFFFFu / span + 1u;  // 2^32 / span, rounded up
  const int l = threadIdx.x % kWave;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint64_t key_a = st->range[0], key_b = st->range[1], w0 = st->range[2];
  const uint64_t len = st->range[3] - w0;
  const uint32_t keys = (uint32_t)(key_b - key_a);
  words += w0;
  const uint32_t tiles = (uint32_t)((len + kEnterTile - 1) / kEnterTile);
  for (uint32_t tile = scan_next_tile(st, &s_tile, tiles, true); tile < tiles;
       tile = scan_next_tile(st, &s_tile, tiles, false)) {
    const uint64_t base = (uint64_t)tile * kEnterTile;
    W4 x[kEnterRows];
    if (base + kEnterTile <= len) {
#pragma unroll
      for (int r = 0; r < kEnterRows; ++r)
        x[r] = load4<true>(words, base + row_at<kEnterRows>(w, l, r), len);
    } else {
#pragma unroll
      for (int r = 0; r < kEnterRows; ++r)
        x[r] = load4<false>(words, base + row_at<kEnterRows>(w, l, r), len);
    }
    if (w < 2) {  // the keys that start in the tile: [s_key0, s_key1)
      const uint64_t k = wave_lower_bound(offsets + key_a, key_b - key_a,
                                          w0 + base + (w ? kEnterTile : 0u)) + key_a;
      if (l == 0) *(w ? &s_key1 : &s_key0) = k;
    }
    __syncthreads();
    const uint64_t key0 = s_key0, key1 = s_key1;
    const bool heads = key0 < key1;  // block-uniform
    uint32_t hb = 0;                 // key starts, bit 4r + k
    if (heads) {
      for (uint32_t i = threadIdx.x; i < kEnterTile / 32; i += kScanThreads) s_mark[i] = 0;
      __syncthreads();
      for (uint64_t k = key0 + threadIdx.x; k < key1; k += kScanThreads) {
        const uint64_t at = (uint64_t)offsets[k] - w0 - base;
        if (at >= kEnterTile) break;
        atomicOr(&s_mark[at / 32], 1u << (at % 32));
      }
      __syncthreads();
#pragma unroll
      for (int r = 0; r < kEnterRows; ++r) {
        const uint32_t e = row_at<kEnterRows>(w, l, r);
        hb |= ((s_mark[e / 32] >> (e % 32)) & 15u) << (4 * r);
      }
    }
    uint32_t q[kEnterRows];  // first chunk of the lane's four words, from its key's start or
    uint32_t openm = 0;      // (bit r) from the wave's
    uint32_t run = 0;        // chunks of the wave's earlier rows
    uint32_t start = 0;      // chunks before the open key's first word
    bool open = true;
#pragma unroll
    for (int r = 0; r < kEnterRows; ++r) {
      const uint32_t p1 = word_chunks(x[r].x), p2 = p1 + word_chunks(x[r].y),
                     p3 = p2 + word_chunks(x[r].z), s = p3 + word_chunks(x[r].w);
      const uint32_t inc = wave_incl_add(s);
      const uint32_t ex = run + inc - s;
      run += readlane(inc, kWave - 1);
      q[r] = ex - start;
      openm |= open ? 1u << r : 0u;
      if (heads) {
        const uint32_t h4 = (hb >> (4 * r)) & 15u;
        const uint32_t b = ex + (h4 & 8u ? p3 : h4 & 4u ? p2 : h4 & 2u ? p1 : 0u);
        const uint64_t hm = ballot(h4 != 0u);
        const uint64_t below = hm & ((1ull << l) - 1ull);
        const uint32_t got = __shfl(b, below ? 63 - __builtin_clzll(below) : 0, kWave);
        if (below) {
          q[r] = ex - got;
          openm &= ~(1u << r);
        }
        if (hm) {  // wave-uniform
          start = readlane(b, 63 - __builtin_clzll(hm));
          open = false;
        }
      }
    }
    if (l == 0) {
      s_sum[w] = open ? run : run - start;
      s_head[w] = open ? 0u : 1u;
    }
    __syncthreads();
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
    for (int r = 0; r < kEnterRows; ++r) {
      const uint64_t at = base + row_at<kEnterRows>(w, l, r);
      // Slices that start in [c, c + n): p1 .. p3 part the chunks between the
      // four words at `word` on.
      auto enter = [&](uint32_t c, uint32_t n, uint32_t p1, uint32_t p2, uint32_t p3,
                       uint64_t word) {
        uint32_t sl = __umulhi(c, recip), d = c - sl * span;  // sl may be one too many
        if ((int32_t)d < 0) {
          d += span;
          --sl;
        }
        if (d) {  // the next slice starts after c
          d = span - d;
          ++sl;
        }
        for (; d < n && sl < slices; d += span, ++sl) {
          const uint32_t k = (d >= p1) + (d >= p2) + (d >= p3);
          const uint32_t pk = k == 3 ? p3 : k == 2 ? p2 : k == 1 ? p1 : 0u;
          // the word's key: the last that starts at or before it
          uint64_t lo = key0, hi = key1;
          while (lo < hi) {
            const uint64_t mid = (lo + hi) / 2;
            if ((uint64_t)offsets[mid] <= w0 + word + k) lo = mid + 1;
            else hi = mid;
          }
          const uint64_t key = lo - 1 - key_a;
          if (key < keys)
            table[(uint64_t)sl * keys + key] = (uint64_t)(c + pk) << 32 | (word + k + 1);
        }
      };
      const uint32_t n0 = word_chunks(x[r].x), n1 = word_chunks(x[r].y),
                     n2 = word_chunks(x[r].z), n3 = word_chunks(x[r].w);
      uint32_t c = q[r] + ((openm >> r) & 1u ? carry : 0u);
      const uint32_t h4 = (hb >> (4 * r)) & 15u;
      if (!ballot(h4 != 0u)) {  // wave-uniform: no key starts in the row
        enter(c, n0 + n1 + n2 + n3, n0, n0 + n1, n0 + n1 + n2, at);
      } else {
#pragma unroll 1
        for (int k = 0; k < 4; ++k) {
          if ((h4 >> k) & 1u) c = 0;
          const uint32_t n = k == 0 ? n0 : k == 1 ? n1 : k == 2 ? n2 : n3;
          enter(c, n, ~0u, ~0u, ~0u, at + k);
          c += n;
        }
      }
    }
  }
  scan_finish(st, status, tiles, host);
}

}  // namespace

// One pass over WAH words: per word its first chunk (a scan of chunk counts,
// with look-back across tiles), then its literal bits or 1-fill rows ORed into
// the row bitmap (zero before).
//   SEG false: two streams, q.words[0 .. len) of each into its own bitmap (the
//     second may be empty), the second's tiles after the first's; the row
//     after the last set row of the first is the result.
//   SEG true: the concatenated streams of keys [range[0], range[1]), words
//     range[2] .. range[3] of q.words, which k_q_range found; each key's words
//     restart at chunk 0.  A tile finds the keys that start in it by a search
//     of their offsets and marks them in LDS, so the words are read once and
//     nothing else is (a flag array took a fill, a marking launch and 4 bytes
//     per word).
// What bounds it: sparse streams the atomic ORs (one per literal, each to a
// line of its own), dense ones the words.  A range of many words per key goes
// by slices instead (enter_slices, then k_q_slices).
template <bool SEG>
__global__ __launch_bounds__(kScanThreads, query_waves_per_eu(kDecBlocks)) void k_q_decode(
    DecodeStream qa, DecodeStream qb, const uint32_t* __restrict__ offsets, uint64_t nrows,
    uint64_t* __restrict__ table, uint32_t slices, ScanState* st, uint64_t* status,
    uint64_t* host) {
  __shared__ uint32_t s_sum[kScanWaves], s_head[kScanWaves];
  __shared__ uint32_t s_mark[SEG ? kDecTile / 32 : 1];
  __shared__ uint64_t s_key0;
  __shared__ uint32_t s_prefix, s_tile;
  const int l = threadIdx.x % kWave;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint32_t chunks = (uint32_t)((nrows + 30) / 31);
  uint64_t key_a = 0, key_b = 0, w0 = 0;
  if (SEG) {
    if (const uint32_t span = st->slice_span) {  // the range decodes by slices
      enter_slices(qa.words, offsets, span, slices, table, st, status, host);
      return;
    }
    key_a = st->range[0];
    key_b = st->range[1];
    w0 = st->range[2];
    qa.words += w0;
    qa.len = st->range[3] - w0;
  }
  const uint32_t tiles_a = (uint32_t)((qa.len + kDecTile - 1) / kDecTile);
  const uint32_t tiles = tiles_a + (SEG ? 0u : (uint32_t)((qb.len + kDecTile - 1) / kDecTile));
  uint64_t my_last = 0;  // row after the last set row of this thread's words (stream a)
  for (uint32_t tile = scan_next_tile(st, &s_tile, tiles, true); tile < tiles;
       tile = scan_next_tile(st, &s_tile, tiles, false)) {
    const bool second = !SEG && tile >= tiles_a;
    const DecodeStream q = second ? qb : qa;
    const uint32_t first = second ? tiles_a : 0u;
    const uint64_t base = (uint64_t)(tile - first) * kDecTile;
    auto body = [&](auto full_tag) {
      constexpr bool FULL = decltype(full_tag)::value;
      W4 x[kDecRows], y[kDecRows];  // words; their first chunks
#pragma unroll
      for (int r = 0; r < kDecRows; ++r)
        x[r] = load4<FULL>(q.words, base + row_at<kDecRows>(w, l, r), q.len);
      uint32_t hb = 0;  // key starts, bit 4r + k
      if (SEG) {
        for (uint32_t i = threadIdx.x; i < kDecTile / 32; i += kScanThreads) s_mark[i] = 0;
        if (w == 0) {
          const uint64_t k0 = wave_lower_bound(offsets + key_a, key_b - key_a, w0 + base) + key_a;
          if (l == 0) s_key0 = k0;
        }
        __syncthreads();
        for (uint64_t k = s_key0 + threadIdx.x; k < key_b; k += kScanThreads) {
          const uint64_t at = (uint64_t)offsets[k] - w0 - base;
          if (at >= kDecTile) break;
          atomicOr(&s_mark[at / 32], 1u << (at % 32));
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kDecRows; ++r) {
          const uint32_t e = row_at<kDecRows>(w, l, r);
          hb |= ((s_mark[e / 32] >> (e % 32)) & 15u) << (4 * r);
        }
      }
      uint32_t run = 0;    // chunks of the wave's earlier rows
      uint32_t start = 0;  // chunks before the open key's first word
      uint32_t openm = 0;  // words whose key began before the wave
      bool open = true;
#pragma unroll
      for (int r = 0; r < kDecRows; ++r) {
        const uint32_t h4 = (hb >> (4 * r)) & 15u;
        const uint32_t p1 = word_chunks(x[r].x), p2 = p1 + word_chunks(x[r].y),
                       p3 = p2 + word_chunks(x[r].z), s = p3 + word_chunks(x[r].w);
        if (!SEG) {
          // saturating: a literal far past nrows stays there
          const uint32_t q1 = word_chunks(x[r].x), q2 = add_sat(q1, word_chunks(x[r].y)),
                         q3 = add_sat(q2, word_chunks(x[r].z));
          const uint32_t sat = wave_incl_add_sat(add_sat(q3, word_chunks(x[r].w)));
          const uint32_t e0 = add_sat(run, lane_before(sat, 0u));
          y[r] = W4{e0, add_sat(e0, q1), add_sat(e0, q2), add_sat(e0, q3)};
          run = add_sat(run, readlane(sat, kWave - 1));
          continue;
        }
        const uint32_t inc = wave_incl_add(s);
        const uint32_t ex = run + inc - s;
        const uint32_t b = ex + (h4 & 8u ? p3 : h4 & 4u ? p2 : h4 & 2u ? p1 : 0u);
        const uint64_t hm = ballot(h4 != 0u);
        const uint64_t below = hm & ((1ull << l) - 1ull);
        const uint32_t got = __shfl(b, below ? 63 - __builtin_clzll(below) : 0, kWave);
        uint32_t cur = below ? got : start;
        bool o = !below && open;
        if (h4 & 1u) { cur = ex; o = false; }
        y[r].x = ex - cur;
        openm |= o ? 1u << (4 * r) : 0u;
        if (h4 & 2u) { cur = ex + p1; o = false; }
        y[r].y = ex + p1 - cur;
        openm |= o ? 2u << (4 * r) : 0u;
        if (h4 & 4u) { cur = ex + p2; o = false; }
        y[r].z = ex + p2 - cur;
        openm |= o ? 4u << (4 * r) : 0u;
        if (h4 & 8u) { cur = ex + p3; o = false; }
        y[r].w = ex + p3 - cur;
        openm |= o ? 8u << (4 * r) : 0u;
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
      uint32_t carry = 0, agg = 0;
      bool closed = false, tile_closed = false;
#pragma unroll
      for (int i = 0; i < kScanWaves; ++i) {
        if (i == w) {
          carry = agg;
          closed = tile_closed;
        }
        const bool h = SEG && s_head[i] != 0u;
        agg = h ? s_sum[i] : SEG ? agg + s_sum[i] : add_sat(agg, s_sum[i]);
        tile_closed |= h;
      }
      if (w == 0) {
        uint32_t hi, p;
        lookback2<kOpNone, SEG ? kOpSum : kOpSumSat>(status, tile, 0u, agg, tile_closed,
                                                     &st->fault, hi, p, first);
        if (l == 0) s_prefix = p;
      }
      __syncthreads();
      if (!closed) carry = SEG ? carry + s_prefix : add_sat(carry, s_prefix);
      // the words before and after the wave's (a single stream's first word
      // has a 0-fill before it, its last word an open one after it)
      uint32_t wb = 1u, wa = 0u;
      if (!SEG) {
        const uint64_t b = base + row_at<kDecRows>(w, 0, 0), e = b + kDecRows * kRowElems;
        if (b > 0 && b <= q.len) wb = q.words[b - 1];
        if (e < q.len) wa = q.words[e];
      }
#pragma unroll
      for (int r = 0; r < kDecRows; ++r) {
        const uint32_t before =
            SEG ? 0u : lane_before(x[r].w, r ? readlane(x[r ? r - 1 : 0].w, kWave - 1) : wb);
        const uint32_t after =
            SEG ? 0u
                : lane_after(x[r].x, r + 1 < kDecRows
                                         ? readlane(x[r + 1 < kDecRows ? r + 1 : r].x, 0)
                                         : wa);
        const uint32_t xs[4] = {x[r].x, x[r].y, x[r].z, x[r].w};
        const uint32_t ys[4] = {y[r].x, y[r].y, y[r].z, y[r].w};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const uint32_t c = SEG ? ys[k] + ((openm >> (4 * r + k)) & 1u ? carry : 0u)
                                 : add_sat(ys[k], carry);
          const uint32_t v = xs[k];  // past the stream's end: 0, a fill of nothing
          if (v & 0x80000000u) {
            const uint32_t bits = v & 0x7FFFFFFFu;
            if (SEG)
              or_literal(q.bitmap, nrows, chunks, c, bits);
            else
              put_literal(q.bitmap, nrows, chunks, c, bits, k ? xs[k - 1] : before,
                          k < 3 ? xs[k + 1] : after);
            if (!SEG && !second && bits) {
              const uint64_t end = 31ull * c + 32u - (uint32_t)__builtin_clz(bits);
              my_last = end > my_last ? end : my_last;
            }
          } else if ((v & 0x40000000u) && (v & 0x3FFFFFFFu)) {
            const uint64_t row0 = 31ull * c, cnt = 31ull * (v & 0x3FFFFFFFu);
            set_rows(q.bitmap, nrows, row0, cnt);
            if (!SEG && !second) my_last = row0 + cnt > my_last ? row0 + cnt : my_last;
          }
        }
      }
    };
    if (base + kDecTile <= q.len) body(std::true_type{});
    else body(std::false_type{});
  }
  if (!SEG) {
    // the block's last row goes to its lane's word, once (8 waves of 1000
    // blocks on one address took 90 us)
    __shared__ uint64_t s_row[kScanWaves];
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
      const uint64_t o = ((uint64_t)__shfl_xor((uint32_t)(my_last >> 32), d, kWave) << 32) |
                         __shfl_xor((uint32_t)my_last, d, kWave);
      my_last = o > my_last ? o : my_last;
    }
    if (l == 0) s_row[w] = my_last;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
      for (int i = 1; i < kScanWaves; ++i) my_last = s_row[i] > my_last ? s_row[i] : my_last;
      const uint32_t lane = blockIdx.x % tile_lanes(gridDim.x);
      if (my_last)
        atomicMax(reinterpret_cast<unsigned long long*>(&st->tiles[lane * kLaneStride + 2]),
                  (unsigned long long)my_last);
    }
  }
  scan_finish(st, status, tiles, host);
}

// Starts a range query: locates the keys of the index in [lo, hi] (keys
// ascend): range[0] = first key index >= lo, range[1] = first > hi, range[2] =
// first word of key range[0], range[3] = one past the last word of key
// range[1] - 1; the number of keys goes to host[3], of words to host[4].  A range
// of more than most_words words, which one whose offsets descend has too, takes
// no words: the caller reports it.  Then zeroes the row bitmap, or, for a range
// that decodes by slices, their table; one whose table would be larger than
// table_cap takes no words either if `grow`, and leaves the bitmap: the caller
// comes back with a table of that size.
// SLICES: whether it does is decided here, so every block locates the keys.
template <bool SLICES>
__global__ __launch_bounds__(kBlock) void k_q_range(
    const uint32_t* __restrict__ keys, const uint32_t* __restrict__ offsets,
    const uint32_t* __restrict__ lengths, uint64_t keycnt, uint32_t lo, uint32_t hi,
    uint64_t most_words, uint32_t* __restrict__ bitmap, uint64_t words,
    uint64_t* __restrict__ table, uint64_t table_cap, uint32_t slices, uint32_t slice_span,
    bool grow, ScanState* st, uint64_t* host) {
  __shared__ uint64_t s_at[2];
  const uint32_t t = threadIdx.x;
  uint64_t entries = 0;
  bool later = false;  // with a larger table
  if (SLICES || blockIdx.x == 0) {
    if (t < 2 * kWave) {
      const uint64_t v = t < kWave ? (uint64_t)lo : (uint64_t)hi + 1;
      const uint64_t at = wave_lower_bound(keys, keycnt, v);
      if (t % kWave == 0) s_at[t / kWave] = at;
    }
    __syncthreads();
    const uint64_t a = s_at[0], b = s_at[1] > a ? s_at[1] : a;  // (keys that descend: none)
    const uint64_t w0 = a < b ? offsets[a] : 0;
    const uint64_t w1 = a < b ? (uint64_t)offsets[b - 1] + lengths[b - 1] : 0;
    const uint64_t found = w1 - w0;  // 2^33 at least if w1 < w0
    uint64_t len = found <= most_words ? found : 0;
    if (SLICES) {
      entries = slice_entries(b - a, len, slices);
      if (entries > table_cap) {
        later = grow;
        entries = 0;
        if (later) len = 0;
      }
    }
    if (blockIdx.x == 0 && t == 0) {
      st->range[0] = a;
      st->range[1] = b;
      st->range[2] = w0;
      st->range[3] = w0 + len;
      st->slice_span = entries ? slice_span : 0u;
      __hip_atomic_store(&host[3], b - a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      __hip_atomic_store(&host[4], found, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }
  const uint64_t i0 = (uint64_t)blockIdx.x * kBlock + t, step = (uint64_t)gridDim.x * kBlock;
  if (later) return;
  if (SLICES && entries) {
    for (uint64_t i = i0; i < entries; i += step) table[i] = 0;
    return;
  }
  for (uint64_t i = i0; i < words; i += step) bitmap[i] = 0;
}

// Decodes a range by slices of the bitmap, one block each, from the table of
// where each key's words enter the slice (first chunk << 32 | word + 1, 0:
// nowhere): the block ORs the literals of its part of every key into LDS and
// stores the slice once.  The ORs of 6.7 million literals (a tenth of 4096
// keys, 2^26 rows) took 260 us as device-scope atomics, which run at 25 G/s
// however they are spread; here the same words take 32 us, and 33 us before for
// the table.  Bound by the instructions per step (about 100 for 128 words, of
// which a key has 124 in a slice), not by the loads: with one, two or three
// steps loaded ahead it takes the same.
__global__ __launch_bounds__(kSliceThreads) void k_q_slices(
    const uint32_t* __restrict__ words, const uint32_t* __restrict__ offsets,
    const uint64_t* __restrict__ table, uint32_t* __restrict__ bitmap, uint64_t nrows,
    const ScanState* __restrict__ st) {
  constexpr uint32_t kWavesHere = kSliceThreads / kWave;
  constexpr uint32_t kStep = 2 * kWave;  // words per step of a wave
  constexpr int kAhead = 2;
  __shared__ alignas(16) uint32_t s_bits[kSliceMax / 32 * 31];
  const uint32_t span = st->slice_span;  // the slice's chunks
  if (!span) return;  // block-uniform
  const uint32_t l = threadIdx.x % kWave;
  const uint32_t w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint32_t bw = span / 32 * 31;  // the slice's bitmap words
  const uint32_t slice = blockIdx.x, slices = gridDim.x;
  const uint32_t first = slice * span;
  const uint64_t key_a = st->range[0], w0 = st->range[2], w1 = st->range[3];
  const uint32_t keys = (uint32_t)(st->range[1] - key_a);
  const uint64_t total = w1 - w0;
  words += w0;
  for (uint32_t i = threadIdx.x; i < bw; i += kSliceThreads) s_bits[i] = 0;
  __syncthreads();
  auto literal = [&](uint32_t c, uint32_t bits) {
    const uint32_t rel = c - first;
    if (rel >= span) return;
    const uint32_t row = 31u * rel, wi = row >> 5, sh = row & 31u;
    atomicOr(&s_bits[wi], bits << sh);
    const uint32_t hi = (uint32_t)(((uint64_t)bits << sh) >> 32);
    if (hi) atomicOr(&s_bits[wi + 1], hi);
  };
  auto ones = [&](uint32_t c, uint32_t n) {  // a 1-fill's part of the slice
    const uint32_t a = c > first ? c - first : 0u;
    const uint64_t e = (uint64_t)c + n < first ? 0u : (uint64_t)c + n - first;
    for (uint32_t i = a; i < span && i < e; ++i) literal(first + i, 0x7FFFFFFFu);
  };
  for (uint32_t k0 = 0; k0 < keys; k0 += kSliceThreads) {
    // lane l holds one key of the wave's 64: its words of the slice
    const uint32_t k = k0 + w + kWavesHere * l;
    uint32_t from = 0, to = 0, at = 0;
    if (k < keys) {
      const uint64_t e = table[(uint64_t)slice * keys + k];
      const uint64_t f = slice + 1 < slices ? table[(uint64_t)(slice + 1) * keys + k] : 0;
      uint64_t end = k + 1 < keys ? (uint64_t)offsets[key_a + k + 1] - w0 : total;
      if (end > total) end = total;
      if (f && (uint32_t)f < end) end = (uint32_t)f;  // with the word that enters the next slice
      if (e && (uint32_t)e <= end) {
        from = (uint32_t)e - 1u;
        to = (uint32_t)end;
        at = (uint32_t)(e >> 32);
      }
    }
    uint64_t left = ballot(from < to);
    // the steps of the wave's keys, one after another; a step's words are
    // loaded while the steps before it are worked on (kAhead of them take
    // turns: a copy from one to the next would wait for its loads)
    uint32_t pos = 0, stop = 0;  // uniform
    struct Step {
      uint2 x;        // words 2l, 2l + 1 (past the key's end: fills of nothing)
      uint32_t c;     // first chunk
      bool on, same;  // there is one; it goes on where the last one ended
    };
    auto next = [&]() -> Step {
      Step q;
      q.c = 0;
      q.same = stop - pos > kStep;
      if (q.same) {
        pos += kStep;
      } else if (left) {
        const int j = __builtin_ctzll(left);
        left &= left - 1;
        pos = readlane(from, j);
        stop = readlane(to, j);
        q.c = readlane(at, j);
      } else {
        pos = stop = 0;
      }
      q.on = stop != 0;
      const uint32_t i = pos + 2 * l;
      q.x = uint2{0u, 0u};
      if (i < stop) q.x.x = words[i];
      if (i + 1 < stop) q.x.y = words[i + 1];
      return q;
    };
    Step q[kAhead];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) q[i] = next();
    uint32_t base = 0;
    for (bool on = true; on;) {
#pragma unroll
      for (int i = 0; i < kAhead; ++i) {
        const Step p = q[i];
        on = p.on;
        if (!on) break;
        if (!p.same) base = p.c;
        const uint32_t n0 = word_chunks(p.x.x), n1 = word_chunks(p.x.y);
        const uint32_t inc = wave_incl_add(n0 + n1);
        const uint32_t c0 = base + inc - n0 - n1;
        if (p.x.x & 0x80000000u) literal(c0, p.x.x & 0x7FFFFFFFu);
        if (p.x.y & 0x80000000u) literal(c0 + n0, p.x.y & 0x7FFFFFFFu);
        if (ballot(p.x.x >> 30 == 1u || p.x.y >> 30 == 1u)) {  // 1-fills, which builds never write
          if (p.x.x >> 30 == 1u) ones(c0, n0);
          if (p.x.y >> 30 == 1u) ones(c0 + n0, n1);
        }
        base += readlane(inc, kWave - 1);
        q[i] = next();
      }
    }
  }
  __syncthreads();
  const uint64_t nwords = (nrows + 31) / 32, out = (uint64_t)slice * bw;
  const uint32_t tail = (uint32_t)(nrows & 31u);
  for (uint32_t i = threadIdx.x; i < bw && out + i < nwords; i += kSliceThreads) {
    uint32_t v = s_bits[i];
    if (tail && out + i == nwords - 1) v &= (1u << tail) - 1u;
    bitmap[out + i] = v;
  }
}

// ---- encoding a row bitmap (or op(a, b) of two) into WAH words -------------

namespace {

// A lane owns 8 consecutive chunks, 248 rows; a wave 512 chunks, which are
// 15872 rows and so whole bitmap words (496); a tile 4096 chunks, 3968 words.
constexpr int kEncItems = 8;
constexpr uint32_t kEncTile = kScanThreads * kEncItems;
static_assert(((1ull << 32) + 30) / 31 <= kScanStatusWords * kEncTile, "2^32 rows");
constexpr uint32_t kEncWaveWords = kWave * kEncItems * 31 / 32;
constexpr uint32_t kEncWords = kEncWaveWords * kScanWaves;
static_assert(kWave * kEncItems * 31 % 32 == 0 && kEncWords % 4 == 0, "whole words per wave");

__device__ __forceinline__ uint32_t combine_bits(int op, uint32_t a, uint32_t b) {
  switch (op) {
    case 0: return a & b;   // AND
    case 1: return a | b;   // OR
    case 2: return a ^ b;   // XOR
    default: return a & ~b; // AND NOT
  }
}

}  // namespace

// One pass over a row bitmap (TWO: over a op b, combined word by word as they
// are loaded): per nonempty chunk c a fill of the chunks skipped since the
// last nonempty one, when there are any, then the literal.  Whether c has a
// fill word depends on chunk c - 1 alone, so the word count of a tile is known
// without its neighbours and the look-back is a plain sum of words, with the
// maximum of the nonempty chunks beside it for the one fill per tile that
// starts in an earlier tile.  The bitmap goes through LDS (a lane's 248 rows
// start off its words), the words too.  Words past cap are not written.
template <bool TWO>
__global__ __launch_bounds__(kScanThreads, query_waves_per_eu(kEncBlocks)) void k_q_encode(
    const uint32_t* __restrict__ a, const uint32_t* __restrict__ b, int op, uint64_t nrows,
    uint32_t* __restrict__ out, uint64_t cap, ScanState* st, uint64_t* status, uint32_t tiles,
    uint64_t* host) {
  // the tile's bitmap words (one before them, one after), then its WAH words
  __shared__ alignas(16) uint32_t s_buf[2 * kEncTile];
  __shared__ uint32_t s_words[kScanWaves], s_first[kScanWaves], s_last[kScanWaves];
  __shared__ uint32_t s_prefix, s_tile;
  static_assert(kEncWords + 5 <= 2 * kEncTile, "the bitmap words fit");
  uint32_t* const s_bits = s_buf + 4;  // 16-byte aligned, room for the word before
  const int l = threadIdx.x % kWave;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint64_t nwords = (nrows + 31) / 32;
  const uint32_t tail = (uint32_t)(nrows & 31u);  // rows of the last word (0: all 32)
  for (uint32_t tile = scan_next_tile(st, &s_tile, tiles, true); tile < tiles;
       tile = scan_next_tile(st, &s_tile, tiles, false)) {
    const uint64_t wbase = (uint64_t)tile * kEncWords;
    const uint32_t c0 = tile * kEncTile;  // chunks are below 2^28
    auto load = [&](auto full_tag) {
      constexpr bool FULL = decltype(full_tag)::value;
#pragma unroll
      for (uint32_t h = 0; h < 2; ++h) {
        const uint32_t qd = h * kScanThreads + threadIdx.x;
        if (4 * qd < kEncWords) {
          const uint64_t g = wbase + 4 * qd;
          W4 x = load4<FULL>(a, g, nwords);
          if (TWO) {
            const W4 y = load4<FULL>(b, g, nwords);
            x.x = combine_bits(op, x.x, y.x);
            x.y = combine_bits(op, x.y, y.y);
            x.z = combine_bits(op, x.z, y.z);
            x.w = combine_bits(op, x.w, y.w);
          }
          if (!FULL && tail && nwords - 1 - g < 4) {  // rows past nrows
            const uint32_t m = (1u << tail) - 1u;
            const uint32_t k = (uint32_t)(nwords - 1 - g);
            x.x &= k == 0 ? m : ~0u;
            x.y &= k == 1 ? m : ~0u;
            x.z &= k == 2 ? m : ~0u;
            x.w &= k == 3 ? m : ~0u;
          }
          *reinterpret_cast<W4*>(&s_bits[4 * qd]) = x;
        }
      }
    };
    if (wbase + kEncWords < nwords) load(std::true_type{});
    else load(std::false_type{});
    if (threadIdx.x == 0) {
      uint32_t x = 0;
      if (tile) {
        x = a[wbase - 1];
        if (TWO) x = combine_bits(op, x, b[wbase - 1]);
      }
      s_bits[-1] = x;
      s_bits[kEncWords] = 0;
    }
    __syncthreads();
    // the lane's 248 rows from bit 0 of v[0] on, then its chunks
    uint32_t e[kEncItems];
    {
      const uint32_t bit = (uint32_t)l * (kEncItems * 31u);
      const uint32_t* p = s_bits + w * kEncWaveWords + (bit >> 5);
      uint32_t x[9], v[8];
#pragma unroll
      for (int i = 0; i < 9; ++i) x[i] = p[i];
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = __builtin_amdgcn_alignbit(x[i + 1], x[i], bit & 31u);
      e[0] = v[0] & 0x7FFFFFFFu;
#pragma unroll
      for (int i = 1; i < kEncItems; ++i)
        e[i] = __builtin_amdgcn_alignbit(v[i], v[i - 1], 32u - (uint32_t)i) & 0x7FFFFFFFu;
    }
    uint32_t ne = 0;  // nonempty chunks of the lane
#pragma unroll
    for (int i = 0; i < kEncItems; ++i) ne |= e[i] ? 1u << i : 0u;
    // the chunk before the lane's first: nonempty?  (before chunk 0: no fill)
    const uint32_t before_wave = s_bits[(int)(w * kEncWaveWords) - 1] >> 1;
    const uint32_t cw = c0 + (uint32_t)w * kWave * kEncItems;  // the wave's first chunk
    const uint32_t pb = lane_before(ne >> (kEncItems - 1), cw == 0 || before_wave ? 1u : 0u);
    const uint32_t fm = ne & ~(ne << 1 | pb);  // chunks whose literal follows a fill
    const uint32_t cnt = (uint32_t)(__builtin_popcount(ne) + __builtin_popcount(fm));
    const uint32_t inc = wave_incl_add(cnt);
    // last nonempty chunk (+ 1) before the lane, within the wave
    const uint64_t hm = ballot(ne != 0u);
    const uint64_t below = hm & ((1ull << l) - 1ull);
    const uint32_t top = 32u - (uint32_t)__builtin_clz(ne | 1u);
    const int src = below ? 63 - __builtin_clzll(below) : 0;
    const uint32_t got = __shfl(top, src, kWave);
    uint32_t prev = below ? cw + (uint32_t)src * kEncItems + got : 0u;
    {
      const int lo = hm ? __builtin_ctzll(hm) : 0, hi = hm ? 63 - __builtin_clzll(hm) : 0;
      const uint32_t low = (uint32_t)__builtin_ctz(ne | 0x100u);
      const uint32_t f = readlane(low, lo), g = readlane(top, hi);
      if (l == 0) {
        s_words[w] = readlane(inc, kWave - 1);
        s_first[w] = hm ? cw + (uint32_t)lo * kEncItems + f + 1u : 0u;  // chunk + 1
        s_last[w] = hm ? cw + (uint32_t)hi * kEncItems + g : 0u;        // chunk + 1
      }
    }
    __syncthreads();  // the bitmap words are consumed: s_buf takes the WAH words
    uint32_t all = 0, wpos = 0, last = 0, wprev = 0, first = 0;
#pragma unroll
    for (int i = 0; i < kScanWaves; ++i) {
      if (i == w) {
        wpos = all;
        wprev = last;
      }
      all += s_words[i];
      if (!first) first = s_first[i];
      if (s_last[i]) last = s_last[i];
    }
    if (!prev) prev = wprev;
    uint32_t pos = wpos + inc - cnt;
#pragma unroll
    for (int i = 0; i < kEncItems; ++i) {
      if ((ne >> i) & 1u) {
        const uint32_t c = cw + (uint32_t)l * kEncItems + i;
        if ((fm >> i) & 1u) {
          // the tile's first entry takes its fill from the look-back, below
          if (prev) s_buf[pos] = c - prev;
          ++pos;
        }
        s_buf[pos++] = 0x80000000u | e[i];
        prev = c + 1u;
      }
    }
    if (w == 0) {
      uint32_t ph, pw;
      lookback2<kOpMax, kOpSum>(status, tile, last, all, false, &st->fault, ph, pw);
      if (l == 0) {
        s_prefix = pw;
        // a first entry right after the tile before's last chunk (or chunk 0)
        // has no fill and its literal stays
        if (first && first - 1u != ph) s_buf[0] = first - 1u - ph;
        if (tile == tiles - 1) st_agent(&st->result, (uint64_t)pw + all);
      }
    }
    __syncthreads();
    const uint64_t pre = s_prefix;
    if (pre < cap) store_staged(s_buf, out + pre, cap - pre < all ? (uint32_t)(cap - pre) : all);
  }
  scan_finish(st, status, tiles, host);
}

// ---- launchers ---------------------------------------------------------------

void launch_decode(const ScanRun& s, const DecodeStream& a, const DecodeStream& b, uint64_t nrows,
                   hipStream_t st) {
  const uint64_t tiles = (a.len + kDecTile - 1) / kDecTile + (b.len + kDecTile - 1) / kDecTile;
  if (!tiles) return;
  const uint32_t most = s.cus * kDecBlocks;
  hipLaunchKernelGGL(k_q_decode<false>, dim3(tiles < most ? (uint32_t)tiles : most),
                     dim3(kScanThreads), 0, st, a, b, nullptr, nrows, nullptr, 0u,
                     s.state, s.status, s.host);
}

void launch_range(const ScanRun& s, const uint32_t* keys, const uint32_t* offsets,
                  const uint32_t* lengths, uint64_t keycnt, const uint32_t* words,
                  uint64_t most_words, uint32_t lo, uint32_t hi, uint32_t* bitmap, uint64_t nrows,
                  uint64_t* table, uint64_t table_cap, bool grow, hipStream_t st) {
  const uint64_t bw = (nrows + 31) / 32;
  uint64_t g = (bw + 4 * kBlock - 1) / (4 * kBlock);
  const uint32_t span = table_cap ? slice_span_of(nrows, s.cus) : 0u;
  const uint32_t slices = span ? (uint32_t)slices_of(nrows, span) : 0u;
  if (span) {
    g = g < 1 ? 1 : g > 1024 ? 1024 : g;
    hipLaunchKernelGGL(k_q_range<true>, dim3((uint32_t)g), dim3(kBlock), 0, st, keys, offsets,
                       lengths, keycnt, lo, hi, most_words, bitmap, bw, table, table_cap, slices, span,
                       grow, s.state, s.host);
  } else {
    g = g < 1 ? 1 : g > 4096 ? 4096 : g;
    hipLaunchKernelGGL(k_q_range<false>, dim3((uint32_t)g), dim3(kBlock), 0, st, keys, offsets,
                       lengths, keycnt, lo, hi, most_words, bitmap, bw, table, table_cap, slices, span,
                       grow, s.state, s.host);
  }
  // the words of the range are known on the device only: a full grid
  hipLaunchKernelGGL(k_q_decode<true>, dim3(s.cus * kDecBlocks), dim3(kScanThreads), 0, st,
                     DecodeStream{words, 0, bitmap}, DecodeStream{nullptr, 0, nullptr}, offsets,
                     nrows, table, slices, s.state, s.status, s.host);
  if (span)
    hipLaunchKernelGGL(k_q_slices, dim3(slices), dim3(kSliceThreads), 0, st, words, offsets, table,
                       bitmap, nrows, s.state);
}

void launch_encode(const ScanRun& s, const uint32_t* a, const uint32_t* b, int op, uint64_t nrows,
                   uint32_t* out, uint64_t cap, hipStream_t st) {
  const uint64_t chunks = (nrows + 30) / 31;
  const uint32_t tiles = (uint32_t)((chunks + kEncTile - 1) / kEncTile);
  if (!tiles) return;
  const uint32_t most = s.cus * kEncBlocks, grid = tiles < most ? tiles : most;
  if (b)
    hipLaunchKernelGGL(k_q_encode<true>, dim3(grid), dim3(kScanThreads), 0, st, a, b, op, nrows,
                       out, cap, s.state, s.status, tiles, s.host);
  else
    hipLaunchKernelGGL(k_q_encode<false>, dim3(grid), dim3(kScanThreads), 0, st, a, b, op, nrows,
                       out, cap, s.state, s.status, tiles, s.host);
}

}  // namespace wah
