// wah_small.hip -- the build of short columns, one workgroup each.
//
// A column of at most kSmallMax rows fits one CU's LDS, so one launch does
// what the general build does in a chain of launches: digits that vary, the
// sort mode, a stable LSD radix sort of (value, row), entries, literals, fills,
// words, keys, offsets and lengths.  Nothing but the column and its index
// touches memory, nothing waits for another workgroup, and no scratch is used.
// What bounds it is latency: a chain of LDS passes and barriers in one CU.
//
// 1000 rows of 10-bit values: 7 us a call, against 67 as the general build's 15
// launches; 4000 rows of 16-bit values 10 against 71, 8000 17 against 78,
// 16000 32 against 90.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "wah_scan.h"

namespace wah {

namespace {

constexpr int kThreads = 1024;
constexpr int kWaves16 = kThreads / kWave;
constexpr uint32_t kCntAt = kSmallMax + kSmallMax / 2;  // LDS word of the digit counts
constexpr uint32_t kDummyAt = kCntAt + kWaves16 * 256;  // and of the rows past the column
static_assert(kDummyAt + kThreads <= 2 * kSmallMax, "the sort's LDS fits the words'");
static_assert(kSmallMax == 16u * kThreads && 2 * kSmallMax < 65536, "16 rows a thread; 16-bit counts");

struct SmallShared {
  // sort: keys, 16-bit rows, the waves' digit counts; then the index's words
  alignas(16) uint32_t raw[2 * kSmallMax];
  uint32_t dsum[4];
  uint32_t vary[kWaves16], vmax[kWaves16], runs[kWaves16], tot[kWaves16], ent[kWaves16];
};

// Exclusive prefix of wave w over the 16 waves' values, and their sum.
__device__ __forceinline__ uint32_t before16(const uint32_t* x, int w, uint32_t* all) {
  const uint32_t l = lane_id();
  const uint32_t v = l < (uint32_t)kWaves16 ? x[l] : 0u;
  const uint32_t inc = wave_incl_add(v);
  *all = readlane(inc, kWaves16 - 1);
  return readlane(inc - v, w);
}

// ITEMS rows per thread, n <= 1024 ITEMS.
template <int ITEMS>
__device__ __forceinline__ void small_build(SmallShared& sh, const Column& cd, bool atomic_rank,
                                            const uint32_t* __restrict__ values,
                                            uint32_t* out_keys, uint32_t* out_offsets,
                                            uint32_t* out_lengths, uint32_t* out_words,
                                            wahgpu_counts_dev* counts) {
  const int t = threadIdx.x, l = t % kWave;
  const int w = __builtin_amdgcn_readfirstlane(t / kWave);
  const uint32_t n = (uint32_t)cd.n;
  const uint32_t* src = values + cd.off;
  uint32_t* const s_key = sh.raw;
  uint16_t* const s_row = reinterpret_cast<uint16_t*>(sh.raw + kSmallMax);
  uint32_t* const s_cnt = sh.raw + kCntAt + (uint32_t)w * 256u;  // the wave's counts

  // ---- rows in wave-striped order: row of item i is r0 + 64 i
  const uint32_t r0 = (uint32_t)w * (kWave * ITEMS) + (uint32_t)l;
  uint32_t key[ITEMS], row[ITEMS];
  const uint32_t v0 = src[0];
  const uint32_t wfirst = (uint32_t)w * (kWave * ITEMS);
  const uint32_t before_wave = wfirst > 0 && wfirst < n ? src[wfirst - 1] : 0u;
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    row[i] = r0 + (uint32_t)(i * kWave);
    key[i] = row[i] < n ? src[row[i]] : v0;
  }
  uint32_t vary = 0, vmax = 0, runs = 0;
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    vary |= key[i] ^ v0;
    vmax = key[i] > vmax ? key[i] : vmax;
    const uint32_t pv = lane_before(key[i], i ? readlane(key[i ? i - 1 : 0], kWave - 1) : before_wave);
    const bool rep = row[i] > 0 && (cd.rid_base + row[i]) % 31u != 0u && key[i] == pv;
    runs += row[i] < n && !rep ? 1u : 0u;
  }
  vary = wave_or(vary);
  vmax = wave_max(vmax);
  runs = wave_sum(runs);
  if (l == 0) {
    sh.vary[w] = vary;
    sh.vmax[w] = vmax;
    sh.runs[w] = runs;
  }
  __syncthreads();
  {
    const uint32_t lw = (uint32_t)l % kWaves16;
    vary = wave_or(sh.vary[lw]);
    vmax = wave_max(sh.vmax[lw]);
    runs = wave_sum(l < kWaves16 ? sh.runs[lw] : 0u);
  }

  // ---- stable LSD radix passes over the 8-bit digits that vary
  uint32_t passes = 0;
#pragma unroll 1
  for (uint32_t shift = 0; shift < 32; shift += 8) {
    if (((vary >> shift) & 255u) == 0u) continue;
    if (passes) {  // the keys and rows of the pass before, in its order
#pragma unroll
      for (int i = 0; i < ITEMS; ++i) {
        const uint32_t at = r0 + (uint32_t)(i * kWave);
        key[i] = s_key[at];
        row[i] = s_row[at];
      }
    }
    ++passes;
    for (uint32_t i = (uint32_t)t; i < kWaves16 * 256u; i += kThreads) sh.raw[kCntAt + i] = 0;
    __syncthreads();
    uint32_t rank[ITEMS];
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      const bool in = r0 + (uint32_t)(i * kWave) < n;
      const uint32_t d = (key[i] >> shift) & 255u;
      if (atomic_rank) {
        rank[i] = atomicAdd(in ? &s_cnt[d] : &sh.raw[kDummyAt + t], 1u);
      } else {
        uint64_t peers = ballot(in);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
          const bool bit = (d >> b) & 1u;
          const uint64_t bb = ballot(bit);
          peers &= bit ? bb : ~bb;
        }
        const uint32_t cnt = (uint32_t)__popcll(peers), below = mbcnt(peers);
        const uint32_t prior = s_cnt[d];
        rank[i] = prior + below;
        if (in && below == cnt - 1) s_cnt[d] = prior + cnt;
      }
    }
    __syncthreads();
    uint32_t total = 0, xw[kWaves16], inc = 0;
    if (t < 256) {
#pragma unroll
      for (int i = 0; i < kWaves16; ++i) xw[i] = sh.raw[kCntAt + i * 256 + t];
#pragma unroll
      for (int i = 0; i < kWaves16; ++i) {
        const uint32_t x = xw[i];
        xw[i] = total;
        total += x;
      }
      inc = wave_incl_add(total);
      if (l == kWave - 1) sh.dsum[w] = inc;
    }
    __syncthreads();
    if (t < 256) {
      uint32_t ex = inc - total;
#pragma unroll
      for (int i = 0; i < 4; ++i) ex += i < w ? sh.dsum[i] : 0u;
#pragma unroll
      for (int i = 0; i < kWaves16; ++i) sh.raw[kCntAt + i * 256 + t] = xw[i] + ex;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      const uint32_t at = r0 + (uint32_t)(i * kWave);
      const uint32_t pos = at < n ? s_cnt[(key[i] >> shift) & 255u] + rank[i] : at;
      s_key[pos] = key[i];
      s_row[pos] = (uint16_t)row[i];
    }
    __syncthreads();
  }

  // ---- sorted items in blocked order: thread t owns [t ITEMS, t ITEMS + ITEMS)
  const uint32_t j0 = (uint32_t)t * ITEMS;
  uint32_t pk = v0, pr = j0 - 1u;  // the item before the thread's
  if (passes) {
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      key[i] = s_key[j0 + i];
      row[i] = s_row[j0 + i];
    }
    if (j0 > 0) {
      pk = s_key[j0 - 1];
      pr = s_row[j0 - 1];
    }
  } else {
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      key[i] = v0;
      row[i] = j0 + i;
    }
  }
  __syncthreads();
  for (uint32_t i = 4u * t; i < 2u * n; i += 4u * kThreads)  // whole quads, inside raw
    *reinterpret_cast<W4*>(&sh.raw[i]) = W4{0u, 0u, 0u, 0u};

  uint32_t f[ITEMS], bit[ITEMS];
  uint32_t stm = 0, khm = 0, fm = 0;
  {
    uint32_t pc = (cd.rid_base + pr) / 31u;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      const uint32_t rid = cd.rid_base + row[i], ch = rid / 31u;
      const bool in = j0 + i < n;
      const bool kh = in && (j0 + i == 0 || key[i] != pk);
      const bool st = kh || (in && ch != pc);
      f[i] = st ? (kh ? ch : ch - pc - 1u) : 0u;
      bit[i] = 0x80000000u | 1u << (rid - 31u * ch);
      stm |= st ? 1u << i : 0u;
      khm |= kh ? 1u << i : 0u;
      fm |= f[i] ? 1u << i : 0u;
      pk = key[i];
      pc = ch;
    }
  }
  const uint32_t nwords = (uint32_t)(__builtin_popcount(stm) + __builtin_popcount(fm));
  const uint32_t packed = (uint32_t)__builtin_popcount(khm) << 16 | nwords;
  const uint32_t inc = wave_incl_add(packed);
  const uint32_t ents = wave_sum((uint32_t)__builtin_popcount(stm));
  if (l == kWave - 1) sh.tot[w] = inc;
  if (l == 0) sh.ent[w] = ents;
  __syncthreads();  // totals written, words zeroed
  uint32_t all, k;
  const uint32_t pre = before16(sh.tot, w, &all) + inc - packed;
  (void)before16(sh.ent, w, &k);
  const uint32_t L = all & 0xFFFFu, K = all >> 16;
  uint32_t* const ok = out_keys + cd.off;
  uint32_t* const oo = out_offsets + cd.off;
  uint32_t* const ol = out_lengths + cd.off;
  uint32_t* const ow = out_words + 2 * cd.off;
  {
    // an item's literal is the last word up to it: the words of a run of items
    // are ORed into it, one LDS OR per thread and entry
    uint32_t pos = pre & 0xFFFFu, ki = pre >> 16, bits = 0;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      if ((stm >> i) & 1u) {
        if (bits) atomicOr(&sh.raw[pos - 1u], bits);
        bits = 0;
        if ((khm >> i) & 1u) {
          ok[ki] = key[i];
          oo[ki] = pos;
          ++ki;
        }
        if ((fm >> i) & 1u) sh.raw[pos++] = f[i];
        ++pos;
      }
      bits |= j0 + i < n ? bit[i] : 0u;
    }
    if (bits) atomicOr(&sh.raw[pos - 1u], bits);
  }
  __syncthreads();  // words whole, offsets written
  store_staged(sh.raw, ow, L);
  for (uint32_t i = (uint32_t)t; i < K; i += kThreads) ol[i] = (i + 1 < K ? oo[i + 1] : L) - oo[i];
  if (t == 0) {
    wahgpu_counts_dev c;
    c.k = k;
    c.length = L;
    c.keycnt = K;
    c.bound = vmax;
    c.passes = passes;
    c.fault = 0;
    c.mode = 3ull * runs < 2ull * n ? kModeRun : kModePair;
    counts[cd.index] = c;
  }
}

}  // namespace

// Block c builds short column c of the descriptor (desc null: column `one`).
__global__ __launch_bounds__(kThreads, 4) void k_small(
    const DescHead* __restrict__ desc, Column one, int atomic_rank,
    const uint32_t* __restrict__ values, uint32_t* out_keys, uint32_t* out_offsets,
    uint32_t* out_lengths, uint32_t* out_words, wahgpu_counts_dev* counts) {
  __shared__ SmallShared sh;
  Column cd = one;
  if (desc) {
    if (blockIdx.x >= desc->dims.shorts) return;
    cd = desc_cols(desc)[desc->dims.ncols + blockIdx.x];
  }
  if (cd.n == 0) {
    if (threadIdx.x == 0) counts[cd.index] = wahgpu_counts_dev{};
    return;
  }
  if (cd.n <= kThreads)
    small_build<1>(sh, cd, atomic_rank, values, out_keys, out_offsets, out_lengths, out_words, counts);
  else if (cd.n <= 4 * kThreads)
    small_build<4>(sh, cd, atomic_rank, values, out_keys, out_offsets, out_lengths, out_words, counts);
  else if (cd.n <= 8 * kThreads)
    small_build<8>(sh, cd, atomic_rank, values, out_keys, out_offsets, out_lengths, out_words, counts);
  else
    small_build<16>(sh, cd, atomic_rank, values, out_keys, out_offsets, out_lengths, out_words, counts);
}

void launch_small(const BuildArgs& a, hipStream_t s) {
  hipLaunchKernelGGL(k_small, dim3(a.inline_desc ? 1u : a.shorts_cap), dim3(kThreads), 0, s,
                     a.inline_desc ? nullptr : a.desc, a.one, (int)a.atomic_rank, a.values,
                     a.out_keys, a.out_offsets, a.out_lengths, a.out_words, a.counts);
}

}  // namespace wah
