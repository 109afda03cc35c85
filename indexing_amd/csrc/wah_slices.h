// wah_slices.h -- when a range query decodes by slices of the row bitmap, and
// the table it needs for that: plain functions that the kernels (wah_query.hip)
// and the host (wahgpu_api.hip) share.
#pragma once

#include <stdint.h>

namespace wah {

// Slices of a range's bitmap, one block each: as many as CUs or a multiple of
// that (264 of 8192 chunks took 44 us for 2^26 rows, 256 of 8480 35: 8 CUs had
// two), of up to kSliceMax chunks.  A range of an index of 2^22 rows or more
// (below that the ORs it replaces take about what its launch does) decodes by
// slices if its words are kSliceWords or more per entry of the table: a wave
// works through a slice's part of a key in steps of 128 words, full or not.
// Slices / ORs: 18 words per entry (2800 keys of 2^26 rows) 179 / 283 us, 15
// (1800 of 2^24) 125 / 156, 13 (12000 of 2^26) 614 / 782, 10 (1000 of 2^26)
// 83 / 81, 8 (410 of 2^22) 52 / 45; 130 (410 of 2^26) 84 / 281.
constexpr uint32_t kSliceMax = 10240;
constexpr uint64_t kSliceMinRows = 1ull << 22;
constexpr uint64_t kSliceWords = 12;
static_assert(kSliceMax % 32 == 0, "a slice's span is rounded up to it at most");

// Chunks per slice: a multiple of 32, so that a slice is whole bitmap words.
constexpr uint32_t slice_span_of(uint64_t nrows, uint32_t cus) {
  if (nrows < kSliceMinRows) return 0;
  const uint64_t chunks = (nrows + 30) / 31, each = (uint64_t)cus * kSliceMax;
  const uint64_t slices = (chunks + each - 1) / each * cus;
  return (uint32_t)((chunks + slices * 32 - 1) / (slices * 32)) * 32;
}
constexpr uint64_t slices_of(uint64_t nrows, uint32_t span) {
  return ((nrows + 30) / 31 + span - 1) / span;
}

// Entries of the table of a range of `keys` keys and `words` words over `slices`
// slices; 0: it does not go by slices.
constexpr uint64_t slice_entries(uint64_t keys, uint64_t words, uint64_t slices) {
  const uint64_t entries = keys * slices;  // below 2^60
  return words < 1ull << 31 && words >= kSliceWords * entries ? entries : 0;
}

// Entries of the table that a query brings before it knows its range: enough
// for any range of the index, kTableFirst (8 MB) at most.  4096 keys of 2^26
// rows need as many.  A range that needs more asks for them (range_wants).
constexpr uint64_t kTableFirst = 1ull << 20;
constexpr uint64_t range_table_first(uint64_t keycnt, uint64_t nrows, uint32_t cus) {
  const uint32_t span = slice_span_of(nrows, cus);
  if (!span) return 0;
  const uint64_t all = keycnt * slices_of(nrows, span);
  return all < kTableFirst ? all : kTableFirst;
}
// Entries that a range of this many keys and words decodes by (0: by ORs).
constexpr uint64_t range_wants(uint64_t keys, uint64_t words, uint64_t nrows, uint32_t cus) {
  const uint32_t span = slice_span_of(nrows, cus);
  return span ? slice_entries(keys, words, slices_of(nrows, span)) : 0;
}

}  // namespace wah
