// radix_tiles.inl -- the tiles of one sort mode (RUN) in k_onesweep, included in
// the kernel's body once per mode it runs.  (As a function or a lambda the same
// code loses the kernel's restrict pointers or keeps its captures in scratch:
// 4% more instructions, and launch 1 of 2^28 rows 872 us instead of 836.)

  // pair mode: launch 0 reads the values (rids implicit); run mode: the run
  // cut wrote the items to B.  Then A -> B, B -> A, ...
  const bool implicit = !RUN && a == 0;
  const uint32_t* src_keys = implicit ? values : ((a % 2) ? keysA : keysB);
  const uint32_t* src_rids = (a % 2) ? ridsA : ridsB;
  const uint32_t* src_lits = (a % 2) ? litsA : litsB;
  uint32_t* dst_keys = (a % 2) ? keysB : keysA;
  uint32_t* dst_rids = (a % 2) ? ridsB : ridsA;
  uint32_t* dst_lits = (a % 2) ? litsB : litsA;
  uint32_t* status = status_base + (uint64_t)(a % 2) * status_stride;
  uint32_t* status_next = status_base + (uint64_t)(1u - a % 2) * status_stride;
  uint32_t* fault = &hdr->fault;
  const Dims dims = desc->dims;
  const Column* cols = desc_cols(desc);
  const int t = threadIdx.x, l = t % kWave;
  const int w = __builtin_amdgcn_readfirstlane(t / kWave);  // scalar: per-wave LDS addresses
  uint32_t* counter = hdr->tiles[(RUN ? kCounterRun : 0) + a];

  uint32_t iter = 0;
  if (hdr->max_active[RUN ? 1 : 0] > a)  // some column has an a-th pass
  for (;;) {
    for (int i = t; i < WAVES * 256; i += THREADS) (&s_wcnt[0][0])[i] = 0;
    const uint32_t tile = __builtin_amdgcn_readfirstlane(
        next_tile(counter, lanes, &s_tile, iter, tile_group(dims.sort_tiles, gridDim.x, lanes, WAH_SORT_TILE_GROUP)));
    if (tile >= dims.sort_tiles) break;
    const uint32_t c = find_segment(&cols[0].sort_tile0, sizeof(Column) / 4, dims.ncols, tile);
    const ColState* col = &cs[c];
    const Column cd = cols[c];
    const uint32_t first = cd.sort_tile0;
    const uint64_t base = (uint64_t)(tile - first) * TILE;  // column-local
    // elements: rows, or the run items of a run-mode column
    const uint64_t n = RUN ? (uint64_t)col->items : cd.n;
    const uint64_t n_out = n;
    if (col->mode != (RUN ? kModeRun : kModePair) || col->wide || col->num_active <= a ||
        base >= n) {
      // other mode, already sorted, or past the run items; a block draws its
      // tiles in increasing order, so past the last column's items it is done
      if (RUN && c + 1 == dims.ncols && col->mode == kModeRun && base >= n) break;
      __syncthreads();  // s_tile is read by every wave before it is rewritten
      continue;
    }
    const uint32_t shift = col->shift[a];
    // 16-bit keys: every pass writes them; the first reads the values (or
    // the run cut's items) as 32-bit words
    const bool narrow = col->narrow != 0u, src_narrow = narrow && !implicit && !(RUN && a == 0);
    if (t < 256) status_next[(uint64_t)tile * 256 + t] = 0;  // next launch's state
    const uint64_t wbase = base + (uint64_t)w * kWave * ITEMS + l;
    // The body is straight-line, so the compiler can wait for the rid loads
    // without draining the key stores, and the ranking atomics issue back to
    // back.  A column's last tile runs it too: items past its end read the
    // last one, count in a word of their own instead of a digit's, and keep
    // their own index as their slot (they are the tile's last in input order,
    // so those slots lie past tile_n), which nothing stores.
    // PACKED: launch 0 of a pair-mode column with keys < 2^16.  Its rids are
    // implicit (rid_base + column row), so one LDS word carries both the key
    // (high half) and the row's tile-local index (low half): one staging
    // round moves keys and rids.
    auto sweep = [&](auto full_tag, auto packed_tag) {
      constexpr bool FULL = decltype(full_tag)::value;
      constexpr bool PACKED = decltype(packed_tag)::value;
      // Keys only for now: the rids are loaded once the keys are staged, so
      // they never occupy registers during ranking and look-back.
      uint32_t key[ITEMS], rank[ITEMS];
      // item i of an array of the column (indices fit 32 bits): one base and
      // immediate offsets in a whole tile; past the column its last item
      // (first: the lane's first item, opaque per array so that the clamped
      // indices are formed again instead of spilled across the ranking)
      const uint32_t j0 = (uint32_t)wbase, jl = (uint32_t)n - 1u;
      auto item = [&](const auto* col0, int i, uint32_t first) -> uint32_t {
        if (FULL) return (uint32_t)(col0 + wbase)[i * kWave];
        const uint32_t j = first + (uint32_t)(i * kWave);
        return (uint32_t)col0[j < jl ? j : jl];
      };
      if (src_narrow) {
        const uint16_t* kp = reinterpret_cast<const uint16_t*>(src_keys + cd.off);
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) key[i] = item(kp, i, j0);
      } else {
        const uint32_t* kp = src_keys + cd.off;
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) key[i] = item(kp, i, j0);
      }
      const uint32_t tile_n = FULL ? (uint32_t)TILE : (uint32_t)(n - base);
      // Rank: peers = lanes with the same digit (8 ballots); rank = peers
      // below this lane + keys of that digit the wave ranked before.
#pragma unroll
      for (int i = 0; i < ITEMS; ++i) {
        const uint32_t d = (key[i] >> shift) & 255u;
        const bool in = FULL || j0 + (uint32_t)(i * kWave) <= jl;
        if (RANK == kRankAtomic) {
          rank[i] = atomicAdd(in ? &s_wcnt[w][d] : &s_stage[t], 1u);
        } else {
          uint64_t peers = ballot(in);
#pragma unroll
          for (int b = 0; b < 8; ++b) {
            const bool bit = (d >> b) & 1u;
            const uint64_t bb = ballot(bit);
            peers &= bit ? bb : ~bb;
          }
          const uint32_t cnt = (uint32_t)__popcll(peers);
          const uint32_t below = mbcnt(peers);
          const uint32_t prior = s_wcnt[w][d];
          rank[i] = prior + below;
          if (in && below == cnt - 1) s_wcnt[w][d] = prior + cnt;
        }
      }
      __syncthreads();
      // Threads 0..255 own one digit each: wave prefixes, tile total,
      // exclusive scan over digits, look-back.
      uint32_t total = 0;
      if (t < 256) {
        const uint32_t goff = col->digit_offset[shift / 8][t];
        // all the wave counts first (independent reads), then the prefixes:
        // interleaved, each read would wait for the write before it
        uint32_t xw[WAVES];
#pragma unroll
        for (int i = 0; i < WAVES; ++i) xw[i] = s_wcnt[i][t];
#pragma unroll
        for (int i = 0; i < WAVES; ++i) {
          s_wcnt[i][t] = total;
          total += xw[i];
        }
        uint32_t* my = &status[(uint64_t)tile * 256 + t];
        st_agent(my, ((tile == first ? kFlagPrefix : kFlagAgg) << 30) | total);
        const uint32_t inc = wave_incl_add(total);
        if (l == kWave - 1) s_dsum[w] = inc;
        s_excl[t] = inc - total;  // within this wave's 64 digits
        uint32_t prev = 0;
        if (tile > first) {
          prev = lookback_digit(status + t, tile, first, 256, fault);
          st_agent(my, (kFlagPrefix << 30) | (prev + total));
        }
        s_glob[t] = goff + prev;  // the tile-local offset is subtracted below
      }
      __syncthreads();
      if (t < 256) {
        uint32_t before = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) before += i < w ? s_dsum[i] : 0u;
        const uint32_t ex = s_excl[t] + before;
        s_glob[t] -= ex;  // column index = s_glob[d] + local index
        // each wave's first slot for digit t: one LDS read per key below
        uint32_t xw[WAVES];
#pragma unroll
        for (int i = 0; i < WAVES; ++i) xw[i] = s_wcnt[i][t];
#pragma unroll
        for (int i = 0; i < WAVES; ++i) s_wcnt[i][t] = xw[i] + ex;
      }
      __syncthreads();
      if constexpr (PACKED) {
        const uint32_t row0 = (uint32_t)(wbase - base);  // tile-local index of item 0
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
          const uint32_t d = (key[i] >> shift) & 255u, row = row0 + (uint32_t)(i * kWave);
          const uint32_t pos = s_wcnt[w][d] + rank[i];
          s_stage[FULL || row < tile_n ? pos : row] = key[i] << 16 | row;
        }
        __syncthreads();
        uint16_t* dk16 = reinterpret_cast<uint16_t*>(dst_keys + cd.off);
        uint32_t* dr = dst_rids + cd.off;
        const uint32_t last = (uint32_t)(n_out - 1);  // stores stay in the column
        const uint32_t rid0 = cd.rid_base + (uint32_t)base;
        bool bad = false;
        // the staged words, then their digits' offsets, then the stores: each
        // batch of LDS reads issues back to back (slots past tile_n hold the
        // items past the column and store nothing)
        uint32_t xs[ITEMS], gs[ITEMS];
#pragma unroll
        for (int j = 0; j < ITEMS; ++j) xs[j] = s_stage[(uint32_t)j * THREADS + t];
#pragma unroll
        for (int j = 0; j < ITEMS; ++j) gs[j] = s_glob[(xs[j] >> (16 + shift)) & 255u];
#pragma unroll
        for (int j = 0; j < ITEMS; ++j) {
          const uint32_t q = (uint32_t)j * THREADS + t;
          if (FULL || q < tile_n) {
            const uint32_t g = gs[j] + q;
            bad |= g > last;
            const uint32_t gc = g < last ? g : last;
            dk16[gc] = (uint16_t)(xs[j] >> 16);
            dr[gc] = rid0 + (xs[j] & 0xFFFFu);
          }
        }
        if (ballot(bad) && l == 0) atomicOr(fault, 2u);  // a scatter index past the column
        return;
      }
#pragma unroll
      for (int i = 0; i < ITEMS; ++i) {
        const uint32_t d = (key[i] >> shift) & 255u;
        const uint32_t row = (uint32_t)(wbase - base) + (uint32_t)(i * kWave);
        const uint32_t pos = FULL || row < tile_n ? s_wcnt[w][d] + rank[i] : row;
        s_stage[pos] = key[i];
        rank[i] = pos;  // keep the LDS slot for the rids
      }
      // LDS slots, two per register (a tile has at most 2^16 items)
      uint32_t slot2[(ITEMS + 1) / 2];
#pragma unroll
      for (int i = 0; i < ITEMS; i += 2)
        slot2[i / 2] = (rank[i] & 0xFFFFu) | (i + 1 < ITEMS ? rank[i + 1 < ITEMS ? i + 1 : i] << 16 : 0u);
      // rids: issued now, in flight while the keys go out
      uint32_t rid[ITEMS];
      if (implicit) {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) rid[i] = cd.rid_base + (uint32_t)wbase + (uint32_t)(i * kWave);
      } else {
        const uint32_t* rp = src_rids + cd.off;
        const uint32_t first = FULL ? j0 : opaque(j0);
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) rid[i] = item(rp, i, first);
      }
      __syncthreads();
      uint32_t* dk = dst_keys + cd.off;
      uint32_t* dr = dst_rids + cd.off;
      const uint32_t last = (uint32_t)(n_out - 1);  // stores stay in the column
      bool bad = false;
      // destination of each slot this thread stores, kept for the rids (and
      // literal bits): the digit comes from the staged key
      uint32_t gq[ITEMS], kq[ITEMS];
      uint16_t* dk16 = reinterpret_cast<uint16_t*>(dk);
      // the staged keys, then their digits' offsets, then the stores: each
      // batch of LDS reads issues back to back (slots past tile_n hold the
      // items past the column and store nothing)
#pragma unroll
      for (int j = 0; j < ITEMS; ++j) kq[j] = s_stage[(uint32_t)j * THREADS + t];
#pragma unroll
      for (int j = 0; j < ITEMS; ++j) gq[j] = s_glob[(kq[j] >> shift) & 255u];
#pragma unroll
      for (int j = 0; j < ITEMS; ++j) {
        const uint32_t q = (uint32_t)j * THREADS + t;
        const uint32_t g = gq[j] + q;
        const bool in = FULL || q < tile_n;
        bad |= in && g > last;
        gq[j] = in && g < last ? g : last;
      }
      if (narrow) {
#pragma unroll
        for (int j = 0; j < ITEMS; ++j)
          if (FULL || (uint32_t)j * THREADS + t < tile_n) dk16[gq[j]] = (uint16_t)kq[j];
      } else {
#pragma unroll
        for (int j = 0; j < ITEMS; ++j)
          if (FULL || (uint32_t)j * THREADS + t < tile_n) dk[gq[j]] = kq[j];
      }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < ITEMS; ++i) s_stage[(slot2[i / 2] >> (16 * (i % 2))) & 0xFFFFu] = rid[i];
      if (RUN) {  // literal bits: issued now, in flight while the rids go out
        const uint32_t* lp = src_lits + cd.off;
        const uint32_t first = FULL ? j0 : opaque(j0);
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) rid[i] = item(lp, i, first);
      }
      __syncthreads();
#pragma unroll
      for (int j = 0; j < ITEMS; ++j) kq[j] = s_stage[(uint32_t)j * THREADS + t];
#pragma unroll
      for (int j = 0; j < ITEMS; ++j)
        if (FULL || (uint32_t)j * THREADS + t < tile_n) dr[gq[j]] = kq[j];
      if (RUN) {
        // literal bits of each run item, moved along with its key and rid
        __syncthreads();
#pragma unroll
        for (int i = 0; i < ITEMS; ++i)
          s_stage[(slot2[i / 2] >> (16 * (i % 2))) & 0xFFFFu] = rid[i];
        __syncthreads();
        uint32_t* dl = dst_lits + cd.off;
#pragma unroll
        for (int j = 0; j < ITEMS; ++j) kq[j] = s_stage[(uint32_t)j * THREADS + t];
#pragma unroll
        for (int j = 0; j < ITEMS; ++j)
          if (FULL || (uint32_t)j * THREADS + t < tile_n) dl[gq[j]] = kq[j];
      }
      if (ballot(bad) && l == 0) atomicOr(fault, 2u);  // a scatter index past the column
    };
    auto dispatch = [&](auto packed_tag) {
      if (base + TILE <= n) sweep(std::true_type{}, packed_tag);
      else sweep(std::false_type{}, packed_tag);
    };
    if constexpr (!RUN) {
      if (implicit && narrow) dispatch(std::true_type{});
      else dispatch(std::false_type{});
    } else {
      dispatch(std::false_type{});
    }
    __syncthreads();
  }
