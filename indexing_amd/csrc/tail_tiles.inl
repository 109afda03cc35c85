// tail_tiles.inl -- the tiles of one sort mode (RUN) in k_tail, included in the
// kernel's body once per mode it runs.
  const Dims dims = desc->dims;
  const Column* cols = desc_cols(desc);
  // the wave index in a scalar register: per-wave LDS addresses stay out of
  // the 64 vector registers
  const int t = threadIdx.x, l = t % kWave;
  const int w = __builtin_amdgcn_readfirstlane(t / kWave);
  uint32_t* fault = &hdr->fault;

  uint32_t iter = 0;
  if (hdr->mode_cols[RUN ? 1 : 0] != 0)  // some column in this mode
  for (;;) {
    const uint32_t tile = __builtin_amdgcn_readfirstlane(next_tile(
        &hdr->tiles[RUN ? kCounterRunTail : kCounterTail][0], lanes, &s_tile, iter,
        tile_group(dims.tail_tiles, gridDim.x, lanes, WAH_TAIL_TILE_GROUP)));
    if (tile >= dims.tail_tiles) break;
    const uint32_t c = find_segment(&cols[0].tail_tile0, sizeof(Column) / 4, dims.ncols, tile);
    const Column cd = cols[c];
    const uint32_t first_tile = cd.tail_tile0;
    // column-local indices fit 32 bits: a column holds fewer than 2^30 items
    const uint32_t base = (tile - first_tile) * (uint32_t)TILE;
    // items: rows, or the runs of a run-mode column (fewer than its tiles)
    const uint32_t n = RUN ? (uint32_t)cs[c].items : (uint32_t)cd.n;
    if (cs[c].mode != (RUN ? kModeRun : kModePair) || base >= n) {
      if (RUN && c + 1 == dims.ncols && cs[c].mode == kModeRun) break;  // past the last items
      __syncthreads();  // s_tile is read by every wave before it is rewritten
      continue;
    }
    // the tile's body, compiled once per key width (16-bit keys load 8 per
    // 16 bytes); the column's width picks one
    // and once for whole aligned tiles (16-byte loads, no per-item checks,
    // and no control-flow merge with the per-item loads of partial tiles)
    const SortedView sv0 =
        sorted_view(&cs[c], cd, values, keysA, ridsA, keysB, ridsB, litsA, litsB);
    const bool aligned = (((uintptr_t)sv0.keys | (uintptr_t)sv0.rids |
                           (RUN ? (uintptr_t)sv0.lits : (uintptr_t)0)) % 16) == 0;
    auto body = [&](auto narrow_tag, auto full_tag) {
    constexpr bool NARROW = decltype(narrow_tag)::value;
    constexpr bool FULL = decltype(full_tag)::value;
    const uint32_t rid_base = cd.rid_base;
    SortedView sv = sv0;
    sv.narrow = NARROW;
    const uint32_t j0 = base + (uint32_t)t * ITEMS;  // the lane's first item
    const uint32_t nv =
        FULL ? (uint32_t)ITEMS
             : (n > j0 ? (n - j0 < (uint32_t)ITEMS ? n - j0 : (uint32_t)ITEMS) : 0u);

    // Loads the tile needs besides its own items, issued before them so that
    // one memory latency covers all: the item before the wave (lane 0's
    // predecessor; wave-uniform) and, for the last wave, the 32 items after
    // the tile (the run that crosses its end).
    // Branch-free: out-of-range indices read item 0 and are masked later
    // (an implicit-rid column's rids array is the unused ping-pong buffer).
    const uint32_t gw = base + (uint32_t)(w * kWave * ITEMS);
    const bool have_pred = gw > 0 && gw <= n;
    const uint32_t gp = have_pred ? gw - 1 : 0u;
    uint32_t k0 = sv.key(gp), r0 = sv.rids[gp];
    const uint32_t gn0 = base + (uint32_t)TILE + (uint32_t)l;
    const bool nv_next = w == WAVES - 1 && l < 32 && gn0 < n;
    const uint32_t gn = nv_next ? gn0 : 0u;
    uint32_t kk = 0, rr = 0, ll = 0;
    if (w == WAVES - 1) {
      kk = sv.key(gn);
      rr = sv.rids[gn];
      if (RUN) ll = sv.lits[gn];
    }

    // ---- items of the lane: key, chid, literal bits (0 past the column)
    uint32_t key[ITEMS], ch[ITEMS], b[ITEMS];
    if constexpr (FULL) {
      if (NARROW) {  // 8 keys per 16-byte load
#pragma unroll
        for (int q = 0; q < ITEMS / 8; ++q) {
          const uint4 k8 = reinterpret_cast<const uint4*>(reinterpret_cast<const uint16_t*>(sv.keys) + j0)[q];
          const uint32_t w4[4] = {k8.x, k8.y, k8.z, k8.w};
#pragma unroll
          for (int h = 0; h < 4; ++h) {
            key[8 * q + 2 * h] = w4[h] & 0xFFFFu;
            key[8 * q + 2 * h + 1] = w4[h] >> 16;
          }
        }
      }
#pragma unroll
      for (int q = 0; q < ITEMS / 4; ++q) {
        if (!NARROW) {
          const uint4 k4 = reinterpret_cast<const uint4*>(sv.keys + j0)[q];
          key[4 * q] = k4.x; key[4 * q + 1] = k4.y; key[4 * q + 2] = k4.z; key[4 * q + 3] = k4.w;
        }
        // loaded either way (an implicit-rid column reads the unused
        // buffer), so the loads are not split by a branch
        const uint4 r4 = reinterpret_cast<const uint4*>(sv.rids + j0)[q];
        ch[4 * q] = r4.x; ch[4 * q + 1] = r4.y; ch[4 * q + 2] = r4.z; ch[4 * q + 3] = r4.w;
        if (RUN) {
          const uint4 l4 = reinterpret_cast<const uint4*>(sv.lits + j0)[q];
          b[4 * q] = l4.x; b[4 * q + 1] = l4.y; b[4 * q + 2] = l4.z; b[4 * q + 3] = l4.w;
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < ITEMS; ++i) {
        const bool v = (uint32_t)i < nv;
        const uint32_t g = j0 + i;
        key[i] = v ? sv.key(g) : 0u;
        ch[i] = v ? (sv.implicit ? rid_base + g : sv.rids[g]) : 0u;
        if (RUN) b[i] = v ? sv.lits[g] : 0u;
      }
    }
    if (FULL && sv.implicit) {
#pragma unroll
      for (int i = 0; i < ITEMS; ++i) ch[i] = rid_base + j0 + (uint32_t)i;
    }
    // ch[] held rids so far: chunk id q = rid / 31 and the literal bit
    // rid % 31 = (rid + q) & 31 (rid + q = 32q + rid % 31).  Rows below 2^31
    // (every column with rid_base + n <= 2^31) divide by a multiply-high,
    // exact there (it first fails at 2369637147); the others by the
    // compiler's full 32-bit division.
    auto chunks = [&](auto fast_tag) {
      constexpr bool FAST = decltype(fast_tag)::value;
#pragma unroll
      for (int i = 0; i < ITEMS; ++i) {
        const uint32_t r = ch[i];
        const uint32_t q = FAST ? __umulhi(r, 0x84210843u) >> 4 : r / 31u;
        ch[i] = q;
        if (!RUN) b[i] = (uint32_t)i < nv ? 1u << ((r + q) & 31u) : 0u;
      }
    };
    if ((uint64_t)rid_base + cd.n <= (1ull << 31)) chunks(std::true_type{});
    else chunks(std::false_type{});
    // predecessor of the lane's first item: lane l-1's last, or for lane 0
    // the item before the wave (one load per wave)
    uint32_t pk, pc;
    {
      // first use of the side loads, tied to the tile's own (so that no
      // arithmetic on them is placed, with its wait, before those loads)
      k0 = __builtin_amdgcn_readfirstlane(k0);
      r0 = __builtin_amdgcn_readfirstlane(r0);
      asm volatile("" : "+s"(k0), "+s"(r0) : "v"(key[ITEMS - 1]), "v"(ch[ITEMS - 1]));
      if (!have_pred) k0 = r0 = 0u;
      else if (sv.implicit) r0 = rid_base + gp;
      const uint32_t c0 = r0 / 31u;
      pk = (uint32_t)__builtin_amdgcn_update_dpp((int)k0, (int)key[ITEMS - 1], 0x138, 0xF, 0xF, false);
      pc = (uint32_t)__builtin_amdgcn_update_dpp((int)c0, (int)ch[ITEMS - 1], 0x138, 0xF, 0xF, false);
    }
    // ---- entry and key starts, fills, counts
    const bool colfirst = base == 0 && t == 0;
    uint32_t f[ITEMS];
    uint32_t stm = 0, khm = 0, fm = 0;  // per item: entry start, key start, nonzero fill
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      const uint32_t kp = i ? key[i - 1] : pk, cp = i ? ch[i - 1] : pc;
      const bool v = (uint32_t)i < nv;
      const bool kh = v && (key[i] != kp || (i == 0 && colfirst));
      const bool st = kh || (v && ch[i] != cp);
      f[i] = st ? (kh ? ch[i] : ch[i] - cp - 1u) : 0u;
      stm |= st ? 1u << i : 0u;
      khm |= kh ? 1u << i : 0u;
      fm |= f[i] != 0u ? 1u << i : 0u;
    }
    // From here on an item's flags are read back from these bits: the
    // compiler would otherwise keep each item's compare masks (64-bit scalar
    // pairs) alive to the staging and spill them to VGPR lanes.
    stm = opaque(stm);
    khm = opaque(khm);
    fm = opaque(fm);
    const uint32_t nwords = (uint32_t)(__builtin_popcount(stm) + __builtin_popcount(fm));
    // lead bits: items before the lane's first stop (entry start or end of items)
    const uint32_t stops = stm | (~0u << nv & kAll);
    const uint32_t fs = stops ? (uint32_t)__builtin_ctz(stops) : (uint32_t)ITEMS;
    uint32_t lead = 0;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) lead |= (uint32_t)i < fs ? b[i] : 0u;
    // continuation of the lane's last run inside the wave: leads of lanes
    // l+1 .. the next lane with a stop (at most 4 lanes on)
    const uint64_t hsm = ballot(stops != 0u);
    const uint64_t above = l == kWave - 1 ? 0ull : hsm >> (l + 1);
    const uint32_t dist = above ? (uint32_t)__builtin_ctzll(above) + 1u : 64u;
    uint32_t cont = 0;
    {
      uint32_t sh = lead;
#pragma unroll
      for (uint32_t s = 1; s <= 4; ++s) {
        sh = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)sh, 0x130, 0xF, 0xF, false);  // wave_shl:1
        cont |= s <= dist ? sh : 0u;
      }
    }
    // wave lead: lane 0's items before its first stop and, without one, the
    // lanes after it
    {
      const uint32_t wl = readlane(stops ? lead : lead | cont, 0);
      if (l == 0) s_wlead[w] = wl;
    }
    // next tile's lead: the run that crosses the tile end (last wave, 32 items)
    if (w == WAVES - 1) {
      const bool v = nv_next;
      if (sv.implicit) rr = rid_base + gn;
      uint32_t cc = 0, bb = 0;
      if (!v) kk = 0u;
      if (v) {
        cc = rr / 31u;
        bb = RUN ? ll : 1u << (rr - cc * 31u);
      }
      const uint32_t kl = readlane(key[ITEMS - 1], kWave - 1), cl = readlane(ch[ITEMS - 1], kWave - 1);
      const uint32_t kq = (uint32_t)__builtin_amdgcn_update_dpp((int)kl, (int)kk, 0x138, 0xF, 0xF, false);
      const uint32_t cq = (uint32_t)__builtin_amdgcn_update_dpp((int)cl, (int)cc, 0x138, 0xF, 0xF, false);
      const uint64_t sm = ballot(!v || kk != kq || cc != cq);  // lanes 32.. always stop
      const int fh = __builtin_ctzll(sm);
      const uint32_t tl = wave_or(l < fh ? bb : 0u);
      if (l == 0) s_wlead[WAVES] = tl;
    }
    // tile-local word and key offsets: one wave scan of (keys << 16 | words)
    const uint32_t packed = ((uint32_t)__builtin_popcount(khm) << 16) | nwords;
    const uint32_t inc = wave_incl_add(packed);
    if (l == kWave - 1) s_wtot[w] = inc;
    {
      // entries of the tile (k of the column is their sum, formed by k_finish)
      const uint32_t e = readlane(wave_incl_add((uint32_t)__builtin_popcount(stm)), kWave - 1);
      if (l == 0) s_went[w] = e;
    }
    __syncthreads();

    // ---- literals: reverse sweep along the lane, seeded with the bits the
    // lane's last run picks up from the lanes (wave, tile) after it
    if (above == 0) cont |= s_wlead[w + 1];
    if (nv < (uint32_t)ITEMS) cont = 0;  // the run ends with the items
    uint32_t woff, tot;
    {
      // wave totals: one LDS read per lane and a wave scan
      const uint32_t lo = opaque((uint32_t)l);
      const uint32_t x = lo < WAVES ? s_wtot[lo] : 0u;
      const uint32_t xi = wave_incl_add(x);
      woff = readlane(xi - x, __builtin_amdgcn_readfirstlane(w));
      tot = readlane(xi, WAVES - 1);
    }
    const uint32_t lpos = woff + inc - packed;  // (keys << 16 | words) before the lane
    if (w == 0) {
      const uint64_t tile_agg = ((uint64_t)(tot >> 16) << 31) | (tot & 0xFFFFu);
      const uint64_t pre = lookback_wave_sum<WAH_TAIL_LOOKBACK_SLOTS>(status, tile, first_tile,
                                                                      tile_agg, fault);
      const uint32_t lo = opaque((uint32_t)l);
      const uint32_t e = readlane(wave_incl_add(lo < WAVES ? s_went[lo] : 0u), kWave - 1);
      if (l == 0) {
        s_prefix = pre;
        tile_entries[tile] = e;
      }
    }
    {
      // from the lane's last word back: [fill,] literal of each entry start
      uint32_t carry = cont;
      uint32_t pos = (lpos & 0xFFFFu) + nwords;
#pragma unroll
      for (int i = ITEMS - 1; i >= 0; --i) {
        const bool st = (stm >> i) & 1u, fw = (fm >> i) & 1u;
        carry |= b[i];
        pos -= st ? 1u : 0u;
        if (st) s_words[pos + (pos >> 4)] = 0x80000000u | carry;
        pos -= fw ? 1u : 0u;
        if (fw) s_words[pos + (pos >> 4)] = f[i];
        carry = st ? 0u : carry;
      }
    }
    uint32_t kv[ITEMS];
    if (khm) {
      // key starts: the values (the lane's keys read again, all at once:
      // the lines are still in L2) and the position of each key's first word
      if (nv == (uint32_t)ITEMS && aligned && !NARROW) {
#pragma unroll
        for (int q = 0; q < ITEMS / 4; ++q) {
          const uint4 k4 = reinterpret_cast<const uint4*>(sv.keys + j0)[q];
          kv[4 * q] = k4.x; kv[4 * q + 1] = k4.y; kv[4 * q + 2] = k4.z; kv[4 * q + 3] = k4.w;
        }
      } else if (nv == (uint32_t)ITEMS && aligned) {
#pragma unroll
        for (int q = 0; q < ITEMS / 8; ++q) {
          const uint4 k8 = reinterpret_cast<const uint4*>(reinterpret_cast<const uint16_t*>(sv.keys) + j0)[q];
          const uint32_t w4[4] = {k8.x, k8.y, k8.z, k8.w};
#pragma unroll
          for (int h = 0; h < 4; ++h) {
            kv[8 * q + 2 * h] = w4[h] & 0xFFFFu;
            kv[8 * q + 2 * h + 1] = w4[h] >> 16;
          }
        }
      } else {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) kv[i] = (uint32_t)i < nv ? sv.key(j0 + i) : 0u;
      }
    }
    __syncthreads();  // words staged, prefix published
    const uint64_t pre = s_prefix;
    const uint32_t Wpre = (uint32_t)(pre & 0x7FFFFFFFu), Kpre = (uint32_t)(pre >> 31);
    uint32_t* out_keys = keys_out + cd.off;
    uint32_t* out_offsets = offsets_out + cd.off;
    uint32_t* out_words = words_out + 2 * cd.off;
    if (khm) {
      bool bad = false;
#pragma unroll
      for (int i = 0; i < ITEMS; ++i) {
        if ((khm >> i) & 1u) {
          const uint32_t below = (1u << i) - 1u;
          const uint32_t kg = Kpre + (lpos >> 16) + __builtin_popcount(khm & below);
          const uint32_t wp = (lpos & 0xFFFFu) + __builtin_popcount(stm & below) +
                              __builtin_popcount(fm & below);
          bad |= kg >= n;
          const uint32_t kc = kg < n ? kg : n - 1u;  // stores stay in the column
          out_keys[kc] = kv[i];
          out_offsets[kc] = Wpre + wp;
        }
      }
      if (bad) atomicOr(fault, 2u);
    }
    const uint32_t Wt = tot & 0xFFFFu;
    if ((uint64_t)Wpre + Wt <= 2ull * n) {
      // single words up to the first 16-byte boundary, then 4 words per
      // 16-byte store, then the rest
      uint32_t* ow = out_words + Wpre;
      const uint32_t head0 = (4u - (uint32_t)(((uintptr_t)ow >> 2) & 3u)) & 3u;
      const uint32_t head = head0 < Wt ? head0 : Wt;
      const uint32_t quads = (Wt - head) / 4u;
      const uint32_t tt = opaque((uint32_t)t);
      if (tt < head) ow[tt] = s_words[tt + (tt >> 4)];
      for (uint32_t qd = tt; qd < quads; qd += THREADS) {
        const uint32_t j = head + 4u * qd;
        uint4 v;
        v.x = s_words[j + (j >> 4)];
        v.y = s_words[j + 1u + ((j + 1u) >> 4)];
        v.z = s_words[j + 2u + ((j + 2u) >> 4)];
        v.w = s_words[j + 3u + ((j + 3u) >> 4)];
        *reinterpret_cast<uint4*>(ow + j) = v;  // 16-byte aligned: j - head is a multiple of 4
      }
      for (uint32_t j = head + 4u * quads + tt; j < Wt; j += THREADS) ow[j] = s_words[j + (j >> 4)];
    } else {
      for (uint32_t j = opaque((uint32_t)t); j < Wt; j += THREADS) {
        const uint32_t o = Wpre + j;
        if (o < 2 * n) out_words[o] = s_words[j + (j >> 4)];
        else atomicOr(fault, 2u);
      }
    }
    if (base + TILE >= n && t == 0) {  // the column's last tile
      counts[cd.index].length = (uint64_t)Wpre + Wt;
      counts[cd.index].keycnt = (uint64_t)Kpre + (tot >> 16);
    }
    };
    const bool full = base + TILE <= n && aligned;
    if (cs[c].narrow) {
      if (full) body(std::true_type{}, std::true_type{});
      else body(std::true_type{}, std::false_type{});
    } else {
      if (full) body(std::false_type{}, std::true_type{});
      else body(std::false_type{}, std::false_type{});
    }
    // the next tile's first barrier (in next_tile) orders these LDS reads
    // before its writes
  }
