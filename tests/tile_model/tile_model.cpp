// Runs the tile rules of wah_tiles.h over launches whose blocks do not all get
// a place: each XCD has some slots, work on other streams holds all but a few of
// them for good, and the dispatcher places an XCD's blocks in order as its
// slots free up.  A placed block takes a tile, publishes it, and holds its slot
// until every earlier tile is published, then takes the next one or ends.  The
// launch must finish every tile once, whatever is withheld, as long as each XCD
// keeps one slot.
//
// Then the wait of the scans' look-back: predecessors that come one after another,
// each short of the limit, are waited for however many there are, in one window
// of 64 and over several; one that never comes is given up at the limit.
//
// Argument: "shipped", or "indexed" for the rule that these kernels must not
// have (a block's first tile is its index even where it stays for more), which
// the model has to see stall.
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include <random>
#include <vector>

#include "wah_tiles.h"

namespace {

enum Rule { kScan, kScanIndexed, kRadix };

struct Launch {
  Rule rule;
  uint32_t tiles, grid, group;
  uint32_t lanes() const { return wah::tile_lanes(grid); }
};

// Tiles finished (each must be 1); false: a stall or a tile taken twice.
bool run(const Launch& L, const std::vector<uint32_t>& slots) {
  struct Block {
    bool placed = false, ended = false, first = true;
    uint32_t tile = UINT32_MAX;  // held
  };
  std::vector<Block> blocks(L.grid);
  std::vector<uint32_t> used(wah::kTileLanes, 0), draws(wah::kTileLanes, 0);
  std::vector<uint8_t> published(L.tiles, 0);
  uint32_t upto = 0, finished = 0;  // tiles below upto are published
  const uint32_t lanes = L.lanes();
  const uint32_t g = L.rule == kRadix ? wah::tile_group(L.tiles, L.grid, lanes, L.group) : 1u;
  auto take = [&](uint32_t b) -> uint32_t {
    const uint32_t lane = b % lanes;
    Block& k = blocks[b];
    const bool first = k.first;
    k.first = false;
    if (L.rule == kScanIndexed) {
      if (first) return b;
      const uint32_t own = (L.grid - lane + lanes - 1) / lanes;
      return (own + draws[lane]++) * lanes + lane;
    }
    if (L.rule == kScan && !wah::scan_draws(L.tiles, L.grid)) return first ? b : L.tiles;
    return wah::drawn_tile(draws[lane]++, lanes, lane, g);
  };
  for (bool moved = true; moved;) {
    moved = false;
    for (uint32_t b = 0; b < L.grid; ++b) {
      Block& k = blocks[b];
      if (k.ended) continue;
      const uint32_t xcd = b % wah::kTileLanes;
      if (!k.placed) {
        bool earlier = false;  // an XCD's blocks are placed in order
        for (uint32_t e = xcd; e < b; e += wah::kTileLanes) earlier |= !blocks[e].placed;
        if (earlier || used[xcd] == slots[xcd]) continue;
        k.placed = true;
        ++used[xcd];
      } else if (k.tile != UINT32_MAX) {
        while (upto < L.tiles && published[upto]) ++upto;
        if (upto < k.tile) continue;  // waits for an earlier tile
        ++finished;
      }
      moved = true;
      k.tile = take(b);
      if (k.tile >= L.tiles) {
        k.ended = true;
        --used[xcd];
      } else {
        if (published[k.tile]) return false;
        published[k.tile] = 1;
      }
    }
  }
  return finished == L.tiles;
}

// A walk over `windows` windows of which each tile comes `gap` polls after the one
// before (never, from tile `lost` on).  Polls until it ended or gave up.
bool walk(uint32_t windows, uint32_t gap, uint32_t lost, uint64_t* polls) {
  wah::ScanWait wait;
  *polls = 0;
  for (uint32_t w = 0; w < windows; ++w) {
    uint64_t empty = ~0ull;
    for (uint32_t t = 0; t < 64; ++t) {
      const bool never = w * 64 + t >= lost;
      for (uint64_t p = 0; never || p < gap; ++p, ++*polls)
        if (wait.poll(empty)) return false;
      empty &= empty - 1;
    }
    wait.next_window();
  }
  return true;
}

int waits() {
  uint64_t polls = 0;
  int bad = 0;
  bad += !walk(1, wah::kSpinLimit - 1, ~0u, &polls);      // 63 limits in one window
  bad += !walk(3, wah::kSpinLimit / 2, ~0u, &polls);      // over three
  bad += walk(1, 0, 0, &polls) || polls != wah::kSpinLimit - 1;  // (the last poll gives up)
  bad += walk(2, 5, 70, &polls) || polls != 70 * 5 + wah::kSpinLimit - 1;
  if (bad) printf("%d waits wrong\n", bad);
  return bad;
}

}  // namespace

int main(int argc, char** argv) {
  const bool indexed = argc > 1 && !strcmp(argv[1], "indexed");
  std::mt19937 rng(7);
  uint32_t stalls = 0, runs = 0;
  for (const Rule rule : {indexed ? kScanIndexed : kScan, kRadix}) {
    for (const uint32_t grid : {1u, 3u, 8u, 9u, 16u, 40u, 64u}) {
      for (const uint32_t tiles : {1u, 2u, 7u, 8u, 9u, 17u, 39u, 40u, 41u, 64u, 65u, 130u, 400u}) {
        for (uint32_t rep = 0; rep < 20; ++rep) {
          std::vector<uint32_t> slots(wah::kTileLanes);
          for (auto& s : slots) s = rep == 0 ? 64u : rep == 1 ? 1u : 1u + rng() % 8u;
          const Launch L{rule, tiles, grid, rep % 2 ? 8u : 4u};
          ++runs;
          if (!run(L, slots)) {
            if (!indexed) printf("stall: rule %d grid %u tiles %u rep %u\n", rule, grid, tiles, rep);
            ++stalls;
          }
        }
      }
    }
  }
  printf("%u of %u launches stalled\n", stalls, runs);
  return stalls != 0 || waits() != 0;
}
