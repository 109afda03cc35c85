// wah_tiles.h -- which tile a block of a single-pass launch takes: the rules
// that the waits of such a launch end by, as plain functions, so that they can
// be run against a model of partly placed launches on the host.
#pragma once

#include <stdint.h>

namespace wah {

constexpr uint32_t kTileLanes = 8;
constexpr uint32_t kLaneStride = 64;

// Counter lanes for a grid of `grid` blocks.
constexpr uint32_t tile_lanes(uint32_t grid) {
  return grid < kTileLanes ? (grid ? grid : 1u) : kTileLanes;
}

// Tile of a lane's j-th draw: lane, lane + lanes, ... or, with group > 1, runs
// of `group` consecutive tiles per lane.  Workgroups are dispatched to the 8
// XCDs round robin, so lane = block % 8 is the XCD, and neighbouring tiles then
// write the cache lines they share (the ends of their output runs) through one
// L2, which merges them.  A lane's draws ascend with any group, so the lowest
// unfinished tile is held by a running block or is its lane's next draw, which
// any block of the lane makes: look-back waits end as long as each lane has a
// block placed.
constexpr uint32_t drawn_tile(uint32_t j, uint32_t lanes, uint32_t lane, uint32_t group = 1) {
  return group == 1 ? j * lanes + lane
                    : (j / group) * group * lanes + lane * group + j % group;
}

// Group of a radix or tail launch over `tiles` tiles: `group` where the blocks
// draw several tiles each.  Where there is a block for every tile, the tiles
// are dealt to the lanes in equal runs, so that each lane has as many tiles as
// blocks (a grid of a multiple of the lanes): with runs of 8, 18 tiles lay in
// three lanes of 2 or 3 blocks, which took them in turn while the other lanes'
// blocks found nothing (a radix pass over 300,007 rows 41 us, over 2^20 rows
// 14 us).
constexpr uint32_t tile_group(uint32_t tiles, uint32_t grid, uint32_t lanes, uint32_t group) {
  return tiles <= grid ? (tiles + lanes - 1) / lanes : group;
}

// The scans of wah_scan.h.  With a block for every tile a block takes the tile
// of its own index, ends after it and so frees its place for the next block:
// that saves the smallest calls two draws.  With more tiles than blocks every
// tile, a block's first one too, is drawn: a block that stays for another tile
// then never waits for a tile that belongs to a block without a place, which
// work on another stream may withhold for as long as it runs.  (That draw costs
// the encode of 2^27 rows, 1058 tiles, 18.7 -> 21.3 us and three primitives of
// 2^24 elements 144 -> 148; the next tile drawn ahead of its use 24 and 154.)
constexpr bool scan_draws(uint32_t tiles, uint32_t grid) { return tiles > grid; }

// Polls of a look-back wait that see nothing new before it gives up.
constexpr uint32_t kSpinLimit = 1u << 18;

// The wait of a scan's look-back: `waiting` is the set of tiles of its window
// that it still waits for.  The limit counts from the last change of that set
// (a tile published, or the next window), not over the whole walk, so tiles that
// come slowly one after another are waited for as long as each of them may take.
struct ScanWait {
  uint32_t polls = 0;
  uint64_t waiting = 0;
  // One more poll that found `now` unpublished; true: give up.
  constexpr bool poll(uint64_t now) {
    if (now != waiting) {
      waiting = now;
      polls = 0;
    }
    return ++polls >= kSpinLimit;
  }
  constexpr void next_window() {
    waiting = 0;
    polls = 0;
  }
};

}  // namespace wah
