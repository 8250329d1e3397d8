// CPU check of the raster's work items when a batch's bin list is too small
// (tile_items, common.h).  A model of the list as the kernels fill it: the
// direct pairs of each tile from its end downwards as long as they alone fit
// (stage_direct), then the scanned pairs from its start up to its capacity
// (stage_bin).  Whatever the raster is then given to draw, every entry it
// reads has to be one of its own tile.  Prints "ok" or the first failure.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "common.h"

using namespace mr;

static uint64_t st = 1;
static uint32_t rnd(uint32_t n) {
  uint64_t z = (st += 0x9E3779B97F4A7C15ull);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  return (uint32_t)((z ^ (z >> 31)) % n);
}

int main(int argc, char** argv) {
  const int cases = argc > 1 ? atoi(argv[1]) : 10000;
  int drawn = 0, mixed = 0;
  for (int c = 0; c < cases; c++) {
    const int ntiles = 1 + (int)rnd(12);
    const uint32_t cap = 1 + rnd(100);
    std::vector<uint32_t> scan(ntiles), direct(ntiles), off(ntiles), first(ntiles, ~0u);
    std::vector<int> bins(cap, -1);  // the tile of each entry, -1: not written
    unsigned long long counters[kNumCounters] = {};
    for (int t = 0; t < ntiles; t++) {
      scan[t] = rnd(3) ? rnd(20) : 0;
      direct[t] = rnd(2) ? rnd(20) : 0;
    }
    for (int t = 0; t < ntiles; t++) {  // offsets, counts and the tile list
      off[t] = (uint32_t)counters[kBinEntries];
      counters[kBinEntries] += scan[t];
      if (scan[t]) counters[kListed]++;
      else if (direct[t]) counters[kDirectTilesListed]++;
      if (!direct[t]) continue;
      const unsigned long long pos = counters[kDirectPairs];
      counters[kDirectPairs] += direct[t];
      if (pos + direct[t] > cap) continue;
      first[t] = (uint32_t)(cap - pos - direct[t]);
      for (uint32_t i = 0; i < direct[t]; i++) bins[first[t] + i] = t;
    }
    if (counters[kBinEntries] > cap) counters[kBinOverflow] = 1;
    for (int t = 0; t < ntiles; t++)
      for (uint32_t i = 0; i < scan[t] && off[t] + i < cap; i++) bins[off[t] + i] = t;
    counters[kBinEntries] += counters[kDirectPairs];  // check_direct_room
    if (counters[kBinEntries] > cap) counters[kBinOverflow] = 1;

    const TileItems items = tile_items(counters, 64, ntiles);
    if (items.parts < 0 || items.whole > items.listed || items.listed > ntiles) {
      printf("case %d: items out of range\n", c);
      return 1;
    }
    if (counters[kBinEntries] <= cap && items.listed != (int64_t)(counters[kListed] + counters[kDirectTilesListed])) {
      printf("case %d: tiles left out of a list that holds all\n", c);
      return 1;
    }
    if (items.listed + items.parts == 0) continue;
    drawn++;
    for (int t = 0; t < ntiles; t++) {
      mixed += scan[t] && direct[t];
      for (uint32_t i = 0; i < scan[t] && off[t] + i < cap; i++)
        if (bins[off[t] + i] != t) {
          printf("case %d: tile %d reads an entry of tile %d\n", c, t, bins[off[t] + i]);
          return 1;
        }
      for (uint32_t i = 0; first[t] != ~0u && i < direct[t]; i++)
        if (bins[first[t] + i] != t) {
          printf("case %d: tile %d reads a direct entry of tile %d\n", c, t, bins[first[t] + i]);
          return 1;
        }
    }
  }
  // A part list that ran over: no parts, whole tiles as they are.
  unsigned long long k[kNumCounters] = {};
  k[kParts] = 9, k[kListed] = 3, k[kHeavyOverflow] = 1;
  const TileItems h = tile_items(k, 4, 16);
  k[kHeavyOverflow] = 0;
  if (h.parts != 0 || h.listed != 3 || tile_items(k, 4, 16).parts != 4 || !drawn || !mixed) {
    printf("parts\n");
    return 1;
  }
  printf("ok\n");
  return 0;
}
