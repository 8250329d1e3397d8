// CPU check of how a tile's direct entries are shared out (common.h): the
// parts of a split tile draw each entry once and about as many each, and a
// tile of few is drawn in bands that cover its rows once, that the raster's
// grid holds, and that leave no workgroup with all rows of a long list while
// the GPU has room.  Prints "ok" or the first failure.
#include <cstdio>
#include <cstdlib>
#include <initializer_list>

#include "common.h"

using namespace mr;

#define FAIL(...) (printf(__VA_ARGS__), printf("\n"), exit(1))

int main() {
  const uint32_t sizes[] = {0, 1, 15, 16, 17, 255, 256, 1023, 4095, 4096, 0xFFFFFFF0u};
  for (uint32_t n : sizes)
    for (uint32_t parts = 1; parts < 70; parts++) {
      uint32_t at = 0;
      for (uint32_t p = 0; p < parts; p++) {
        const DirectShare s = direct_share(n, p, parts);
        if (s.first != at || s.end < s.first || s.end - s.first > n / parts + 1)
          FAIL("%u entries, part %u of %u: %u - %u", n, p, parts, s.first, s.end);
        at = s.end;
      }
      if (at != n) FAIL("%u entries in %u parts: %u drawn", n, parts, at);
    }
  const int heights[] = {8, 16, 32};
  for (int h : heights)
    for (int ntiles = 1; ntiles < 9000; ntiles = ntiles < 1200 ? ntiles + 1 : ntiles * 2)
      for (unsigned long long direct : {0ull, 255ull, 256ull, 4096ull, 1000000ull})
        for (uint32_t parts_cap : {0u, 100u, 4000u})
          for (int listed : {0, 1, (ntiles + 1) / 2, ntiles})
            for (int64_t parts : {(int64_t)0, (int64_t)parts_cap}) {
              unsigned long long k[kNumCounters] = {};
              k[kDirect] = direct;
              const TileItems r = {parts, listed, listed};
              const int n = whole_bands(k, r, parts_cap, ntiles, h);
              if (n < 1 || n > 8 || h % n) FAIL("%d bands of %d rows", n, h);
              if (r.parts + n * r.listed > (int64_t)ntiles + parts_cap) FAIL("%d bands: more than the grid", n);
              if (n > 1 && (direct < kBandDirect || n * r.listed > kBandGroups)) FAIL("%d bands of %d tiles", n, listed);
              if (direct >= 4096 && ntiles <= 128 && parts_cap == 4000 && parts == 0 && n != 8)
                FAIL("%d bands of %d tiles: workgroups to spare", n, ntiles);
            }
  printf("ok\n");
  return 0;
}
