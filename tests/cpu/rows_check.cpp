// CPU check of cover_rows (exact.h): for random triangles (small, large,
// slivers, vertices far beyond the screen, axis-aligned edges) and column ranges, no
// row it drops covers a pixel in the raster's own walk (edge_start at the
// bbox's left column, e += n.x per column, Renderer.cpp:238-245), and it
// drops most rows that cover nothing.  Also: xcd_chunks (common.h) is a
// bijection on [0, n).  Built with g++ -O2 -ffp-contract=off.
// Prints "ok" or the first failure.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "common.h"
#include "exact.h"

using namespace mr;

static uint64_t st;
static uint64_t rnd() {
  uint64_t z = (st += 0x9E3779B97F4A7C15ull);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}
static double u01() { return (double)(rnd() >> 11) / 9007199254740992.0; }

int main(int argc, char** argv) {
  const int cases = argc > 1 ? atoi(argv[1]) : 100000;
  st = argc > 2 ? strtoull(argv[2], nullptr, 10) : 1;
  for (uint32_t n = 1; n < 1200; n++) {
    std::vector<char> seen(n, 0);
    for (uint32_t b = 0; b < n; b++) {
      const uint32_t r = xcd_chunks<kXcdChunk>(b, n);
      if (r >= n || seen[r]++) {
        printf("xcd_chunks(%u, %u) = %u\n", b, n, r);
        return 1;
      }
    }
  }
  long empty = 0, dropped = 0, tested = 0;
  for (int i = 0; i < cases; i++) {
    const float W = (float)(16 + rnd() % 500), H = (float)(16 + rnd() % 300);
    const int kind = (int)(rnd() % 6);
    const double size = kind == 0 ? 8.0 : kind == 1 ? 60.0 : kind == 2 ? 800.0 : kind == 3 ? 40000.0 : 300.0;
    const double cx = u01() * W, cy = u01() * H;
    ScreenVtx v[3];
    for (int k = 0; k < 3; k++) {
      v[k].px = (float)(cx + (u01() - 0.5) * size);
      v[k].py = (float)(cy + (u01() - 0.5) * size);
      v[k].zv = 1.0f;
    }
    if (kind == 4) v[1].px = v[0].px, v[2].py = v[0].py;  // edges along the axes
    if (kind == 5) {                                       // slivers
      v[2].px = v[0].px + (v[1].px - v[0].px) * 0.7f;
      v[2].py = v[0].py + (v[1].py - v[0].py) * 0.7f + (float)((u01() - 0.5) * 0.02);
    }
    if (rnd() % 16 == 0) {  // a vertex 2^10 to 2^31 pixels away
      ScreenVtx& f = v[rnd() % 3];
      const double r = ldexp(1.0 + u01(), 10 + (int)(rnd() % 22)), a = u01() * 6.2831853;
      f.px += (float)(r * cos(a));
      f.py += (float)(r * sin(a));
    }
    TriSetup s;
    if (!setup_screen(W, H, v[0], v[1], v[2], s) &&
        !setup_screen(W, H, v[2], v[1], v[0], s))
      continue;
    const int tw = 8 << (rnd() % 3);
    const int tx = (int)(rnd() % ((uint64_t)W / tw + 1)), ty = (int)(rnd() % ((uint64_t)H / tw + 1));
    const int c0 = s.bx0 > tx * tw ? s.bx0 : tx * tw, c1 = s.bx1 < tx * tw + tw - 1 ? s.bx1 : tx * tw + tw - 1;
    const int a0 = s.by0 > ty * tw ? s.by0 : ty * tw, a1 = s.by1 < ty * tw + tw - 1 ? s.by1 : ty * tw + tw - 1;
    if (c0 > c1 || a0 > a1) continue;
    int r0 = a0, r1 = a1;
    cover_rows(s, c0, c1, r0, r1);
    if (r0 < a0 || r1 > a1) {
      printf("case %d: rows [%d, %d] outside [%d, %d]\n", i, r0, r1, a0, a1);
      return 1;
    }
    for (int row = a0; row <= a1; row++) {
      float e1, e2;
      edge_start(s.n1x, s.n1y, s.n2x, s.n2y, s.p0x, s.p0y, s.p2x, s.p2y, (float)s.bx0 + 0.5f,
                 (float)row + 0.5f, e1, e2);
      bool any = false;
      for (int c = s.bx0; c <= c1; c++) {
        if (c >= c0 && covered(e1, e2)) any = true;
        e1 = e1 + s.n1x;
        e2 = e2 + s.n2x;
      }
      const bool kept = row >= r0 && row <= r1;
      tested++;
      if (any && !kept) {
        printf("case %d: row %d covered but dropped ([%d, %d])\n", i, row, r0, r1);
        return 1;
      }
      empty += !any;
      dropped += !any && !kept;
    }
  }
  if (dropped * 2 < empty) {
    printf("dropped %ld of %ld rows that cover nothing (%ld rows)\n", dropped, empty, tested);
    return 1;
  }
  printf("ok\n");
  return 0;
}
