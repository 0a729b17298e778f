// CPU check of the 2-D cutting (lbgpu-prime-dev_amd/csrc/lbm_plan2d.hpp): for
// sizes over the whole range, devices with and without the LDS that the
// kernels are made for (0: not reported) and few or many compute units, a
// plan covers the lattice and keeps the kernels' limits, or is refused.
// Prints "ok" or the first violation.
#include <math.h>
#include <stdio.h>
#include <stdlib.h>

#include "lbm_plan2d.hpp"

using namespace lbm;

#define CHECK(x)                                                                                       \
  do {                                                                                                 \
    if (!(x)) {                                                                                        \
      printf("%d x %d, %d components, handed %d, LDS %d, %d CUs: %s\n", ni, nj, ns, handed, lds, cus, #x); \
      exit(1);                                                                                         \
    }                                                                                                  \
  } while (0)

static bool covers(int n, int size, int count) { return size > 0 && count > 0 && (long)size * count >= n && (long)size * (count - 1) < n; }

int main() {
  long plans = 0;
  for (int lds : {0, 1, 1000, 20000, 65536, 163840})
    for (int cus : {1, 32, 256, 304})
      for (int ns = 1; ns <= 2; ns++)
        for (int handed = 0; handed < 2; handed++)
          for (double x = 1; x < 32768; x = x * 1.23 + 0.4)
            for (double y = 1; x * y < 2e7; y = y * 1.31 + 0.3) {
              const int ni = (int)x, nj = (int)y;
              Plan2d P;
              if (!plan2d(ni, nj, ns, handed, lds, cus, P)) {
                CHECK(lds < 163840);  // the device that the kernels are made for takes every size
                continue;
              }
              plans++;
              CHECK(lds > 0 && P.lds > 0 && P.lds <= (size_t)lds);
              CHECK(P.steps >= 2 && P.steps <= kTileSteps && P.steps % 2 == 0);
              CHECK(P.shrink == (handed ? 3 : 2));
              if (P.sweep) {
                const SweepGeo &S = P.S;
                CHECK(ns == 2 && !handed && P.steps == kSweepSteps && P.threads == kSweepBlock);
                CHECK(covers(ni, S.cw, S.strips) && covers(nj, S.ch, S.pieces));
                CHECK(S.rw == S.cw + 2 * kSweepHalo && S.rw <= kSweepCols);
                CHECK(8 * S.blocks8 >= S.strips * S.pieces);
                CHECK(P.lds >= (size_t)S.rw * (kSweepRows * (9 * 16 + 8) + kSweepEntries * 8));
                continue;
              }
              const TileGeo &T = P.T;
              CHECK(T.ni == ni && T.nj == nj && covers(ni, T.cx, T.tx) && covers(nj, T.cy, T.ty));
              CHECK(T.halo == P.shrink * P.steps / 2);
              CHECK(T.rx == T.cx + 2 * T.halo && T.rn == T.rx * (T.cy + 2 * T.halo) && T.rn <= kTileRegion);
              CHECK(8 * T.tiles8 >= T.tx * T.ty);
              CHECK(P.lds == (size_t)T.rn * 9 * 8 * ns);
              CHECK(P.threads % 64 == 0 && P.threads <= kTileThreads);
              // a node of the outermost ring may be left over: it is loaded and never computed
              CHECK(P.keep ? P.threads >= T.rn : 2 * P.threads >= T.rn - 1);
            }
  if (plans < 10000) {
    printf("only %ld plans\n", plans);
    return 1;
  }
  printf("ok\n");
  return 0;
}
