// How an FP64 D2Q9 lattice is cut for several steps per launch (k_tile2d,
// k_sweep2d in lbm_tile2d.hpp): host arithmetic only, no GPU and no memory.
#pragma once

#include <stddef.h>

#include <algorithm>

namespace lbm {

constexpr int kTileSteps = 16;   // most steps of one launch
constexpr int kTileRegion = 2048;  // most region nodes (below 4096: 12-bit region index)
constexpr int kTileThreads = 1024;  // most threads of k_tile2d, which take at most two nodes each

struct TileGeo {
  int ni, nj;
  int cx, cy;      // core size
  int tx, ty;      // tiles
  int halo;        // H
  int rx, rn;      // region row length cx + 2 H and node count
  int tiles8;      // launched tiles / 8 (XCD mapping)
};

constexpr int kSweepSteps = 4, kSweepHalo = 4, kSweepRows = 9;
constexpr int kSweepEntries = 16;  // rows whose table entries are in LDS (i - 6 .. i + 4)
// one thread per column and stage
constexpr int kSweepCols = 128, kSweepBlock = 4 * kSweepCols;

struct SweepGeo {
  int cw, strips;   // core columns of a strip
  int rw;           // table row length cw + 2 kSweepHalo
  int ch, pieces;   // rows of a piece, pieces of a strip
  int blocks8;      // launched workgroups / 8
};

struct Plan2d {
  bool sweep = false;  // strips instead of tiles
  TileGeo T{};
  SweepGeo S{};
  int steps = 0, shrink = 0, threads = 0;
  bool keep = false;  // one tile per CU, one node per thread
  size_t lds = 0;
};

// Steps per launch and core of k_tile2d.
//
// Up to 29 x 29 (flow) or 25 x 25 nodes per CU (two components, by what LDS
// holds) the core is the smallest square of at least a CU's share of the nodes,
// so that about as many tiles as CUs run, each on its own.  Time is then launch
// (2 us) and per-step latency (1 us), and a launch takes as many steps as the
// halo's work allows: 8 (flow with cores up to 10: 10; two components with cores
// above 12: 6, above 20: 4).  us per step, flow | flow + solute with rows: 128^2
// 1.10 | 1.68, 200 x 170 1.27 | 1.87, 300 x 310 1.77 | 2.55, 413 x 307 2.00 | 3.29
// (fewer steps, measured with an earlier form of the kernel: 128^2 1.74 with 4
// against 1.54 with 8, 300 x 310 2.3 against 1.97 | 2.86 against 2.71 with 6; 413
// x 307 flow in 32 x 16 cores with 4 steps 3.02).
// The share is one of area: where neither side is near a multiple of the core,
// the rounded tile counts exceed the CUs and some run a second tile (420 x 300
// 266 tiles, 3.27 | 4.81 us; 130 x 126 272, 1.51 | 2.83; 480 x 340 266, 3.48 |
// 5.30).  Handed-on rows keep these step counts with halos half as wide again (a
// 128^2 flow then has regions of 38 x 38, two nodes a thread: 1.68 us).
//
// Larger lattices run several tiles per CU and are bound by the loads of the
// halo and the FP64 units together: 4 steps, flow in 32 x 16 cores of which a
// CU holds two (1000^2 9.9, 2100 x 1900 40.1 us; 30 x 30 cores with 8 steps,
// measured when the former took 10.8 and 44.9: 11.3, 43.7), flow + solute in the
// largest square core that LDS holds, 25 x 25 (600 x 500 6.5, 1000^2 18.5 us; when
// 1000^2 took 19.7, 32 x 16 cores 20.4 and 20 x 20 with 6 steps 22.2).
inline void tile_shape(int ni, int nj, int ns, int shrink, int lds_cu, int cus, int &steps, int &cx, int &cy) {
  const double per_cu = (double)ni * nj / cus;
  int s = 8;
  while ((double)s * s < per_cu && s < 64) s++;
  // most one-tile cores: what LDS holds with 8 (flow) and 6 steps
  const int one = ns == 1 ? 29 : 20;
  steps = s <= 10 && ns == 1 ? 10 : (s <= 12 ? 8 : (s <= one ? (ns == 1 ? 8 : 6) : 4));
  auto most = [&](int k) {  // largest square core of k steps
    int c = 0;
    const int halo = shrink * k / 2;
    auto fits = [&](int r) { return r * r <= kTileRegion && (size_t)r * r * 72 * ns <= (size_t)lds_cu; };
    while (fits(c + 1 + 2 * halo)) c++;
    return c;
  };
  if (most(steps) < s) steps = 4;
  cx = cy = std::min(s, most(steps));
  if (s > one && ns == 1) {
    cx = 32;
    cy = 16;
  }
}

// The plan for an ni x nj lattice with ns components on a device of cus
// compute units with lds_cu bytes of LDS; handed: row conditions hand values
// to a neighbour.  False when the lattice cannot be cut so (a device that
// does not report its LDS).
inline bool plan2d(int ni, int nj, int ns, bool handed, int lds_cu, int cus, Plan2d &P) {
  P = Plan2d{};
  if (lds_cu <= 0 || cus <= 0) return false;
  P.shrink = handed ? 3 : 2;
  P.T.ni = ni;
  P.T.nj = nj;
  // Strips (k_sweep2d) for flow + solute lattices of many tiles per CU, us per
  // step, tiles -> strips: 1000^2 18.2 -> 19.6, 1088 x 1224 28 -> 23.7,
  // 2100 x 1900 80 -> 61.0, below that tiles are faster (600 x 500 6.5
  // against 9.2: short strips repeat their pipeline's start too often).  The
  // node count decides alone; narrow lattices, whose strips fill half of their
  // lanes, take strips too (102 x 11500 28.7 us, half-steps 50.5; tiles were not
  // tried there).  Flow alone keeps tiles (1088 x 1224 12.2 against 17.2, 2100 x
  // 1900 40.1 against 41.9).  Rows that hand values to a neighbour need the
  // tiles' barrier.
  if (ns == 2 && !handed && (long)ni * nj >= 4500L * cus) {
    SweepGeo &S = P.S;
    const size_t col = (size_t)kSweepRows * (72 * ns + 8) + 8 * kSweepEntries;
    const int most = (int)std::min<size_t>(kSweepCols, lds_cu / col) - 2 * kSweepHalo;
    if (most < kSweepHalo) return false;
    P.sweep = true;
    S.strips = (ni + most - 1) / most;
    S.cw = (ni + S.strips - 1) / S.strips;
    S.strips = (ni + S.cw - 1) / S.cw;
    S.rw = S.cw + 2 * kSweepHalo;
    S.pieces = std::max(1, cus / S.strips);
    S.ch = (nj + S.pieces - 1) / S.pieces;
    S.pieces = (nj + S.ch - 1) / S.ch;
    S.blocks8 = (S.strips * S.pieces + 7) / 8;
    P.lds = col * S.rw;
    P.steps = kSweepSteps;
    P.threads = kSweepBlock;
    return true;
  }
  int cx, cy;
  tile_shape(ni, nj, ns, P.shrink, lds_cu, cus, P.steps, cx, cy);
  if (cx < 1 || cy < 1) return false;
  TileGeo &T = P.T;
  T.halo = P.shrink * P.steps / 2;
  T.tx = (ni + cx - 1) / cx;
  T.ty = (nj + cy - 1) / cy;
  T.cx = (ni + T.tx - 1) / T.tx;
  T.cy = (nj + T.ty - 1) / T.ty;
  T.tx = (ni + T.cx - 1) / T.cx;
  T.ty = (nj + T.cy - 1) / T.cy;
  T.rx = T.cx + 2 * T.halo;
  T.rn = T.rx * (T.cy + 2 * T.halo);
  T.tiles8 = (T.tx * T.ty + 7) / 8;
  P.lds = (size_t)T.rn * 72 * ns;
  P.threads = std::min(kTileThreads, (T.rn + 63) / 64 * 64);
  P.keep = T.rn <= kTileThreads && T.tx * T.ty <= cus;
  // two workgroups of a CU fit its registers with 512 threads each
  if (!P.keep && 2 * P.lds <= (size_t)lds_cu) P.threads = std::max(512, (T.rn / 2 + 63) / 64 * 64);
  return T.rn <= kTileRegion && P.lds <= (size_t)lds_cu;
}

// The fewest steps a launch has to take to beat as many half-steps launched
// one by one.  With row conditions, two: a step by itself costs two to four
// launches more (run(2) of 102 x 11500 flow + solute 57.6 us a step one by one,
// 56.8 in a launch; 420 x 300 31 and 12).  Without them a launch of two steps
// pays only where it loads little more than the half-steps do; us a step in
// runs of two, one by one and in a launch:
//   flow in one round of tiles (128^2 8.9 8.2, 413 x 307 10.0 10.0), and in
//   many tiles while both arrays stay in the 256 MB memory-side cache (512^2
//   12.6 10.6, 1000^2 25.9 20.6, 1300^2 36.8 29.9; beyond it 2100 x 1900 74.6
//   78.0, with partial bounce-back 78 and 88);
//   a resting solute, whose half-steps touch its lines all the same (1000^2
//   47.8 34.3, 2100 x 1900 170 104);
//   not flow + solute (200 x 170 9.4 9.7, with partial bounce-back 9.6 10.8; in
//   strips of 51 columns, 102 x 11500, 45.1 57.1);
//   nor where some CUs run a second tile (420 x 300 flow 10.0 12.1, 480 x 340
//   10.7 13.1), where cores beyond 20 x 20 do not pay in four steps either
//   (480 x 340 8.0 7.9, with partial bounce-back 8.1 8.4; in six 7.3 6.5).
inline int least_steps(const Plan2d &P, int ns, bool rows, bool resting, size_t state_bytes, int cus) {
  if (rows) return 2;
  const long tiles = P.sweep ? 0 : (long)P.T.tx * P.T.ty;
  if (tiles > cus && tiles < 2L * cus) return std::min(P.steps, P.T.cx * P.T.cy > 400 ? 6 : 4);
  if (resting || (ns == 1 && (tiles <= cus || 2 * state_bytes <= 200000000))) return 2;
  return std::min(P.steps, 4);
}

}  // namespace lbm
