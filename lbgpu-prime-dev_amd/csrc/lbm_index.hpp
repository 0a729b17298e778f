// Index arithmetic shared by the host set-up, the device kernels and the
// CPU index test (tests/index_check.cpp compiles this header with g++).
//
// Populations live in tiles of kTile consecutive fluid nodes:
//   one distribution:  element (slot a, node x) at
//     (x / kTile) * Q*kTile + a * kTile + x % kTile
//   flow + solute:     element (subs s, slot a, node x) at
//     (x / kTile) * 2*Q*kTile + (a * kTile + x % kTile) * 2 + s
// so that one slot of a wave's 64 nodes is one contiguous 512-byte run
// (FP64), consecutive waves continue the same runs, and the flow and solute
// populations of a slot sit side by side (one 2-wide load or store moves
// both).  kTile = 2048 (a tile spans eight workgroups): against 64-node
// tiles (one wave each) it raised the even half-step from 73% to 79% of
// HBM peak at 256^3 and the odd one by 1-2%; 512, 1024 and 4096 measured
// between the two or, for flow + solute, below.
//
// Neighbours are not stored per node.  Each lattice row (fixed j, k) is
// split in 64-node words; for word w of row r, RowWord holds the fluid
// bitmask (bit b set when node 64w+b is fluid) and the compact index of
// the first fluid node at or after 64w.  The compact index of a fluid node
// is then base + popcount(bits below it), read from a few MB that stay in
// cache, instead of 72 bytes of neighbour table per node from HBM.
#pragma once

#include <stdint.h>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define LBM_HD __host__ __device__ __forceinline__
#else
#define LBM_HD inline
#endif

namespace lbm {

constexpr int kTile = 2048;

// Unsigned 32-bit division by an invariant d >= 1 (Granlund & Montgomery,
// PLDI 1994, Fig. 4.1): q = (t + ((n - t) >> s1)) >> s2, t = mulhi(m, n).
struct FastDiv {
  uint32_t d, m, s1, s2;
};

LBM_HD FastDiv make_fastdiv(uint32_t d) {
  uint32_t l = 0;
  while (l < 32 && (1ull << l) < d) l++;
  FastDiv f;
  f.d = d;
  f.m = (uint32_t)((((1ull << l) - d) << 32) / d + 1);
  f.s1 = l < 1 ? l : 1;
  f.s2 = l > 0 ? l - 1 : 0;
  return f;
}

LBM_HD uint32_t mulhi32(uint32_t a, uint32_t b) { return (uint32_t)(((uint64_t)a * b) >> 32); }

LBM_HD uint32_t fdiv(uint32_t n, const FastDiv &f) {
  uint32_t t = mulhi32(f.m, n);
  return (t + ((n - t) >> f.s1)) >> f.s2;
}

LBM_HD int popc64(uint64_t v) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __popcll(v);
#else
  return __builtin_popcountll(v);
#endif
}

struct alignas(16) RowWord {
  uint64_t bits;  // fluid bitmask of nodes 64w .. 64w+63 of the row
  int32_t base;   // compact index of the first fluid node at or after 64w
  int16_t dprev;  // rank of the row's node before 64w (periodic) - base, or kSolidRank
  int16_t dnext;  // rank of the row's node after the word (periodic) - base, or kSolidRank
};
constexpr int16_t kSolidRank = -32768;

struct Geo {
  const RowWord *rw;  // [rows][W]
  const int *node;    // compact index -> dense index
  int ni, nj, nk;     // nk = 1 in 2-D
  int W;              // words per row
  int halo;           // last axis through ghost entries
  int ghost;          // first ghost compact index (= number of fluid nodes)
  int E;              // nodes per plane across the last axis
  FastDiv div_ni, div_nj;
};

template <int Q, int NS>
LBM_HD uint32_t foff(int s, int a, uint32_t x) {
  if (NS == 2) return (x / kTile) * (uint32_t)(2 * Q * kTile) + (uint32_t)(a * kTile + (x % kTile)) * 2u + (uint32_t)s;
  return (x / kTile) * (uint32_t)(Q * kTile) + (uint32_t)(a * kTile) + (x % kTile);
}

// The same location in units of U per node (U = NS elements, or the NS
// populations' bytes) with one multiplication.
template <int Q, uint32_t U>
LBM_HD uint32_t loc_at(int a, uint32_t x) {
  return x * U + (x / kTile) * ((uint32_t)(Q - 1) * kTile * U) + (uint32_t)a * (kTile * U);
}

// fluid test and compact index of node (i, row r): one 16-byte load and
// no branch, so the loads of all neighbours can be in flight together
LBM_HD int rank_of(const Geo &G, int i, int r) {
#if defined(__HIP_DEVICE_COMPILE__)
  const uint4 v = *reinterpret_cast<const uint4 *>(G.rw + ((long)r * G.W + (i >> 6)));
  const uint64_t bits = (uint64_t)v.x | ((uint64_t)v.y << 32);
  const int base = (int)v.z;
#else
  const RowWord &w = G.rw[(long)r * G.W + (i >> 6)];
  const uint64_t bits = w.bits;
  const int base = w.base;
#endif
  const int b = i & 63;
  const int idx = base + popc64(bits & ((1ull << b) - 1ull));
  return ((bits >> b) & 1ull) ? idx : -1;
}

// coordinates of a dense node index: i fastest, then j, then k
template <int D>
LBM_HD void coords(const Geo &G, uint32_t n, int &i, int &j, int &k) {
  uint32_t r = fdiv(n, G.div_ni);
  i = (int)(n - r * (uint32_t)G.ni);
  if (D == 2) {
    j = (int)r;
    k = 0;
  } else {
    uint32_t q = fdiv(r, G.div_nj);
    j = (int)(r - q * (uint32_t)G.nj);
    k = (int)q;
  }
}

// compact index of (i+dx, j+dy, k+dz): periodic in every axis, or across
// the last axis through ghost entries in halo mode; -1 when solid.
// Ghost entries [ghost, ghost+E) stand for the plane before the first one,
// [ghost+E, ghost+2E) for the plane after the last one; their solidity is
// that of the periodic image.  Written with selects only, so the compiler
// can issue the row-word loads of all directions back to back.
LBM_HD int wrap1(int v, int n) { return v < 0 ? v + n : (v >= n ? v - n : v); }

template <int D>
LBM_HD int neighbor(const Geo &G, int i, int j, int k, int dx, int dy, int dz) {
  const int ii = wrap1(i + dx, G.ni);
  int last, lastw, row, p;
  if (D == 2) {
    last = j + dy;
    lastw = wrap1(last, G.nj);
    row = lastw;
    p = ii;
  } else {
    const int jj = wrap1(j + dy, G.nj);
    last = k + dz;
    lastw = wrap1(last, G.nk);
    row = jj + G.nj * lastw;
    p = ii + G.ni * jj;
  }
  const int r = rank_of(G, ii, row);
  const int gh = G.ghost + (last < 0 ? 0 : G.E) + p;
  return (G.halo && last != lastw && r >= 0) ? gh : r;
}

// The same for several directions at once, in two phases: every row-word
// load is issued before any rank is formed, so their latencies overlap.
template <int D, int K>
LBM_HD void neighbors_of(const Geo &G, int i, int j, int k, const int (&dx)[K], const int (&dy)[K],
                         const int (&dz)[K], int (&out)[K]) {
  int col[K], gh[K];
  bool cross[K];
  const RowWord *ptr[K];
#pragma unroll
  for (int q = 0; q < K; q++) {
    const int ii = wrap1(i + dx[q], G.ni);
    int last, lastw, row, p;
    if (D == 2) {
      last = j + dy[q];
      lastw = wrap1(last, G.nj);
      row = lastw;
      p = ii;
    } else {
      const int jj = wrap1(j + dy[q], G.nj);
      last = k + dz[q];
      lastw = wrap1(last, G.nk);
      row = jj + G.nj * lastw;
      p = ii + G.ni * jj;
    }
    col[q] = ii & 63;
    ptr[q] = G.rw + ((long)row * G.W + (ii >> 6));
    cross[q] = G.halo && last != lastw;
    gh[q] = G.ghost + (last < 0 ? 0 : G.E) + p;
  }
  uint64_t bits[K];
  int base[K];
#pragma unroll
  for (int q = 0; q < K; q++) {
#if defined(__HIP_DEVICE_COMPILE__)
    const uint4 v = *reinterpret_cast<const uint4 *>(ptr[q]);
    bits[q] = (uint64_t)v.x | ((uint64_t)v.y << 32);
    base[q] = (int)v.z;
#else
    bits[q] = ptr[q]->bits;
    base[q] = ptr[q]->base;
#endif
  }
#pragma unroll
  for (int q = 0; q < K; q++) {
    const int b = col[q];
    const int r = ((bits[q] >> b) & 1ull) ? base[q] + popc64(bits[q] & ((1ull << b) - 1ull)) : -1;
    out[q] = (cross[q] && r >= 0) ? gh[q] : r;
  }
}

// All neighbours of one node, one row-word load per lattice row: the
// nodes i-1, i, i+1 of a row come from the word holding i, its bitmask and
// the ranks of the row's nodes just outside the word (dprev / dnext, which
// also carry the periodic wrap at the row ends).  Every load is issued
// before any rank is formed.  For a = 1..Q-1: rank[a-1] = compact index of
// x - c_a where fluid[a-1], else of no meaning.
//
// The half-steps of the narrow storage types are bound by the number of
// vector instructions they issue (FP16 odd step, 192^3: 1312 of them, at 4
// cycles a wave 106 of its 112 us), so a row costs one popcount (the ranks of
// i - 1 and i + 1 follow from it by the bits of i - 1 and i) and one rotation
// that brings those three bits down, everything else is selects, and the halo
// form runs only in halo mode.
template <int D>
LBM_HD void neighbors_core(const Geo &G, int i, int j, int k, int (&rank)[D == 2 ? 8 : 18],
                           bool (&fluid)[D == 2 ? 8 : 18]) {
  // lattice rows (dy, dz) of the nodes x - c_a, in the reference order
  constexpr int R = D == 2 ? 3 : 9, M = D == 2 ? 8 : 18;
  constexpr int rdy[9] = {0, -1, 1, 0, 0, -1, 1, 1, -1};
  constexpr int rdz[9] = {0, 0, 0, -1, 1, -1, 1, -1, 1};
  // row and column offset of x - c_a
  constexpr int row2[8] = {0, 0, 1, 2, 1, 2, 1, 2}, col2[8] = {-1, 1, 0, 0, -1, 1, 1, -1};
  constexpr int row3[18] = {0, 0, 1, 2, 1, 2, 1, 2, 3, 4, 3, 4, 3, 4, 5, 6, 7, 8};
  constexpr int col3[18] = {-1, 1, 0, 0, -1, 1, 1, -1, 0, 0, -1, 1, 1, -1, 0, 0, 0, 0};
  const int b = i & 63, w = i >> 6;
  const bool left = b == 0, right = b == 63 || i == G.ni - 1;  // no such node in the word
  const uint32_t s = (uint32_t)(b + 63) & 63u;                 // rotation: bits i-1, i, i+1 become 0, 1, 2
  const uint64_t below = (1ull << b) - 1ull;
  const RowWord *ptr[R];
#pragma unroll
  for (int q = 0; q < R; q++) {
    const int last = D == 2 ? j + rdy[q] : k + rdz[q];
    const int lastw = wrap1(last, D == 2 ? G.nj : G.nk);
    const int row = D == 2 ? lastw : wrap1(j + rdy[q], G.nj) + G.nj * lastw;
    ptr[q] = G.rw + ((long)row * G.W + w);
  }
  int at[R], base[R];     // rank of the first fluid node at or after i, of the word's first
  uint32_t near[R];       // bits 0..2: nodes i-1, i, i+1 (within the word)
  int dp[R], dn[R];
#pragma unroll
  for (int q = 0; q < R; q++) {
#if defined(__HIP_DEVICE_COMPILE__)
    const uint4 v = *reinterpret_cast<const uint4 *>(ptr[q]);
    const uint32_t x0 = s & 32u ? v.y : v.x, x1 = s & 32u ? v.x : v.y;
    near[q] = __builtin_amdgcn_alignbit(x1, x0, s);
    base[q] = (int)v.z;
    at[q] = base[q] + __popc(v.x & (uint32_t)below) + __popc(v.y & (uint32_t)(below >> 32));
    dp[q] = (int)(int16_t)(v.w & 0xffffu);
    dn[q] = (int)v.w >> 16;
#else
    const RowWord &v = *ptr[q];
    near[q] = (uint32_t)(s ? (v.bits >> s) | (v.bits << (64 - s)) : v.bits);
    base[q] = v.base;
    at[q] = v.base + popc64(v.bits & below);
    dp[q] = v.dprev;
    dn[q] = v.dnext;
#endif
  }
#pragma unroll
  for (int a = 0; a < M; a++) {
    const int q = D == 2 ? row2[a & 7] : row3[a], dx = D == 2 ? col2[a & 7] : col3[a];
    if (dx == 0) {
      fluid[a] = near[q] & 2u;
      rank[a] = at[q];
    } else if (dx < 0) {
      const int in = at[q] - 1, out = base[q] + dp[q];
      const bool fin = near[q] & 1u, fout = dp[q] != kSolidRank;
      fluid[a] = left ? fout : fin;
      rank[a] = left ? out : in;
    } else {
      const int in = at[q] + (int)((near[q] >> 1) & 1u), out = base[q] + dn[q];
      const bool fin = near[q] & 4u, fout = dn[q] != kSolidRank;
      fluid[a] = right ? fout : fin;
      rank[a] = right ? out : in;
    }
  }
  if (G.halo) {
    // across the last axis: ghost entries, as solid as the periodic image
#pragma unroll
    for (int a = 0; a < M; a++) {
      const int q = D == 2 ? row2[a & 7] : row3[a], dx = D == 2 ? col2[a & 7] : col3[a];
      const int last = D == 2 ? j + rdy[q] : k + rdz[q];
      const int col = wrap1(i + dx, G.ni) + (D == 2 ? 0 : G.ni * wrap1(j + rdy[q], G.nj));
      const int gh = G.ghost + (last < 0 ? 0 : G.E) + col;
      rank[a] = last != wrap1(last, D == 2 ? G.nj : G.nk) ? gh : rank[a];
    }
  }
}

// out[a-1] = compact index of x - c_a, -1 when solid
template <int D>
LBM_HD void neighbors_rows(const Geo &G, int i, int j, int k, int (&out)[D == 2 ? 8 : 18]) {
  bool fluid[D == 2 ? 8 : 18];
  neighbors_core<D>(G, i, j, k, out, fluid);
#pragma unroll
  for (int a = 0; a < (D == 2 ? 8 : 18); a++) out[a] = fluid[a] ? out[a] : -1;
}

// Host: fill the row words from the dense -> compact map (fid[n] = -1 for
// solid).  base is the number of fluid nodes before the word in dense
// order, so base(word) + popcount(word) = base(next word) everywhere.
inline void fill_row_words(const int *fid, long rows, int ni, RowWord *rw) {
  const int W = (ni + 63) / 64;
  long count = 0;
  for (long r = 0; r < rows; r++)
    for (int w = 0; w < W; w++) {
      RowWord &x = rw[r * W + w];
      x.base = (int32_t)count;
      const int n = ni - 64 * w < 64 ? ni - 64 * w : 64;
      const int *f = fid + r * ni + 64 * w;
      uint64_t bits = 0;
      for (int b = 0; b < n; b++) bits |= (uint64_t)(f[b] >= 0) << b;
      x.bits = bits;
      count += popc64(bits);
      const int pc = w > 0 ? 64 * w - 1 : ni - 1;
      const int nc = 64 * (w + 1) < ni ? 64 * (w + 1) : 0;
      const int pid = fid[r * ni + pc], nid = fid[r * ni + nc];
      x.dprev = pid < 0 ? kSolidRank : (int16_t)(pid - x.base);
      x.dnext = nid < 0 ? kSolidRank : (int16_t)(nid - x.base);
    }
}

}  // namespace lbm
