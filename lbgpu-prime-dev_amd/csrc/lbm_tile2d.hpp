// Several D2Q9 time steps per launch (FP64 storage and collision).
//
// A single 2-D step is short of work for this GPU: the lattices that users
// run (10^3 to 10^6 nodes) live in cache, and each step costs two to five
// launches (the half-step and the boundary rows) and one read and one write
// of every population.  k_tile2d advances a tile of the lattice by an even
// number of steps inside one workgroup instead: it loads the tile's core and
// a halo of nodes around it into LDS, runs the in-place AA half-steps there
// (odd, even, odd, ...), boundary rows included, and stores the core into a
// second population array.  The halo shrinks with every odd half-step, so
// neighbouring tiles repeat each other's halo work and need no exchange.
//
// Validity of LDS locations (slot b of region node y), by the distance of y
// from the region's edge: all are valid at the start (s = 0).  An odd
// half-step at x reads and writes the locations (b, x - c_b): it can run
// where dist(x) >= s + 1, and a location is valid afterwards where its
// writer ran: dist >= s + 2.  An even half-step is node-local: it runs where
// dist >= s.  A row condition whose source node is solid hands its value to
// a neighbour's input (the reference's own-slot rule), which costs one more
// node per odd half-step.  The halo is thus 2 (or 3) nodes per pair of steps.
//
// The arithmetic is collide() of the half-step kernel on the same values, so
// results equal the step-by-step launches bit for bit.
//
// Measured per step in runs of 240 to 1200, against half-steps and row launches
// one by one: 128^2 flow 3.3 -> 1.1 us; flow + solute with rows: 413 x 307 18.5
// -> 3.3, 600 x 500 with partial bounce-back 24 -> 7.3, 1088 x 1224 58 -> 23.7
// (strips, below; tiles 28).  Small lattices are bound by the latency of a step
// inside the workgroup (about 1 us: LDS gathers, the collision's serial sums,
// the barrier), large ones by the loads of core and halo (1.7 times the core at
// 25 x 25 with 4 steps) followed by the FP64 units, which one workgroup per CU
// does not overlap.
#pragma once

#include "lbm_device.hpp"
#include "lbm_plan2d.hpp"

namespace lbm {

// list entry of a fluid region node: region index, bit 12 + a - 1 set when
// x - c_a is fluid, the boundary rows, and from bit 22 its distance from the
// region's edge (at most the halo)
constexpr uint32_t kTileNorth = 1u << 20, kTileSouth = 1u << 21;
constexpr int kTileDist = 22;

// core origin, core size and region size of tile t
LBM_HD void tile_span(const TileGeo &T, int t, int &x0, int &y0, int &cw, int &ch) {
  const int ty = t / T.tx, tx = t - ty * T.tx;
  x0 = tx * T.cx;
  y0 = ty * T.cy;
  cw = T.ni - x0 < T.cx ? T.ni - x0 : T.cx;
  ch = T.nj - y0 < T.cy ? T.nj - y0 : T.cy;
}

// Per tile: gidx[rn] (compact index of each region node, -1: solid or
// outside), the list of its fluid nodes ordered by distance from the region's
// edge (core first, then ring by ring inwards to outwards, each row-major,
// so that whole waves fall idle as the halo shrinks), and their number.
__global__ __launch_bounds__(256) void k_tile_build(Geo G, TileGeo T, int *gidx, uint32_t *list, int *cnt) {
  __shared__ int wsum[4];
  const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  int x0, y0, cw, ch;
  tile_span(T, t, x0, y0, cw, ch);
  const int rw = cw + 2 * T.halo, rh = ch + 2 * T.halo;
  int *g = gidx + (long)t * T.rn;
  uint32_t *l = list + (long)t * T.rn;
  auto wrap = [](int v, int n) {
    v %= n;
    return v < 0 ? v + n : v;
  };
  for (int n = tid; n < T.rn; n += 256) {
    const int ry = n / T.rx, rx = n - ry * T.rx;
    g[n] = rx < rw && ry < rh ? rank_of(G, wrap(x0 - T.halo + rx, T.ni), wrap(y0 - T.halo + ry, T.nj)) : -1;
  }
  int run = 0;
  for (int d = T.halo; d >= 0; d--) {
    for (int base = 0; base < T.rn; base += 256) {
      const int n = base + tid;
      bool in = false;
      int rx = 0, ry = 0;
      if (n < T.rn) {
        ry = n / T.rx;
        rx = n - ry * T.rx;
        int dist = rx < rw - 1 - rx ? rx : rw - 1 - rx;
        dist = ry < dist ? ry : dist;
        dist = rh - 1 - ry < dist ? rh - 1 - ry : dist;
        dist = T.halo < dist ? T.halo : dist;
        in = g[n] >= 0 && dist == d;
      }
      const uint64_t bal = __ballot(in);
      if (lane == 0) wsum[wv] = __popcll(bal);
      __syncthreads();
      int at = run + __popcll(bal & ((1ull << lane) - 1ull));
      for (int q = 0; q < wv; q++) at += wsum[q];
      if (in) {
        const int i = wrap(x0 - T.halo + rx, T.ni), j = wrap(y0 - T.halo + ry, T.nj);
        uint32_t e = (uint32_t)n | (uint32_t)d << kTileDist;
#pragma unroll
        for (int a = 1; a < 9; a++)
          if (rank_of(G, wrap1(i - CX(a), T.ni), wrap1(j - CY(a), T.nj)) >= 0) e |= 1u << (11 + a);
        if (j == T.nj - 1) e |= kTileNorth;
        if (j == 0) e |= kTileSouth;
        l[at] = e;
      }
      run += wsum[0] + wsum[1] + wsum[2] + wsum[3];
      __syncthreads();
    }
  }
  if (tid == 0) cnt[t] = run;
}

struct TileArgs {
  StepArgs<double, double> A;  // A.F: populations read, A.Fo: where they are written
  TileGeo T;
  const int *gidx;
  const uint32_t *list;
  const int *cnt;
  int steps;             // even, the first one odd
  int shrink;            // halo nodes an odd half-step uses up: 2, or 3 with handed-on row values
  int flow[2];           // row condition of the flow, [0] north, [1] south: 0 none, 1 density, 2 y momentum
  int grad[2];           // solute zero gradient
  double val[2][kTileSteps];  // prescribed value per step
};

// the pair of one location in LDS
template <int NS>
using tile_t = double __attribute__((ext_vector_type(NS)));

// Row conditions of one region node on the populations it has gathered; f
// and gs hold what the node collides.  put(s, a, v, own_opp) takes the value
// of unknown a of component s.
template <int NS, typename Put>
__device__ __forceinline__ void tile_rows(const TileArgs &B, uint32_t e, int step, const double (&f)[9],
                                          const double (&gs)[9], Put &&put) {
  auto side = [&](bool north, int q, int u0, int u1, int u2) {
    double v[3];
    if (B.flow[q]) {
      bc2d_flow_values<double>(f, north, B.val[q][step], B.A.rhoA, B.flow[q] == 2, v);
      put(0, u0, v[0], B.flow[q] == 2);
      put(0, u1, v[1], B.flow[q] == 2);
      put(0, u2, v[2], B.flow[q] == 2);
    }
    if (NS == 2 && B.grad[q]) {
      bc2d_zerograd_values<double>(gs, north, v);
      put(1, u0, v[0], false);
      put(1, u1, v[1], false);
      put(1, u2, v[2], false);
    }
  };
  if (e & kTileNorth) side(true, 0, 4, 8, 6);
  if (e & kTileSouth) side(false, 1, 3, 5, 7);
}

// Where a node's populations lie in LDS: slot a of the node is element
// a * plane + n0; the same column in the rows below and above is dm and dp
// elements away (all but n0 the same for the whole wave).
struct TileAt {
  int plane, n0, dm, dp;
};

// the nine locations a node collides from: slot a of x - c_a (own slot
// opp(a) when that node is solid) before an odd half-step, own slot opp(a)
// before an even one; an odd half-step pushes f_a to location opp(a).  The
// two choices differ by a wave-uniform distance, added under the node's bit
// (three integer operations a direction).
template <bool ODD>
__device__ __forceinline__ void tile_locs(const TileAt &P, uint32_t e, int (&loc)[9]) {
  loc[0] = P.n0;
#pragma unroll
  for (int a = 1; a < 9; a++) {
    loc[a] = OPP(a) * P.plane + P.n0;
    if (ODD) {
      const int row = CY(a) == 0 ? 0 : (CY(a) > 0 ? P.dm : P.dp);
      loc[a] += ((int)(e << (20 - a)) >> 31) & ((a - OPP(a)) * P.plane + row - CX(a));
    }
  }
}

// one half-step of one node, which collides from loc; LAST: the result goes to
// the output array (the node's compact index is idx), else back to LDS; ns:
// partial bounce-back
template <int NS, bool SOL, bool WALSH, bool ODD, bool LAST>
__device__ __forceinline__ void tile_node(const TileArgs &B, const StepArgs<double, double> &A, tile_t<NS> *lds,
                                          const int (&loc)[9], int idx, double ns, uint32_t e, bool rows, int step) {
  double f[9], gs[9], u[3];
#pragma unroll
  for (int a = 0; a < 9; a++) {
    const tile_t<NS> v = lds[loc[a]];
    f[a] = v[0];
    if constexpr (NS == 2) gs[a] = v[NS - 1];
  }
  if (rows && (e & (kTileNorth | kTileSouth)))
    tile_rows<NS>(B, e, step, f, gs, [&](int s, int a, double v, bool) {
      if (s == 0) f[a] = v;
      else gs[a] = v;
      // a resting solute is not collided: its row values are stored
      if constexpr (NS == 2 && !SOL && !LAST)
        if (s == 1) lds[loc[a]][NS - 1] = v;
    });
  if constexpr (WALSH) {
    const double kns = 1. - ns;
    double fp[9], gp[9];
#pragma unroll
    for (int a = 0; a < 9; a++) {
      fp[a] = f[a];
      if (SOL) gp[a] = gs[a];
    }
    collide<9, double, double, 0, ODD, true>(A, idx, f, u, kns);
    if constexpr (SOL) collide<9, double, double, 1, ODD, true>(A, idx, gs, u, kns);
    walsh_mix<9, double>(f, fp, ns, kns);
    if constexpr (SOL) walsh_mix<9, double>(gs, gp, ns, kns);
  } else {
    collide<9, double, double, 0, ODD>(A, idx, f, u);
    if constexpr (SOL) collide<9, double, double, 1, ODD>(A, idx, gs, u);
  }
#pragma unroll
  for (int a = 0; a < 9; a++) {
    // even: own slot a (a resting solute keeps its slot a, gathered as direction opp(a))
    const int at = loc[OPP(a)];
    tile_t<NS> v;
    v[0] = f[a];
    if constexpr (NS == 2) v[NS - 1] = SOL ? gs[a] : gs[OPP(a)];
    if constexpr (LAST)
      *(tile_t<NS> *)(A.Fo + (size_t)foff<9, NS>(0, a, (uint32_t)idx)) = v;
    else if constexpr (NS == 2 && !SOL)
      lds[at][0] = v[0];
    else
      lds[at] = v;
  }
}

// A thread takes list entry tid and keeps what it needs in every step, its
// locations among it, in registers (KEEP: lattices of one tile per CU, whose
// steps are bound by their latency; with the list in LDS, counts in global
// memory and locations formed in every step, 128^2 took 1.55 us a step instead
// of 1.33).  Larger lattices want the registers for a second workgroup on the
// CU: they take entry tid + blockDim.x too and form locations as they go.
template <int NS, bool SOL, bool WALSH, bool KEEP>
__global__ __launch_bounds__(kTileThreads) void k_tile2d(TileArgs B) {
  constexpr int PER = KEEP ? 1 : 2;
  extern __shared__ __align__(16) char tile_lds[];
  const int t = xcd_block(B.T.tiles8);
  if (t >= B.T.tx * B.T.ty) return;
  const int tid = threadIdx.x, nt = blockDim.x, rn = B.T.rn;
  tile_t<NS> *lds = (tile_t<NS> *)tile_lds;
  const int *g = B.gidx + (long)t * rn;
  const uint32_t *list = B.list + (long)t * rn;
  const int fluid = B.cnt[t];
  for (int n = tid; n < rn; n += nt) {
    const int idx = g[n];
    if (idx < 0) continue;
    tile_t<NS> v[9];
#pragma unroll
    for (int a = 0; a < 9; a++) v[a] = *(const tile_t<NS> *)(B.A.F + (size_t)foff<9, NS>(0, a, (uint32_t)idx));
#pragma unroll
    for (int a = 0; a < 9; a++) lds[a * rn + n] = v[a];
  }
  uint32_t e[PER];
  int dist[PER], idx[PER], keep_odd[9], keep_even[9];
  double ns[PER];
  const TileAt at0{rn, 0, -B.T.rx, B.T.rx};
#pragma unroll
  for (int q = 0; q < PER; q++) {
    const int p = tid + q * nt;
    e[q] = p < fluid ? list[p] : 0u;
    dist[q] = p < fluid ? (int)(e[q] >> kTileDist) : -1;
    const int n = (int)(e[q] & 4095u);
    idx[q] = p < fluid && (KEEP || WALSH) ? g[n] : 0;
    ns[q] = WALSH ? B.A.ns[idx[q]] : 0.;
  }
  auto at = [&](int q) {
    TileAt P = at0;
    P.n0 = (int)(e[q] & 4095u);
    return P;
  };
  if constexpr (KEEP) {
    tile_locs<true>(at(0), e[0], keep_odd);
    tile_locs<false>(at(0), e[0], keep_even);
  }
  auto locs = [&](auto odd, int q, int (&loc)[9]) __attribute__((always_inline)) {
    if constexpr (!KEEP) {
      asm("" : "+v"(e[q]));  // formed here, not ahead of the loop
      tile_locs<decltype(odd)::value>(at(q), e[q], loc);
    } else {
#pragma unroll
      for (int a = 0; a < 9; a++) loc[a] = decltype(odd)::value ? keep_odd[a] : keep_even[a];
    }
  };
  using Odd = std::true_type;
  using Even = std::false_type;
  __syncthreads();
  const bool rows = B.flow[0] || B.flow[1] || (NS == 2 && (B.grad[0] || B.grad[1]));
  const bool handed = B.shrink > 2;
  StepArgs<double, double> A = B.A;
  A.write_mv = 0;
  int s = 0;
  for (int k = 0; k < B.steps; k += 2) {
    if (handed) {
      // row values that go to a neighbour's input: stored before any node collides
#pragma unroll
      for (int q = 0; q < PER; q++) {
        if (dist[q] < s + 1 || !(e[q] & (kTileNorth | kTileSouth))) continue;
        int loc[9];
        locs(Odd(), q, loc);
        double f[9], gs[9];
#pragma unroll
        for (int a = 0; a < 9; a++) {
          f[a] = lds[loc[a]][0];
          if constexpr (NS == 2) gs[a] = lds[loc[a]][NS - 1];
        }
        // the rule of bc_store: own slot a (or opp(a)) when the source is solid
        tile_rows<NS>(B, e[q], k, f, gs, [&](int c, int a, double v, bool own_opp) {
          const int own = (own_opp ? OPP(a) : a) * rn + (int)(e[q] & 4095u);
          lds[(e[q] >> (11 + a)) & 1u ? loc[a] : own][c ? NS - 1 : 0] = v;
        });
      }
      __syncthreads();
    }
#pragma unroll
    for (int q = 0; q < PER; q++)
      if (dist[q] >= s + B.shrink - 1) {
        int loc[9];
        locs(Odd(), q, loc);
        tile_node<NS, SOL, WALSH, true, false>(B, A, lds, loc, 0, ns[q], e[q], rows && !handed, k);
      }
    s += B.shrink;
    __syncthreads();
    if (k + 2 < B.steps) {
#pragma unroll
      for (int q = 0; q < PER; q++)
        if (dist[q] >= s) {
          int loc[9];
          locs(Even(), q, loc);
          tile_node<NS, SOL, WALSH, false, false>(B, A, lds, loc, 0, ns[q], e[q], rows, k + 1);
        }
      __syncthreads();
    } else {
      A.write_mv = B.A.write_mv;
#pragma unroll
      for (int q = 0; q < PER; q++)
        if (dist[q] >= B.T.halo) {
          int loc[9];
          locs(Even(), q, loc);
          tile_node<NS, SOL, WALSH, false, true>(B, A, lds, loc, KEEP ? idx[q] : g[e[q] & 4095u], ns[q], e[q], rows,
                                                 k + 1);
        }
    }
  }
}

// ---- large lattices: strips swept along y ----------------------------------
//
// A lattice of several tiles per CU spends most of a tile's time on loading
// it, and 25 x 25 cores load 1.7 times their populations.  k_sweep2d gives a
// workgroup a strip of columns and sweeps it along y: the rows enter LDS one
// by one, and four stages follow each other two rows apart, so that one
// iteration advances
//   odd half-step 1 on row i, even 2 on row i - 2, odd 3 on row i - 4, even 4
//   on row i - 6 (stored to the output array),
// with one barrier.  An odd stage on row r touches rows r - 1 .. r + 1 and
// needs them to have passed the stage before, which they have; the rows the
// stages touch are disjoint.  Nine rows are live (i - 6 .. i + 1 and the row
// i + 2 being filled).  Populations are loaded two iterations before they are
// written to LDS and their indices two more, and the barrier orders LDS only,
// so the loads stay in flight across it.  The halo is kSweepHalo columns on
// either side and, once per strip piece, rows at either end.
//
// Measured (flow + solute, porosity 0.7, row conditions), us per step, tiles
// -> strips: 1088 x 1224 28 -> 23.7, 2100 x 1900 80 -> 61.0.  An iteration
// takes 1.7 us: 0.9 us without the collision (LDS traffic and latency of two
// waves per SIMD, which is all that 160 KB of rows feed), 0.1 us of it waiting
// for the global loads; solid columns leave 30 % of the lanes idle.

// tab[strip][row][column] = {compact index (-1 solid or past the strip),
// entry bits of the node}
__global__ __launch_bounds__(256) void k_sweep_build(Geo G, SweepGeo S, int2 *tab) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long)S.strips * G.nj * S.rw) return;
  const int x = (int)(t % S.rw), j = (int)(t / S.rw % G.nj), strip = (int)(t / S.rw / G.nj);
  const int x0 = strip * S.cw, cw = G.ni - x0 < S.cw ? G.ni - x0 : S.cw;
  int2 v = {-1, 0};
  if (x < cw + 2 * kSweepHalo) {
    int i = (x0 - kSweepHalo + x) % G.ni;
    if (i < 0) i += G.ni;
    v.x = rank_of(G, i, j);
    uint32_t e = 0;
#pragma unroll
    for (int a = 1; a < 9; a++)
      if (rank_of(G, wrap1(i - CX(a), G.ni), wrap1(j - CY(a), G.nj)) >= 0) e |= 1u << (11 + a);
    if (j == G.nj - 1) e |= kTileNorth;
    if (j == 0) e |= kTileSouth;
    v.y = (int)e;
  }
  tab[t] = v;
}

// barrier that orders LDS accesses only
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <bool SOL, bool WALSH>
__global__ __launch_bounds__(kSweepBlock) void k_sweep2d(TileArgs B, SweepGeo S, const int2 *tab) {
  extern __shared__ __align__(16) char sweep_lds[];
  constexpr int NS = 2, R = kSweepRows, H = kSweepHalo;
  const int t = xcd_block(S.blocks8);
  if (t >= S.strips * S.pieces) return;
  const int strip = t % S.strips, piece = t / S.strips;
  const int ni = B.T.ni, nj = B.T.nj;
  const int cw = ni - strip * S.cw < S.cw ? ni - strip * S.cw : S.cw;
  const int y0 = piece * S.ch, ch = nj - y0 < S.ch ? nj - y0 : S.ch;
  const int rw = cw + 2 * H, stride = S.rw, plane = R * stride;
  tile_t<NS> *lds = (tile_t<NS> *)sweep_lds;
  int2 *ent = (int2 *)(lds + 9 * plane);
  double *nsl = (double *)(ent + kSweepEntries * stride);
  // a thread computes column n of one stage (a SIMD's two waves take an odd
  // and an even stage); the threads of stages 0 to 2 also load column n of
  // slots 3 stage .. 3 stage + 2.  Those of stage 3, which store the results,
  // do not load: waiting for a load would wait for the stores before it.
  const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int stage = (wv & 3) ^ (wv >> 2);
  const int n = ((int)threadIdx.x & 63) + 64 * (wv >> 2);
  const bool rows = B.flow[0] || B.flow[1] || (NS == 2 && (B.grad[0] || B.grad[1]));
  const bool last = stage == B.steps - 1;
  const int first = last ? H : 1 + stage;  // distance from the strip's edge and ends
  const bool on = stage < B.steps && n >= first && n < rw - first;
  StepArgs<double, double> A = B.A;
  A.write_mv = last ? B.A.write_mv : 0;

  // row y0 - H + q has number q and lies in slot q % R; iteration k has stage
  // 0 on number k + 1, with numbers k .. k + 2 in LDS
  const int iters = ch + 2 * H - 2 + 2 * (B.steps - 1) - (H - 1), most = ch + 2 * H - 1;
  auto compute = [&](int k, bool stores) __attribute__((always_inline)) {
    const int c = k + 1 - 2 * stage;  // this stage's row number
    if (!on || c < first || c > most - first) return;
    const int s0 = c % R, sm = (c + R - 1) % R, sp = (c + 1) % R;
    const int2 en = ent[(c & (kSweepEntries - 1)) * stride + n];
    if (en.x < 0) return;
    const TileAt P{plane, s0 * stride + n, (sm - s0) * stride, (sp - s0) * stride};
    const double ns = WALSH ? nsl[s0 * stride + n] : 0.;
    int loc[9];
    if (!stores && !(stage & 1)) tile_locs<true>(P, (uint32_t)en.y, loc);
    else tile_locs<false>(P, (uint32_t)en.y, loc);
    if (!stores && !(stage & 1))
      tile_node<NS, SOL, WALSH, true, false>(B, A, lds, loc, en.x, ns, (uint32_t)en.y, rows, stage);
    else if (stores || last) tile_node<NS, SOL, WALSH, false, true>(B, A, lds, loc, en.x, ns, (uint32_t)en.y, rows, stage);
    else tile_node<NS, SOL, WALSH, false, false>(B, A, lds, loc, en.x, ns, (uint32_t)en.y, rows, stage);
  };
  if (stage == 3) {
    lds_barrier();
    for (int k = 0; k < iters; k++) {
      compute(k, true);
      lds_barrier();
    }
    return;
  }

  // loads are issued by every thread in every iteration (clamped, so that
  // their number is known and only the oldest are waited for)
  const int2 *mine = tab + (long)strip * nj * stride + (n < rw ? n : rw - 1);
  auto entry = [&](int q) __attribute__((always_inline)) -> int2 {
    int r = (y0 - H + (q < most ? q : most)) % nj;
    r = r < 0 ? r + nj : r;
    return mine[(long)r * stride];
  };
  struct Rows {
    tile_t<NS> v[3];
    double ns;
  };
  auto load = [&](Rows &q, int2 e, int number) __attribute__((always_inline)) {
    if (stage == 0 && n < rw) ent[(number & (kSweepEntries - 1)) * stride + n] = e;
    const uint32_t idx = e.x < 0 ? 0u : (uint32_t)e.x;
    const double *p = B.A.F + (size_t)foff<9, NS>(0, 3 * stage, idx);
#pragma unroll
    for (int k = 0; k < 3; k++) q.v[k] = *(const tile_t<NS> *)(p + k * kTile * NS);
    if (WALSH) q.ns = A.ns[idx];
  };
  auto fill = [&](const Rows &q, int number) __attribute__((always_inline)) {
    if (number > most || n >= rw) return;
    const int at = number % R * stride + n;
#pragma unroll
    for (int k = 0; k < 3; k++) lds[(3 * stage + k) * plane + at] = q.v[k];
    if (WALSH && stage == 0) nsl[at] = q.ns;
  };
  Rows q0, q1;
  {
    const int2 e0 = entry(0), e1 = entry(1), e2 = entry(2);
    Rows q2;
    load(q0, e0, 0);
    load(q1, e1, 1);
    load(q2, e2, 2);
    fill(q0, 0);
    fill(q1, 1);
    fill(q2, 2);
  }
  load(q0, entry(3), 3);
  load(q1, entry(4), 4);
  int2 e0 = entry(5), e1 = entry(6);
  lds_barrier();
  auto iterate = [&](int k, Rows &q, int2 &e) __attribute__((always_inline)) {
    fill(q, k + 3);
    load(q, e, k + 5);
    e = entry(k + 7);
    compute(k, false);
    lds_barrier();
  };
  for (int k = 0; k < iters; k += 2) {
    iterate(k, q0, e0);
    if (k + 1 < iters) iterate(k + 1, q1, e1);
  }
}

}  // namespace lbm
