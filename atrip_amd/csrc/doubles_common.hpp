// Work decomposition shared by the doubles kernels (FP64 and split FP32):
// the class/segment table of the regrouped doubles contractions.
#pragma once

#include <algorithm>

#include "internal.hpp"

namespace atrip_amd {

// One workgroup's share of a launch over windows of eb x ec columns (see
// BatchArgs): a class, an A-pair of its window and one tile of that pair's
// GEMM.  The GEMM's columns are only those of valid tuples: the valid third
// indices of a pair are consecutive (the tuples of a pair are ordered along
// the third index, so a tuple range cuts them at the ends), so column n is
// index n % No of third index y0 + n / No, n < ncols.  Column tuple slot:
// slot0 + (n / No) slot_step.
struct TileWork {
  int cl, mt, nt, w;
  int32_t x1, x2;  // A-pair: w (a,b), v (a,c), u (b,c)
  int32_t y0;      // first valid third index
  int ncols;
  int slot0, slot_step;
};

// Work of this workgroup; false when its tile holds no column.  Workgroup b
// runs on XCD b % 8, and an XCD hands its workgroups to its shader engines in
// turn, whatever they cost.  So
//  - the units (class, pair) of a window go round the XCDs and a unit's tiles
//    stay on one, where they share the pair's A rows and columns in its L2
//    (one contiguous eighth of the launch per XCD left the XCDs without
//    diagonal windows to work longer), and
//  - each unit starts its tiles, and each window its units, one place further
//    on, and the column tiles of a row of tiles are turned by a mix of the
//    row's bits: with a fixed order the tiles at the GEMM's edges, or those
//    without a valid column, came to the same shader engines in every unit
//    (No=20, Nv=183 with 4x4 tiles, columns 128 + 32: half the chip idle,
//    29.7 TFLOP/s against 50.7; No=38, Nv=204 with 3x3: 37.7 against 50.6).
//    Column tiles stay next to each other (row tiles first costs 4x4 at No=40
//    5 %: neighbours then share no A rows).
__device__ __forceinline__ bool tile_work(const WindowArgs &W, uint64_t Nv,
                                          int No, int ntile_cols,
                                          TileWork &T) {
  const uint32_t bid = blockIdx.x, j = bid >> 3;
  const uint32_t tiles = (uint32_t)(W.mtiles * W.ntiles);
  const uint32_t units =
      (uint32_t)(W.ea * W.eb + W.ea * W.ec + W.eb * W.ec);
  const uint32_t per = (units + 7) / 8 * tiles;  // of a window, per XCD
  T.w = (int)(j / per);
  uint32_t q = j - (uint32_t)T.w * per + (uint32_t)T.w % per;
  if (q >= per) q -= per;
  const uint32_t uq = q / tiles;
  uint32_t tile = q - uq * tiles + uq % tiles;
  if (tile >= tiles) tile -= tiles;
  int u = (int)(8 * uq + (bid & 7));
  if (u >= (int)units) return false;
  const uint32_t mt = tile / (uint32_t)W.ntiles;
  T.mt = (int)mt;
  T.nt = (int)((tile + mt + (mt >> 1) + (mt >> 2)) % (uint32_t)W.ntiles);
  const int32_t a0 = W.windows[3 * T.w], b0 = W.windows[3 * T.w + 1],
                c0 = W.windows[3 * T.w + 2];
  int edge;
  int32_t y;
  if (u < W.ea * W.eb) {
    const int o1 = u / W.eb, o2 = u - o1 * W.eb;
    T.cl = 0; T.x1 = a0 + o1; T.x2 = b0 + o2;
    y = c0; edge = W.ec;
    T.slot0 = u * W.ec; T.slot_step = 1;
  } else if ((u -= W.ea * W.eb) < W.ea * W.ec) {
    const int o1 = u / W.ec, o2 = u - o1 * W.ec;
    T.cl = 1; T.x1 = a0 + o1; T.x2 = c0 + o2;
    y = b0; edge = W.eb;
    T.slot0 = o1 * W.eb * W.ec + o2; T.slot_step = W.ec;
  } else {
    u -= W.ea * W.ec;
    const int o1 = u / W.ec, o2 = u - o1 * W.ec;
    T.cl = 2; T.x1 = b0 + o1; T.x2 = c0 + o2;
    y = a0; edge = W.ea;
    T.slot0 = u; T.slot_step = W.eb * W.ec;
  }
  const int lane = threadIdx.x & 63;
  const int64_t yl = y + lane;
  const uint64_t a = T.cl == 2 ? yl : T.x1,
                 b = T.cl == 0 ? T.x2 : T.cl == 1 ? yl : T.x1,
                 c = T.cl == 0 ? yl : T.x2;
  bool ok = lane < edge && tuple_ok(Nv, a, b, c);
  if (ok && (W.first > 0 || W.last != ~0ULL)) {
    const uint64_t idx = tuple_index(W.aprefix, Nv, a, b, c);
    ok = idx >= W.first && idx < W.last;
  }
  const uint64_t mask = __ballot(ok);
  if (!mask) return false;
  const int t0 = __builtin_ctzll(mask), n = __popcll(mask);
  T.y0 = y + t0;
  T.slot0 += t0 * T.slot_step;
  T.ncols = n * No;
  return T.nt * ntile_cols < T.ncols;
}

// Fragments of `width` that wave w of nw holds of `left` rows or columns of a
// tile of at most `most` fragments, taken in turn (w, w + nw, ...).
__device__ __forceinline__ int occupied(int64_t left, int w, int nw, int width,
                                        int most) {
  const int64_t all = (left + width - 1) / width;
  const int frags = all < most ? (int)all : most;
  return frags > w ? (frags - w + nw - 1) / nw : 0;
}

// Row of segment sg's B operand at column (y, rr) of class cl with A-pair
// (x1, x2), and its array (0: V(xy) slabs, 1: -T(xy)[L,n], 2: -T(xy)[n,L]).
// By segment, with (a,b,c) the column's tuple:
//   class w: P0 V(bc), P1 V(ac), H5 -TAC[L,k], H2 -TBC[L,k]
//   class v: P3 V(cb), P5 V(ab), H1 -TAB[L,j], H4 -TBC[j,L]
//   class u: P4 V(ca), P2 V(ba), H0 -TAB[i,L], H3 -TAC[i,L]
// against T(x1) straight, T(x2) swapped, Vhhh(x2) straight, Vhhh(x1) swapped.
__device__ __forceinline__ int64_t b_row(int cl, int sg, int32_t x1,
                                         int32_t x2, int32_t y, int32_t rr,
                                         int64_t Nv, int64_t No, int &which) {
  const int64_t x = sg == 0 || sg == 3 ? x2 : x1;
  const bool tr = sg >= 2 && (cl == 2 || (cl == 1 && sg == 3));
  which = sg < 2 ? 0 : tr ? 2 : 1;
  return (tr ? y + Nv * x : x + Nv * y) * No + rr;
}

// Grid of a doubles launch: units padded to the eight XCDs times the tiles
// of a unit; 0 when it holds nothing.
inline int64_t doubles_grid(WindowArgs &W, int64_t No, int64_t mt_rows,
                            int64_t nt_cols) {
  const int64_t emax = std::max(W.ea, std::max(W.eb, W.ec));
  W.mtiles = (int)((No * No + mt_rows - 1) / mt_rows);
  W.ntiles = (int)((emax * No + nt_cols - 1) / nt_cols);
  const int64_t units = W.ea * W.eb + W.ea * W.ec + W.eb * W.ec;
  return (units + 7) / 8 * 8 * W.nw * W.mtiles * W.ntiles;
}

// Tile shapes (FM x FN fragments of 16x16 of each of 2x2 waves; 5x5, 4x5 and
// 5x4 run as 4x2 waves of half the rows) and the rate of each per useful
// tile element in FP64, as fitted to kernels that computed a tile's padding and
// the columns of tuples that do not exist (whole-system runs at No=20, 26, 31,
// 38 and 40; 2x2 and 2x4 older still).  The present kernels compute neither.
// Their rates, in TFLOP/s of the doubles kernel over a sample of the whole
// space at edge 8, as picked / with 4x4: No=20, Nv=183 54.0 (5x5) / 55.0, 26/308
// 52.3 (5x4) / 55.2, 31/270 55.5 (5x4) / 59.2, 38/204 55.3 (4x5) / 56.1, 40/400
// (edge 12) 65.6 (5x5) / 66.8, where the same tile timed twice differs by 3 %.
// The table stands until it is fitted anew; host tests hold its picks.
constexpr int N_TILES = 8;
__host__ __device__ inline int tile_fm(int t) {
  const int v[N_TILES] = {2, 4, 2, 4, 3, 5, 4, 5};
  return v[t];
}
__host__ __device__ inline int tile_fn(int t) {
  const int v[N_TILES] = {2, 2, 4, 4, 3, 5, 5, 4};
  return v[t];
}
inline double tile_rate(int t) {
  const double v[N_TILES] = {0.44, 0.575, 0.51, 0.627, 0.61, 0.69, 0.677, 0.69};
  return v[t];
}

// Automatic tile: best of the rates above times the useful fraction of the
// padded M = No^2 by N = nb*No tile grid.
inline int pick_tile(int tile, int64_t No, int nb) {
  if (tile >= 0 && tile < N_TILES) return tile;
  double best = -1.0;
  int pick = 0;
  const double M = (double)No * No, N = (double)nb * No;
  for (int t = 0; t < N_TILES; t++) {
    const double mt = 32.0 * tile_fm(t), nt = 32.0 * tile_fn(t);
    const double use = M / (__builtin_ceil(M / mt) * mt) *
                       N / (__builtin_ceil(N / nt) * nt);
    const double score = tile_rate(t) * use;
    if (score > best) {
      best = score;
      pick = t;
    }
  }
  return pick;
}

// Automatic window edge of the plain path: the doubles GEMMs of a window
// have N = nb No columns, so the edge sets how much of the last column tile
// is empty.  Each candidate edge is scored by its best tile's modelled
// rate (pick_tile's model) times the share of valid tuples in the windows;
// an edge other than 8 is taken only when it scores 15 % above 8 (the
// model's own error).  The model charges empty columns as the earlier kernels
// paid for them (No=26, Nv=308: 40.6 TFLOP/s with edge 6, its pick, 33.2 with 8).
// With the present ones edges 6, 8 and 12 lie within 5 % there (51.6, 52.3, 53.9)
// and within 7 % at No=20, 31 and 38 but for edge 6 at No=20 and 38 (11 % and
// 8 % below 8).
inline int auto_window(int64_t No, int64_t Nv) {
  auto score = [&](int nb) {
    const int t = pick_tile(-1, No, nb);
    const double mt = 32.0 * tile_fm(t), nt = 32.0 * tile_fn(t);
    const double M = (double)No * No, N = (double)nb * No;
    const double use = M / (__builtin_ceil(M / mt) * mt) *
                       N / (__builtin_ceil(N / nt) * nt);
    const double nblk = __builtin_ceil((double)Nv / nb);
    const double cells = nblk * (nblk + 1) * (nblk + 2) / 6 * nb * nb * nb;
    const double tuples = (double)Nv * (Nv + 1) * (Nv + 2) / 6;
    return tile_rate(t) * use * tuples / cells;
  };
  const double base = score(8);
  int pick = 8;
  double best = 1.15 * base;
  for (int nb : {6, 12}) {
    const double s = score(nb);
    if (s > best) {
      best = s;
      pick = nb;
    }
  }
  return pick;
}

// Windows per launch when the caller set none: as many as keep the launch's
// class buffers (slot_bytes per tuple slot, `per` slots per window) within
// LAUNCH_BYTES, at least LEAST_BATCH of the plan's.  Every launch ends in a partly
// filled chip and is followed by an epilogue that starts on an empty one, and
// small systems are launch-bound: against four windows per launch, No=4,
// Nv=36 takes 0.11 ms instead of 0.16, No=10, Nv=50 1.25 instead of 2.10,
// No=16, Nv=120 42.5 instead of 45.6, No=26, Nv=308 (100,000 tuples) 160
// instead of 174; beyond 2 GiB the gain is below 1 %.  (LEAST_BATCH windows
// pass 2 GiB from No=33 in FP64: 3.1 GB at No=40, where five fit in FP32, and
// 12.9 GB at No=60; twice that with (cT).)
constexpr int LEAST_BATCH = 4;
constexpr int64_t LAUNCH_BYTES = (int64_t)2 << 30;
inline int auto_batch(int64_t slot_bytes, int64_t per) {
  return (int)std::min<int64_t>(4096, LAUNCH_BYTES / (slot_bytes * per));
}

// Wave tiles of FM x FN fragments of 32 x 32 (2 x 2 waves per workgroup)
// of the 32x32-MFMA kernels (bf16x3, split FP32), variant t of the "tile"
// option.
constexpr int N_T32_TILES = 10;
__host__ __device__ inline int t32_fm(int t) {
  const int v[N_T32_TILES] = {2, 2, 3, 2, 3, 2, 3, 4, 3, 4};
  return v[t];
}
__host__ __device__ inline int t32_fn(int t) {
  const int v[N_T32_TILES] = {2, 3, 2, 4, 3, 5, 5, 4, 4, 3};
  return v[t];
}
// Rate of each variant relative to 4x4, per useful tile element: variants
// 4-9 measured in bf16x3 on MI355X (mean of No=40, Nv=400 and No=60,
// Nv=600, each divided by its padded-grid fraction; 2x5 re-measured against
// 3x5 at No=40 with the one-pipeline K loop, 1.5 % faster there); variants
// 0-3 from the operand bytes per MFMA cycle, FM FN / (FM + FN), scaled by the
// ratio that measured variants 4 and 5 show over the same formula.
inline double t32_rate(int t) {
  const double v[N_T32_TILES] = {0.62, 0.75, 0.75, 0.83, 0.985,
                                 0.966, 0.988, 1.0, 0.989, 0.952};
  return v[t];
}
// Automatic variant: rate times the useful fraction of the padded
// M = No^2 by N = nb No tile grid.
inline int pick_t32_tile(int tile, int64_t No, int nb) {
  if (tile >= 0 && tile < N_T32_TILES) return tile;
  double best = -1.0;
  int pick = 0;
  const double M = (double)No * No, N = (double)nb * No;
  for (int t = 0; t < N_T32_TILES; t++) {
    const double mt = 64.0 * t32_fm(t), nt = 64.0 * t32_fn(t);
    const double use = M / (__builtin_ceil(M / mt) * mt) *
                       N / (__builtin_ceil(N / nt) * nt);
    const double score = t32_rate(t) * use;
    if (score > best) {
      best = score;
      pick = t;
    }
  }
  return pick;
}

}  // namespace atrip_amd
