// Doubles contractions W(ijk) of the (T) hot path on FP64 MFMA (gfx950).
//
// The twelve GEMM terms of doubles_contribution (reference
// src/atrip/Equations.cxx:620-680, loop form :686-726) are regrouped by the
// W index that the single-occupied-index operand carries:
//   class w ("ij|k"): P0, P1, H5, H2   A-pair (a,b), columns over c
//   class v ("ik|j"): P3, P5, H1, H4   A-pair (a,c), columns over b
//   class u ("jk|i"): P4, P2, H0, H3   A-pair (b,c), columns over a
// Within a class the four terms share one output layout, so they are one GEMM
//   C[(p,q), (t,r)] = sum_kappa A[(p,q), kappa] B[kappa, (t,r)]
// with kappa running over four segments (E, E, L, L) and the hole operands
// stored pre-negated.  The A operand depends only on the class's index pair,
// so one A tile serves every tuple of the window that shares the pair (the
// cross-tuple reuse that per-tuple GEMMs lack), and the t index runs over
// the third tuple index inside the window.  Each class writes its own buffer
// in the W layout W[i + No j + No^2 k]; the energy kernel sums the three.
//
// MFMA v_mfma_f64_16x16x4f64, operands straight from global memory (L2/MALL
// resident) into registers.  Operands are 16-row x 8-kappa tiles in lane
// order (f64_at): lane group q = lane/16 feeds kappa k0 + 2q (k-step 0) and
// k0 + 2q + 1 (k-step 1) of an 8-deep chunk, one 16-byte load per lane and
// fragment over 1 KiB of consecutive addresses.  Read from rows K apart, as
// before, the same load touched 64 lines, one L1 tag access each, and the
// texture units were 80 % busy with them at 5x5 and the bound of every
// smaller tile (No=16, Nv=120 with 4x4: 290 -> 245 us per launch of 2048
// slots; 5x5 at No=40: 10.42 -> 10.25 ms).  An 8-deep chunk needs half the
// operand registers of a 16-deep one, so tiles up to 4x4 run two waves per
// SIMD.
#include "doubles_common.hpp"

namespace atrip_amd {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef double d2 __attribute__((ext_vector_type(2)));

constexpr int KC = 8;     // kappa per chunk: one operand tile
constexpr int TILE = 128;  // doubles per operand tile

// Operands of one set of four K segments.
struct OperandSet {
  // T3s, H3s: row-swapped copies (null: read the swapped rows of T3, H3)
  const double *T3, *T3s, *V3, *H3, *H3s, *T2N, *T2TN;
};
struct DoublesParams {
  OperandSet op;
  // bytes from each array of the first set to the second's (chosen at run
  // time by mask: a choice between two pointer members put P in scratch)
  struct {
    int64_t T3, T3s, V3, H3, H3s, T2N, T2TN;
  } to2;
  int nseg;  // K segments: 4, or 8 over both sets (a complex product's plane)
  WindowArgs win;
  double *G;
  int64_t No, Nv, Kv, Ko, N2, N2p, W3, slots;
  GLayout lay;
};

// Operand sets of a wave of FM x FN fragments: two, four where a chunk is
// shorter than 1000 cycles (2x2 at No=40: 52.1 -> 55.4 TFLOP/s; deeper sets
// from 4x2 on cost more registers than they hide: 59.7 -> 57.0 at No=16).
constexpr int depth(int FM, int FN) {
  return FM * FN >= 8 ? 2 : 4;
}

// The FM x FN occupied fragments of one wave of a tile of 32 TM x 32 TN.  The
// two waves of each direction take the tile's fragments in turn, so a tile at
// the edge of the GEMM leaves both about the same number.
template <int TM, int TN, int WR, int FM, int FN>
__device__ __forceinline__ void f64_wave(const DoublesParams &P,
                                         const TileWork &T, int No, int lane,
                                         int wm, int wn) {
  constexpr int MT = 32 * TM, NT = 32 * TN;
  const int kk = lane >> 4, l16 = lane & 15;
  const int64_t N2 = P.N2, Nv = P.Nv, N2p = P.N2p;
  int32_t cy[FN], crr[FN];  // third index and column index of the columns
#pragma unroll
  for (int g = 0; g < FN; g++) {
    int n = T.nt * NT + (2 * g + wn) * 16 + l16;
    if (n >= T.ncols) n = T.ncols - 1;  // safe load address, not stored
    cy[g] = T.y0 + n / No;
    crr[g] = n % No;
  }
  // rows: straight (p + No q) and swapped (q + No p) row of the A slab
  // (rows past the last occupied tile read its last row, not stored)
  int32_t rowS[FM], rowW[FM];
#pragma unroll
  for (int f = 0; f < FM; f++) {
    int m = T.mt * MT + (WR * f + wm) * 16 + l16;
    rowS[f] = m < N2p ? m : (int)N2p - 16 + l16;
    if (m >= N2) m = (int)N2 - 1;
    rowW[f] = m / No + No * (m % No);
  }

  const int64_t Kv = P.Kv, Ko = P.Ko;
  // segments: 0 T3[x1] straight, 1 T3[x2] swapped, 2 H3[x2] straight,
  //           3 H3[x1] swapped
#define SEL(x) ((const double *)((const char *)P.op.x + (o2_ & P.to2.x)))
#define SET_PTRS(SG)                                                        \
  {                                                                         \
    const int64_t o2_ = (SG) >= 4 ? -1 : 0;                                 \
    const int s_ = (SG)&3;                                                  \
    const int64_t K_ = s_ < 2 ? Kv : Ko;                                    \
    const int64_t xr_ = (s_ == 0 || s_ == 3 ? T.x1 : T.x2) * N2p;           \
    const bool sw_ = (s_ & 1) && (s_ < 2 ? P.op.T3s : P.op.H3s);            \
    const double *Ab_ = sw_ ? (s_ < 2 ? SEL(T3s) : SEL(H3s))                \
                            : (s_ < 2 ? SEL(T3) : SEL(H3));                 \
    _Pragma("unroll") for (int f = 0; f < FM; f++) ap[f] =                  \
        Ab_ + f64_row(xr_ + ((s_ & 1) && !sw_ ? rowW[f] : rowS[f]), K_) +   \
        32 * kk;                                                            \
    _Pragma("unroll") for (int g = 0; g < FN; g++) {                        \
      int wh_;                                                              \
      const int64_t R_ =                                                    \
          b_row(T.cl, s_, T.x1, T.x2, cy[g], crr[g], Nv, No, wh_);          \
      const double *B_ = wh_ == 0 ? SEL(V3) : wh_ == 1 ? SEL(T2N)           \
                                                       : SEL(T2TN);         \
      bp[g] = B_ + f64_row(R_, K_) + 32 * kk;                               \
    }                                                                       \
  }
  d4 acc[FM][FN];
#pragma unroll
  for (int f = 0; f < FM; f++)
#pragma unroll
    for (int g = 0; g < FN; g++) acc[f][g] = d4{0.0, 0.0, 0.0, 0.0};

  // Software pipeline of D operand sets used in turn: the loads of D - 1
  // chunks are in flight behind the MFMAs of one (no register copies between
  // the sets, hence no wait on the in-flight loads).  A chunk is 128 FM FN
  // cycles of MFMA against a load latency of 1000 (L2) to 2500 cycles, so
  // small fragments need more sets: see depth().
  constexpr int D = depth(FM, FN);
  const double *ap[FM], *bp[FN];
  d2 a[D][FM], b[D][FN];
#define LOAD(J)                                                             \
  {                                                                         \
    const int64_t at_ = TILE * (int64_t)(sg < nseg ? c : nch - 1);          \
    _Pragma("unroll") for (int f = 0; f < FM; f++) a[J][f] =                \
        *(const d2 *)(ap[f] + at_);                                         \
    _Pragma("unroll") for (int g = 0; g < FN; g++) b[J][g] =                \
        *(const d2 *)(bp[g] + at_);                                         \
    __builtin_amdgcn_sched_barrier(0);                                      \
  }
#define COMPUTE(J)                                                          \
  _Pragma("unroll") for (int s = 0; s < 2; s++)                             \
      _Pragma("unroll") for (int f = 0; f < FM; f++)                        \
          _Pragma("unroll") for (int g = 0; g < FN; g++) acc[f][g] =        \
              __builtin_amdgcn_mfma_f64_16x16x4f64(a[J][f][s], b[J][g][s],  \
                                                   acc[f][g], 0, 0, 0);
  // One pipeline through the segments: (sg, c) is the next chunk to
  // load, and past a segment's end the pointers move to the next segment's
  // chunk 0 in place, so every segment but the first starts with its first
  // chunks in flight (3 % faster at No=40 than a pipeline restarted per
  // segment).  A segment ends at the last chunk that holds an occupied
  // kappa.  The prefetch is issued unconditionally (after the last chunk it
  // re-reads it, a load never used) so every path into a COMPUTE has the
  // same loads outstanding.
  const int nseg = P.nseg;
  int sg = 0;
  int nch = (int)((Nv + KC - 1) / KC), c = 0;
  SET_PTRS(0);
#define ADVANCE()                                                            \
  if (sg < nseg && ++c == nch && ++sg < nseg) {                              \
    SET_PTRS(sg);                                                            \
    nch = (int)((((sg & 3) < 2 ? Nv : No) + KC - 1) / KC);                   \
    c = 0;                                                                   \
  }
#pragma unroll
  for (int j = 0; j < D - 1; j++) {
    LOAD(j);
    ADVANCE();
  }
  // (one exit: leaving the loop between two sets made the compiler copy the
  // accumulators between register files on every turn; the chunks of a last
  // part turn follow it)
  int left = nseg / 2 * (int)((Nv + KC - 1) / KC + (No + KC - 1) / KC);
#pragma unroll 1
  for (; left >= D; left -= D) {
#pragma unroll
    for (int j = 0; j < D; j++) {
      LOAD((j + D - 1) % D);
      ADVANCE();
      COMPUTE(j);
    }
  }
#pragma unroll
  for (int j = 0; j < D - 1; j++)
    if (j < left) COMPUTE(j);
#undef ADVANCE
#undef LOAD
#undef COMPUTE

#undef SET_PTRS
#undef SEL
  // store: for v_mfma_f64_16x16x4f64, D[i][j] sits in lane j + 16*(i%4),
  // register i/4 (measured on gfx950)
  const int64_t per = (int64_t)P.win.ea * P.win.eb * P.win.ec;
  double *Gc = P.G + (T.cl * P.slots + T.w * per) * P.W3;
  double *Gs[FN];  // column bases; null past the last column
#pragma unroll
  for (int g = 0; g < FN; g++) {
    const int n = T.nt * NT + (2 * g + wn) * 16 + l16;
    const int t = n / No;
    Gs[g] = n < T.ncols ? Gc + (int64_t)(T.slot0 + t * T.slot_step) * P.W3 +
                              g_col(n - t * No)
                        : nullptr;
  }
#pragma unroll
  for (int f = 0; f < FM; f++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int m = T.mt * MT + (WR * f + wm) * 16 + 4 * r + kk;
      if (m >= N2) continue;
      const uint32_t o = g_row(P.lay, m);
#pragma unroll
      for (int g = 0; g < FN; g++)
        if (Gs[g]) Gs[g][o] = acc[f][g][r];
    }
}

// Dispatch on the wave's occupied column fragments, n <= FN of them.
template <int TM, int TN, int WR, int FM, int FN>
__device__ __forceinline__ void f64_columns(const DoublesParams &P,
                                            const TileWork &T, int No,
                                            int lane, int wm, int wn, int n) {
  if constexpr (FN > 1) {
    if (n < FN) {
      f64_columns<TM, TN, WR, FM, FN - 1>(P, T, No, lane, wm, wn, n);
      return;
    }
  }
  f64_wave<TM, TN, WR, FM, FN>(P, T, No, lane, wm, wn);
}

// Dispatch on the wave's occupied row fragments, m <= FM of them.
template <int TM, int TN, int WR, int FM, int FN>
__device__ __forceinline__ void f64_rows(const DoublesParams &P,
                                         const TileWork &T, int No, int lane,
                                         int wm, int wn, int m, int n) {
  if constexpr (FM > 1) {
    if (m < FM) {
      f64_rows<TM, TN, WR, FM - 1, FN>(P, T, No, lane, wm, wn, m, n);
      return;
    }
  }
  f64_columns<TM, TN, WR, FM, FN>(P, T, No, lane, wm, wn, n);
}

template <int FM, int FN, int WR>
__global__ __launch_bounds__(128 * WR, 2) void doubles_f64_kernel(
    DoublesParams P) {
  const int No = (int)P.No;
  TileWork T;
  if (!tile_work(P.win, (uint64_t)P.Nv, No, 32 * FN, T)) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // wave -> (row, column) of the WR x 2 waves.  The tiles beyond 4x4 run
  // eight waves (four rows), two per SIMD, instead of four of twice the
  // registers: the second wave covers the other's loads (5x5 at No=40,
  // Nv=400 61.4 -> 66.3 TFLOP/s with the valid columns, 4x5 at No=26 44.7 ->
  // 50.7, 5x4 at No=31 48.5 -> 50.7).  The two waves of a SIMD (w, w + 4) are
  // two rows apart, so that they hold five of ten row fragments between them.
  const int wn = WR == 2 ? wave & 1 : wave >> 2;
  const int wm = WR == 2 ? wave >> 1 : (wave + 2 * wn) & 3;
  // Fragments of this wave that hold rows and columns.  Tiles at the edges
  // of the GEMM run the instance of their size instead of the whole tile on
  // padding (one instance with per-fragment branches doubled the
  // accumulators; with only whole and half row counts No=14, 12.25 row
  // fragments, paid for 16 instead of 14).
  constexpr int RF = (2 * FM + WR - 1) / WR;  // row fragments of a wave
  const int m = occupied(P.N2 - (int64_t)T.mt * 32 * FM, wm, WR, 16, 2 * FM);
  const int n = occupied(T.ncols - (int64_t)T.nt * 32 * FN, wn, 2, 16, 2 * FN);
  if (!m || !n) return;
  f64_rows<FM, FN, WR, RF, FN>(P, T, No, lane, wm, wn, m, n);
}

}  // namespace

hipError_t launch_doubles_f64(const DevSystem &s, const DevSystem *s2,
                              const BatchArgs &b, bool use_j, double *G,
                              int tile, hipStream_t st) {
  DoublesParams P;
  P.nseg = s2 ? 8 : 4;
  auto set = [&](const DevSystem &x) {
    return OperandSet{x.T3, x.T3s, use_j ? x.V3J : x.V3, use_j ? x.H3J : x.H3,
                      use_j ? x.H3Js : x.H3s, x.T2N, x.T2TN};
  };
  const OperandSet a = set(s), z = set(s2 ? *s2 : s);
  P.op = a;
  // (swapped copies are used when both sets have them)
  if (!a.T3s || !z.T3s) P.op.T3s = nullptr;
  if (!a.H3s || !z.H3s) P.op.H3s = nullptr;
  auto to = [](const double *x, const double *y) {
    return (int64_t)((intptr_t)y - (intptr_t)x);
  };
  P.to2 = {to(a.T3, z.T3), to(a.T3s, z.T3s), to(a.V3, z.V3), to(a.H3, z.H3),
           to(a.H3s, z.H3s), to(a.T2N, z.T2N), to(a.T2TN, z.T2TN)};
  P.win = b;
  P.G = G;
  P.No = s.No;
  P.Nv = s.Nv;
  P.Kv = s.Kv;
  P.Ko = s.Ko;
  P.N2 = s.No * s.No;
  P.N2p = pad16(P.N2);
  P.lay = g_layout(s.No);
  P.W3 = g_elems(s.No);
  P.slots = b.slots;
  tile = pick_tile(tile, s.No, std::max(b.ea, std::max(b.eb, b.ec)));
  const int FM = tile_fm(tile), FN = tile_fn(tile);
  const int64_t grid = doubles_grid(P.win, s.No, 32 * FM, 32 * FN);
  if (grid <= 0) return hipSuccess;
  if (grid > MAX_GRID) return hipErrorInvalidConfiguration;
#define LAUNCH(A, B, WR)                                                     \
  if (FM == A && FN == B)                                                    \
    hipLaunchKernelGGL((doubles_f64_kernel<A, B, WR>), dim3((unsigned)grid), \
                       dim3(128 * WR), 0, st, P);
  LAUNCH(2, 2, 2) LAUNCH(4, 2, 2) LAUNCH(2, 4, 2) LAUNCH(4, 4, 2)
  LAUNCH(3, 3, 2) LAUNCH(5, 5, 4) LAUNCH(4, 5, 4) LAUNCH(5, 4, 4)
#undef LAUNCH
  return hipGetLastError();
}

}  // namespace atrip_amd
