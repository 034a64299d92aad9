// Doubles contractions W(ijk) from three-part bf16 operands (the bf16x3
// mixed-precision form).
//
// Same regrouped class GEMMs and tuple windows as the FP64 kernel
// (doubles_f64.hip).  Every operand x is held as three bf16 parts,
//     b0 = bf16(x),  b1 = bf16(x - b0),  b2 = bf16(x - b0 - b1),
// which carry 24 significant bits, as many as an FP32 value (each part is
// at most 2^-9 of the one before).  A product is formed from the six part
// products down to the 2^-18 level,
//     a0 b0 + a0 b1 + a1 b0 + a1 b1 + a0 b2 + a2 b0,
// on v_mfma_f32_32x32x16_bf16 with FP32 accumulation; the three dropped
// terms (a1 b2, a2 b1, a2 b2) are at most 2^-27 of the product, below an
// FP32 rounding (2^-24).  Each MFMA takes one part of a 32-row A fragment
// and one part of a 32-column B fragment over a whole 16-deep K chunk (lane
// l feeds row/column l % 32 at kappa k0 + 8 (l / 32) + 0..7), so a chunk is
// six MFMAs per fragment pair (6 x 32 cycles per 32 x 32 block, against
// 16 x 64 cycles in FP64) and the operands are the loaded registers as
// they are.  Operands are in the tiled layout (TriGeom): each part of a
// 32 x 16 fragment chunk is 1 KiB contiguous in lane order, one 16-byte load
// per lane; the swapped A segments read the row-swapped copies, so every A
// fragment is 32 consecutive rows.  Class buffers are FP32 and are widened
// to FP64 by the class-sum kernel; singles, the energy and all sums stay
// FP64 (energy.hip).
#include "doubles_common.hpp"

namespace atrip_amd {
namespace {

typedef float f16v __attribute__((ext_vector_type(16)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

// A lane's three parts at its eight kappa of a chunk.
struct Parts {
  bf8 p0, p1, p2;
};

__device__ __forceinline__ Parts load_parts(const __bf16 *p) {
  Parts r;
  r.p0 = *(const bf8 *)p;
  r.p1 = *(const bf8 *)(p + 512);
  r.p2 = *(const bf8 *)(p + 1024);
  return r;
}

struct TriParams {
  // tiled parts; T3s / H3s: the row-swapped copies
  const __bf16 *T3, *T3s, *H3, *H3s, *V3, *T2N, *T2TN;
  WindowArgs win;
  float *G;
  int64_t No, Nv, Kv, Ko, N2, N2p, W3, slots;
  GLayout lay;
};

// The FM x FN occupied fragments of one wave of a tile of 64 TM x 64 TN (the
// waves of each direction take the fragments in turn, as the FP64 kernel).
template <int TM, int TN, int FM, int FN>
__device__ __forceinline__ void tri_wave(const TriParams &P, const TileWork &T, int No,
                                         int lane, int wm, int wn) {
  constexpr int MT = 64 * TM, NT = 64 * TN;
  const int kh = lane >> 5, l32 = lane & 31;
  const int64_t N2 = P.N2, Nv = P.Nv;
  int32_t cy[FN], crr[FN];  // third index and column index of the columns
#pragma unroll
  for (int g = 0; g < FN; g++) {
    int n = T.nt * NT + (2 * g + wn) * 32 + l32;
    if (n >= T.ncols) n = T.ncols - 1;  // safe load address, not stored
    cy[g] = T.y0 + n / No;
    crr[g] = n % No;
  }
  // A rows: the swapped segments read the same rows of the row-swapped
  // copies (rows past the last occupied tile read its own, not stored).
  const int64_t Kv = P.Kv, Ko = P.Ko, N2p = P.N2p;
  int32_t rowS[FM];
#pragma unroll
  for (int f = 0; f < FM; f++) {
    const int m = T.mt * MT + (2 * f + wm) * 32 + l32;
    rowS[f] = m < N2p ? m : (int)N2p - 32 + l32;
  }

  // a lane's parts of chunk k0 start at its slot of the tile of k0: the
  // tile of k0 = 0 plus 96 k0 (1536 parts per 16-deep chunk); A lanes sit
  // at slot lane (aligned rows), B lanes at the slot of their row
  const __bf16 *ap[FM], *bp[FN];
#define SET_PTRS(SG)                                                          \
  {                                                                           \
    const int64_t K_ = (SG) < 2 ? Kv : Ko;                                    \
    const int64_t xa_ = ((SG) == 0 || (SG) == 3) ? T.x1 : T.x2;                   \
    const __bf16 *A_ = (SG) == 0   ? P.T3                                     \
                       : (SG) == 1 ? P.T3s                                    \
                       : (SG) == 2 ? P.H3                                     \
                                   : P.H3s;                                   \
    _Pragma("unroll") for (int f = 0; f < FM; f++) ap[f] =                    \
        A_ + tri_tile(xa_ * N2p + rowS[f], 0, K_) + 8 * lane;                 \
    _Pragma("unroll") for (int g = 0; g < FN; g++) {                          \
      int wh_;                                                                \
      const int64_t R_ =                                                      \
          b_row(T.cl, (SG), T.x1, T.x2, cy[g], crr[g], Nv, No, wh_);          \
      const __bf16 *B_ = wh_ == 0 ? P.V3 : wh_ == 1 ? P.T2N : P.T2TN;         \
      bp[g] = B_ + tri_tile(R_, 0, K_) + 8 * tri_lane(R_, 8 * kh);            \
    }                                                                         \
  }
#define LOAD(A, B, KOFF)                                                     \
  {                                                                          \
    _Pragma("unroll") for (int f = 0; f < FM; f++) A[f] =                    \
        load_parts(ap[f] + 96 * (KOFF));                                     \
    _Pragma("unroll") for (int g = 0; g < FN; g++) B[g] =                    \
        load_parts(bp[g] + 96 * (KOFF));                                     \
    __builtin_amdgcn_sched_barrier(0);                                       \
  }
  // a0 b0, a0 b1, a1 b0, a1 b1, a0 b2, a2 b0: each term over all blocks
  // before the next, so consecutive MFMAs update different accumulators
#define TERM(A, B, AP, BP)                                                   \
  _Pragma("unroll") for (int f = 0; f < FM; f++)                             \
      _Pragma("unroll") for (int g = 0; g < FN; g++) acc[f][g] =             \
          __builtin_amdgcn_mfma_f32_32x32x16_bf16(A[f].AP, B[g].BP,          \
                                                  acc[f][g], 0, 0, 0);
#define COMPUTE(A, B)                                                        \
  {                                                                          \
    TERM(A, B, p0, p0) TERM(A, B, p0, p1) TERM(A, B, p1, p0)                 \
    TERM(A, B, p1, p1) TERM(A, B, p0, p2) TERM(A, B, p2, p0)                 \
  }

  f16v acc[FM][FN];
#pragma unroll
  for (int f = 0; f < FM; f++)
#pragma unroll
    for (int g = 0; g < FN; g++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[f][g][r] = 0.f;

  // two operand sets in ping-pong: the loads of chunk c + 1 are in flight
  // behind the MFMAs of chunk c (a chunk is 6 FM FN MFMAs of 32 cycles, at
  // least 24 x 32 cycles; a third set would cost the registers the largest
  // tiles need and measured slower).  One pipeline runs through the four
  // segments: (sg, c) is the next chunk to load, and past a segment's end
  // the pointers move to the next segment's chunk 0 in place, so every
  // segment but the first starts with its first chunk in flight (2.7 %
  // faster at No=60 than a pipeline restarted per segment).  After the last
  // chunk the prefetch re-reads it (a load never used).
  static_assert(6 * (FM + FN) <= 63, "two chunks of loads must fit vmcnt");
  Parts a0[FM], b0[FN], a1[FM], b1[FN];
  int sg = 0;
  int64_t nch = Kv / KCHUNK, c = 0;
  SET_PTRS(0);
#define ADVANCE()                                                            \
  {                                                                          \
    if (++c == nch && ++sg < 4) {                                            \
      SET_PTRS(sg);                                                          \
      nch = (sg < 2 ? Kv : Ko) / KCHUNK;                                     \
      c = 0;                                                                 \
    }                                                                        \
  }
#define NEXT_OFF() (KCHUNK * (sg < 4 ? c : nch - 1))
  LOAD(a0, b0, 0);
  ADVANCE();
  // (each segment length occurs twice, so the number of chunks is even; a
  // second exit in the middle of the loop made the compiler copy the
  // accumulators between register files on every turn)
#pragma unroll 1
  for (int left = 2 * (int)((Kv + Ko) / KCHUNK); left; left -= 2) {
    LOAD(a1, b1, NEXT_OFF());
    ADVANCE();
    COMPUTE(a0, b0);
    LOAD(a0, b0, NEXT_OFF());
    if (sg < 4) ADVANCE();
    COMPUTE(a1, b1);
  }
#undef ADVANCE
#undef NEXT_OFF
#undef SET_PTRS
#undef LOAD
#undef TERM
#undef COMPUTE

  // 32x32 FP32-output MFMAs: D[i][j] in lane j + 32 ((i / 4) % 2), register
  // 4 (i / 8) + i % 4 (measured on gfx950)
  const int64_t per = (int64_t)P.win.ea * P.win.eb * P.win.ec;
  float *Gc = P.G + (T.cl * P.slots + T.w * per) * P.W3;
  float *Gs[FN];  // column bases; null past the last column
#pragma unroll
  for (int g = 0; g < FN; g++) {
    const int n = T.nt * NT + (2 * g + wn) * 32 + l32;
    const int t = n / No;
    Gs[g] = n < T.ncols ? Gc + (int64_t)(T.slot0 + t * T.slot_step) * P.W3 +
                              g_col(n - t * No)
                        : nullptr;
  }
#pragma unroll
  for (int f = 0; f < FM; f++)
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const int m = T.mt * MT + (2 * f + wm) * 32 + 8 * (r >> 2) + 4 * kh + (r & 3);
      if (m >= N2) continue;
      const uint32_t o = g_row(P.lay, m);
#pragma unroll
      for (int g = 0; g < FN; g++)
        if (Gs[g]) Gs[g][o] = acc[f][g][r];
    }
}

// Dispatch on the wave's occupied column fragments, n <= FN of them.
template <int TM, int TN, int FM, int FN>
__device__ __forceinline__ void tri_columns(const TriParams &P, const TileWork &T,
                                            int No, int lane, int wm, int wn,
                                            int n) {
  if constexpr (FN > 1) {
    if (n < FN) {
      tri_columns<TM, TN, FM, FN - 1>(P, T, No, lane, wm, wn, n);
      return;
    }
  }
  tri_wave<TM, TN, FM, FN>(P, T, No, lane, wm, wn);
}

// Dispatch on the wave's occupied row fragments, m <= FM of them.
template <int TM, int TN, int FM, int FN>
__device__ __forceinline__ void tri_rows(const TriParams &P, const TileWork &T, int No,
                                         int lane, int wm, int wn, int m,
                                         int n) {
  if constexpr (FM > 1) {
    if (m < FM) {
      tri_rows<TM, TN, FM - 1, FN>(P, T, No, lane, wm, wn, m, n);
      return;
    }
  }
  tri_columns<TM, TN, FM, FN>(P, T, No, lane, wm, wn, n);
}

template <int FM, int FN>
__global__ __launch_bounds__(256) void doubles_tri_kernel(TriParams P) {
  const int No = (int)P.No;
  TileWork T;
  if (!tile_work(P.win, (uint64_t)P.Nv, No, 64 * FN, T)) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  // edge tiles run the instance of their occupied fragments (FP64 kernel)
  const int m = occupied(P.N2 - (int64_t)T.mt * 64 * FM, wm, 2, 32, 2 * FM);
  const int n = occupied(T.ncols - (int64_t)T.nt * 64 * FN, wn, 2, 32, 2 * FN);
  if (!m || !n) return;
  tri_rows<FM, FN, FM, FN>(P, T, No, lane, wm, wn, m, n);
}

}  // namespace

hipError_t launch_doubles_tri(const DevSystem &s, const BatchArgs &b,
                              bool use_j, float *G, int tile, hipStream_t st) {
  TriParams P;
  const TriOp &H = use_j ? s.tH3J : s.tH3;
  P.T3 = (const __bf16 *)s.tT3.p;
  P.T3s = (const __bf16 *)s.tT3.sw;
  P.H3 = (const __bf16 *)H.p;
  P.H3s = (const __bf16 *)H.sw;
  P.V3 = (const __bf16 *)(use_j ? s.tV3J.p : s.tV3.p);
  P.T2N = (const __bf16 *)s.tT2N.p;
  P.T2TN = (const __bf16 *)s.tT2TN.p;
  P.win = b;
  P.G = G;
  P.No = s.No;
  P.Nv = s.Nv;
  P.Kv = s.Kv;
  P.Ko = s.Ko;
  P.N2 = s.No * s.No;
  P.N2p = pad32(P.N2);
  P.lay = g_layout(s.No);
  P.W3 = g_elems(s.No);
  P.slots = b.slots;
  tile = pick_t32_tile(tile, s.No, std::max(b.ea, std::max(b.eb, b.ec)));
  const int FM = t32_fm(tile), FN = t32_fn(tile);
  const int64_t grid = doubles_grid(P.win, s.No, 64 * FM, 64 * FN);
  if (grid <= 0) return hipSuccess;
  if (grid > MAX_GRID) return hipErrorInvalidConfiguration;
#define LAUNCH(A, B)                                                         \
  if (FM == A && FN == B)                                                    \
    hipLaunchKernelGGL((doubles_tri_kernel<A, B>), dim3((unsigned)grid),     \
                       dim3(256), 0, st, P);
  LAUNCH(2, 2) LAUNCH(2, 3) LAUNCH(3, 2) LAUNCH(2, 4) LAUNCH(3, 3)
  LAUNCH(2, 5) LAUNCH(3, 5) LAUNCH(4, 4) LAUNCH(3, 4) LAUNCH(4, 3)
#undef LAUNCH
  return hipGetLastError();
}

}  // namespace atrip_amd
