// Doubles contractions W(ijk) in split FP32 (the mixed-precision form).
//
// Same regrouped class GEMMs and tuple windows as the FP64 kernel
// (doubles_f64.hip).  Every operand x is held as hi = (float)x plus the
// residual lo = bf16(x - hi); a product is formed as
//     hi_a hi_b                      on v_mfma_f32_32x32x2_f32
//   + hi_a lo_b + lo_a hi_b          on two v_mfma_f32_32x32x16_bf16
// (the FP32 form drops the corrections: one FP32 product per product), all
// accumulating into the same FP32 accumulator.  Fragments are 32 rows
// (columns); for a K chunk of 16, lane l feeds row/column l % 32 at the 8
// consecutive kappa k0 + 8 (l / 32) + m: FP32 MFMA m (m < 8) takes kappa
// m of each half, and the bf16 MFMAs take all 8 (bf16(hi) made in
// registers from the hi already loaded, lo loaded): bf16(hi_a) . lo_b and
// lo_a . bf16(hi_b).  Per 32 x 32 block and chunk: 8 x 64 + 2 x 32 cycles,
// against 16 x 64 in FP64.  The corrections carry the part of each product
// below FP32's 24 bits (their own bf16 rounding is 2^-8 of an already
// 2^-24-small term).  The FP32 result of each class GEMM is stored as FP32
// (it carries no more bits) and widened to FP64 by the class-sum kernel;
// singles, the energy and all sums stay FP64 (energy.hip).
#include "doubles_common.hpp"

#ifndef ATRIP_SPLIT_CORR
#define ATRIP_SPLIT_CORR true
#define ATRIP_SPLIT_LAUNCH launch_doubles_split
#endif

namespace atrip_amd {
namespace {

typedef float f8 __attribute__((ext_vector_type(8)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

// A lane's 8 hi values and 8 lo values of a chunk.
struct SParts {
  f8 h;
  bf8 l;
};

struct SplitParams {
  // per operand family: hi (float) and lo (bf16), row-major [row][K]
  const float *T3h, *H3h, *V3h, *T2Nh, *T2TNh;
  const __bf16 *T3l, *H3l, *V3l, *T2Nl, *T2TNl;
  WindowArgs win;
  float *G;
  int64_t No, Nv, Kv, Ko, N2, W3, slots;
  GLayout lay;
};

// The FM x FN occupied fragments of one wave of a tile of 64 TM x 64 TN (the
// waves of each direction take the fragments in turn, as the FP64 kernel).
template <int TM, int TN, int FM, int FN, bool CORR>
__device__ __forceinline__ void split_wave(const SplitParams &P, const TileWork &T, int No,
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
  // A rows: straight (p + No q) and swapped (q + No p)
  int32_t rowS[FM], rowW[FM];
#pragma unroll
  for (int f = 0; f < FM; f++) {
    int m = T.mt * MT + (2 * f + wm) * 32 + l32;
    if (m >= N2) m = (int)N2 - 1;
    rowS[f] = m;
    rowW[f] = m / No + No * (m % No);
  }

  const int64_t Kv = P.Kv, Ko = P.Ko;
  const float *aph[FM], *bph[FN];
  const __bf16 *apc[FM], *bpc[FN];
#define SET_PTRS(SG)                                                          \
  {                                                                           \
    const int64_t K_ = (SG) < 2 ? Kv : Ko;                                    \
    const int64_t xa_ = ((SG) == 0 || (SG) == 3) ? T.x1 : T.x2;                   \
    const int64_t abase_ = xa_ * N2 * K_;                                     \
    const float *Ah_ = ((SG) < 2 ? P.T3h : P.H3h) + abase_;                   \
    const __bf16 *Al_ = ((SG) < 2 ? P.T3l : P.H3l) + abase_;                  \
    _Pragma("unroll") for (int f = 0; f < FM; f++) {                          \
      const int64_t r_ = (((SG)&1) ? rowW[f] : rowS[f]) * K_;                 \
      aph[f] = Ah_ + r_ + 8 * kh;                                             \
      apc[f] = Al_ + r_ + 8 * kh;                                             \
    }                                                                         \
    _Pragma("unroll") for (int g = 0; g < FN; g++) {                          \
      int wh_;                                                                \
      const int64_t c_ =                                                      \
          b_row(T.cl, (SG), T.x1, T.x2, cy[g], crr[g], Nv, No, wh_) * K_;     \
      const float *Bh_ = wh_ == 0 ? P.V3h : wh_ == 1 ? P.T2Nh : P.T2TNh;      \
      const __bf16 *Bl_ = wh_ == 0 ? P.V3l : wh_ == 1 ? P.T2Nl : P.T2TNl;     \
      bph[g] = Bh_ + c_ + 8 * kh;                                             \
      bpc[g] = Bl_ + c_ + 8 * kh;                                             \
    }                                                                         \
  }
#define LOAD(A, B, KOFF)                                                     \
  {                                                                          \
    _Pragma("unroll") for (int f = 0; f < FM; f++) {                         \
      A[f].h = *(const f8 *)(aph[f] + (KOFF));                               \
      if constexpr (CORR) A[f].l = *(const bf8 *)(apc[f] + (KOFF));         \
    }                                                                        \
    _Pragma("unroll") for (int g = 0; g < FN; g++) {                         \
      B[g].h = *(const f8 *)(bph[g] + (KOFF));                               \
      if constexpr (CORR) B[g].l = *(const bf8 *)(bpc[g] + (KOFF));         \
    }                                                                        \
    __builtin_amdgcn_sched_barrier(0);                                       \
  }
  // FP32 MFMA m over all blocks before m + 1 (consecutive MFMAs update
  // different accumulators), then the two correction MFMAs
#define COMPUTE(A, B)                                                        \
  {                                                                          \
    _Pragma("unroll") for (int m = 0; m < 8; m++)                            \
        _Pragma("unroll") for (int f = 0; f < FM; f++)                       \
            _Pragma("unroll") for (int g = 0; g < FN; g++) acc[f][g] =       \
                __builtin_amdgcn_mfma_f32_32x32x2f32(A[f].h[m], B[g].h[m],   \
                                                     acc[f][g], 0, 0, 0);    \
    if constexpr (CORR) {                                                    \
      bf8 ha_[FM], hb_[FN];                                                  \
      _Pragma("unroll") for (int f = 0; f < FM; f++) ha_[f] =                \
          __builtin_convertvector(A[f].h, bf8);                              \
      _Pragma("unroll") for (int g = 0; g < FN; g++) hb_[g] =                \
          __builtin_convertvector(B[g].h, bf8);                              \
      _Pragma("unroll") for (int f = 0; f < FM; f++)                         \
          _Pragma("unroll") for (int g = 0; g < FN; g++) acc[f][g] =         \
              __builtin_amdgcn_mfma_f32_32x32x16_bf16(ha_[f], B[g].l,        \
                                                      acc[f][g], 0, 0, 0);   \
      _Pragma("unroll") for (int f = 0; f < FM; f++)                         \
          _Pragma("unroll") for (int g = 0; g < FN; g++) acc[f][g] =         \
              __builtin_amdgcn_mfma_f32_32x32x16_bf16(A[f].l, hb_[g],        \
                                                      acc[f][g], 0, 0, 0);   \
    }                                                                        \
  }

  f16v acc[FM][FN];
#pragma unroll
  for (int f = 0; f < FM; f++)
#pragma unroll
    for (int g = 0; g < FN; g++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[f][g][r] = 0.f;

  // two operand sets in ping-pong: the loads of chunk c + 1 are in flight
  // behind the MFMAs of chunk c.  One pipeline runs through the four
  // segments: (sg, c) is the next chunk to load, and past a segment's end
  // the pointers move to the next segment's chunk 0 in place, so every
  // segment but the first starts with its first chunk in flight.  After the
  // last chunk the prefetch re-reads it (a load never used).
  static_assert(6 * (FM + FN) <= 63, "two chunks of loads must fit vmcnt");
  SParts a0[FM], b0[FN], a1[FM], b1[FN];
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
#undef COMPUTE

  // 32x32 FP32-output MFMAs: D[i][j] in lane j + 32 ((i / 4) % 2), register
  // 4 (i / 8) + i % 4
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
template <int TM, int TN, int FM, int FN, bool CORR>
__device__ __forceinline__ void split_columns(const SplitParams &P, const TileWork &T,
                                            int No, int lane, int wm, int wn,
                                            int n) {
  if constexpr (FN > 1) {
    if (n < FN) {
      split_columns<TM, TN, FM, FN - 1, CORR>(P, T, No, lane, wm, wn, n);
      return;
    }
  }
  split_wave<TM, TN, FM, FN, CORR>(P, T, No, lane, wm, wn);
}

// Dispatch on the wave's occupied row fragments, m <= FM of them.
template <int TM, int TN, int FM, int FN, bool CORR>
__device__ __forceinline__ void split_rows(const SplitParams &P, const TileWork &T, int No,
                                         int lane, int wm, int wn, int m,
                                         int n) {
  if constexpr (FM > 1) {
    if (m < FM) {
      split_rows<TM, TN, FM - 1, FN, CORR>(P, T, No, lane, wm, wn, m, n);
      return;
    }
  }
  split_columns<TM, TN, FM, FN, CORR>(P, T, No, lane, wm, wn, n);
}

template <int FM, int FN, bool CORR>
__global__ __launch_bounds__(256) void doubles_split_kernel(SplitParams P) {
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
  split_rows<FM, FN, FM, FN, CORR>(P, T, No, lane, wm, wn, m, n);
}

}  // namespace

// (compiled once per form, in parallel: doubles_fp32.hip includes this file)
hipError_t ATRIP_SPLIT_LAUNCH(const DevSystem &s, const BatchArgs &b,
                              bool use_j, float *G, int tile, hipStream_t st) {
  SplitParams P;
  const DevSystem::Split &V = use_j ? s.sV3J : s.sV3;
  const DevSystem::Split &H = use_j ? s.sH3J : s.sH3;
  P.T3h = s.sT3.h; P.H3h = H.h; P.V3h = V.h; P.T2Nh = s.sT2N.h;
  P.T2TNh = s.sT2TN.h;
  P.T3l = (const __bf16 *)s.sT3.l; P.H3l = (const __bf16 *)H.l;
  P.V3l = (const __bf16 *)V.l; P.T2Nl = (const __bf16 *)s.sT2N.l;
  P.T2TNl = (const __bf16 *)s.sT2TN.l;
  P.win = b;
  P.G = G;
  P.No = s.No;
  P.Nv = s.Nv;
  P.Kv = s.Kv;
  P.Ko = s.Ko;
  P.N2 = s.No * s.No;
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
    hipLaunchKernelGGL((doubles_split_kernel<A, B, ATRIP_SPLIT_CORR>),       \
                       dim3((unsigned)grid), dim3(256), 0, st, P);
  LAUNCH(2, 2) LAUNCH(2, 3) LAUNCH(3, 2) LAUNCH(2, 4) LAUNCH(3, 3)
  LAUNCH(2, 5) LAUNCH(3, 5) LAUNCH(4, 4) LAUNCH(3, 4) LAUNCH(4, 3)
#undef LAUNCH
  return hipGetLastError();
}

}  // namespace atrip_amd
