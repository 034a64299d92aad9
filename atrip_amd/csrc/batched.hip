// Batched form of the (T) hot path: the tuples of many small resident
// systems of uneven No/Nv in one persistent launch.
//
// A work item is one window (block triple of edge nb) of one system.  A
// workgroup takes work items from a device counter in the dispatch order the
// host scheduler chose, and does everything for its window itself:
//   1. the doubles contractions (reference src/atrip/Equations.cxx:455-728,
//      regrouped into the three classes w, v, u of the FP64 doubles kernel),
//      class by class, over the columns of valid tuples only.  Each of the four
//      waves takes wave tiles of (16*FM) x (16*FN) outputs (FM, FN per system,
//      from the tuner; a tile at the edge takes the variant of the fragments
//      it holds), runs the FP64 MFMA K loop with operands straight from
//      global memory and adds the tile into W of the window's tuples in the
//      workgroup's own scratch (class w stores, v and u add after a barrier,
//      so W sums the classes in the fixed order (w + v) + u);
//   2. singles and energy of each tuple of the window (reference
//      src/atrip/Equations.cxx:101-238 and :387-426, selection as
//      src/atrip/Atrip.cxx:636-670), one wave per tuple over the i>=j>=k
//      points, reduced by a fixed butterfly;
//   3. a compensated sum of the window's tuple energies in slot order.
// Nothing depends on which workgroup runs which window or on the other
// systems of the launch, so a system's energy is the same alone and in any
// mix.  No workgroup waits on another; the loop ends when the counter passes
// the number of work items.
//
// Bound by FP64 MFMA issue at the clock the chip holds under it: the matrix
// units are busy 64 % of the time at No=12, Nv=120 (window edge 4, 3x3 tiles,
// 43 TFLOP/s), the rest is what two waves a SIMD do not hide of a wave's setup,
// W updates and energies.  Three waves a SIMD raise it to 68 % at a lower clock
// and the same rate.  Before operands were swapped for w and v, W added to by
// atomics, empty columns left out and a tile's place kept in scalar registers
// it was 54 % and 37 TFLOP/s; 64 systems of No 4..16, Nv 20..120: 329 ms then,
// 287 ms now.  Task lists per XCD change nothing (L2 hit rates of operands do
// not bound it).
#include "doubles_common.hpp"

namespace atrip_amd {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef double d2 __attribute__((ext_vector_type(2)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

// correction-MFMA operands from four hi and four lo values of one kappa
// range: A [bf16(hi), lo], B [lo, bf16(hi)] (as the plain split kernel)
__device__ inline bf8 corr_a(f4 h, bf4 l) {
  const bf4 b = __builtin_convertvector(h, bf4);
  return __builtin_shufflevector(b, l, 0, 1, 2, 3, 4, 5, 6, 7);
}
__device__ inline bf8 corr_b(f4 h, bf4 l) {
  const bf4 b = __builtin_convertvector(h, bf4);
  return __builtin_shufflevector(l, b, 0, 1, 2, 3, 4, 5, 6, 7);
}

__device__ inline double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// n / d for 0 <= n < 2^16, 0 < d <= 64, from r = 1 / d: the quotient of n + 1/2
// is at least 1 / 128 away from a whole number, far beyond the error of the
// two FP32 operations, so the integer part is exact.
__device__ __forceinline__ int small_div(int n, float r) {
  return (int)(((float)n + 0.5f) * r);
}

// One A-pair of a class in a window.  The valid third indices of a pair are
// consecutive, y0 .. y0 + ncols / No - 1, and only their columns exist:
// column n is index n % No of third index y0 + n / No, of the window slot
// slot0 + (n / No) step.
struct Sub {
  int32_t x1, x2, y0;  // w (a,b), v (a,c), u (b,c); first valid third index
  int ncols, slot0, step;
};
__device__ __forceinline__ Sub sub_work(const BSys &S, const BTask &T, int cl,
                                        int o1, int o2) {
  const int nb = S.nb, Nv = (int)S.Nv;
  const int a0 = T.al * nb, b0 = T.be * nb, c0 = T.ga * nb;
  Sub u;
  int hi;
  bool ok;
  if (cl == 0) {
    u.x1 = a0 + o1; u.x2 = b0 + o2;
    u.y0 = max(c0, u.x2 + (u.x1 == u.x2));
    hi = min(c0 + nb, Nv);
    ok = u.x1 <= u.x2 && u.x2 < Nv;
    u.step = 1;
    u.slot0 = (o1 * nb + o2) * nb + (u.y0 - c0);
  } else if (cl == 1) {
    u.x1 = a0 + o1; u.x2 = c0 + o2;
    u.y0 = max(b0, u.x1);
    hi = min(b0 + nb, u.x2 + 1);
    ok = u.x1 < u.x2 && u.x2 < Nv;
    u.step = nb;
    u.slot0 = (o1 * nb + (u.y0 - b0)) * nb + o2;
  } else {
    u.x1 = b0 + o1; u.x2 = c0 + o2;
    u.y0 = a0;
    hi = min(a0 + nb, u.x1 + (u.x1 != u.x2));
    ok = u.x1 <= u.x2 && u.x2 < Nv;
    u.step = nb * nb;
    u.slot0 = o1 * nb + o2;
  }
  u.ncols = ok && hi > u.y0 ? (hi - u.y0) * (int)S.No : 0;
  return u;
}

// A lane's columns and rows of a wave tile (fragment f / g: row or column
// 16 f + lane % 16 behind the tile's first), clamped into the GEMM.
template <int FM, int FN>
struct TileAt {
  // column: index of the third index behind y0 in the upper, column index in
  // the lower half; row: p in the upper, q in the lower half
  uint32_t col[FN], row[FM];
  __device__ __forceinline__ void set(int no, const Sub &u, int r0, int c0,
                                      int l16) {
    const float r = 1.0f / (float)no;
#pragma unroll
    for (int g = 0; g < FN; g++) {
      const int n = min((c0 + g) * 16 + l16, u.ncols - 1), t = small_div(n, r);
      col[g] = (uint32_t)t << 16 | (uint32_t)(n - t * no);
    }
#pragma unroll
    for (int f = 0; f < FM; f++) {
      const int m = min((r0 + f) * 16 + l16, no * no - 1), q = small_div(m, r);
      row[f] = (uint32_t)(m - q * no) << 16 | (uint32_t)q;
    }
  }
};

// Adds one wave tile into W (order i + No j + No^2 k).  W's offset is a row
// part plus a column part: class w m + No^2 r, class v p + No^2 q + No r, class
// u No m + r.  The lanes of a fragment run along the index that is consecutive
// in W: the rows for w and v (SW, the MFMA's operands swapped: the fragment
// then comes out transposed and nothing passes through LDS), the column
// index for u.  Class w stores; v and u add with atomics that return nothing
// and are carried out in L2, so a wave never waits for old values: with loads
// and stores instead a 3x3 tile at No=12, Nv=120 spent 22 of its 101 k cycles
// here.  Every element receives one contribution per class and the
// classes are separated by barriers, so the sum is (w + v) + u whatever the
// order of the tiles.
// OUT = 8: FP64 MFMA layout D[i][j] in lane j + 16 (i % 4), register i / 4;
// OUT = 4: FP32 MFMA layout D[i][j] in lane j + 16 (i / 4), register i % 4.
template <bool SW, int OUT, int FM, int FN, typename V4>
__device__ __forceinline__ void store_tile(const V4 (&acc)[FM][FN],
                                           const TileAt<FM, FN> &at,
                                           const Sub &u, int cl, int r0, int c0,
                                           int no, double *Gwin, int lane) {
  const int kk = lane >> 4, l16 = lane & 15, n2 = no * no;
  int wcol[FN], wrow[FM];
#pragma unroll
  for (int g = 0; g < FN; g++) {
    const int t = at.col[g] >> 16, rr = at.col[g] & 0xffff;
    wcol[g] = (c0 + g) * 16 + l16 < u.ncols
                  ? (u.slot0 + t * u.step) * n2 * no +
                        rr * (cl == 0 ? n2 : cl == 1 ? no : 1)
                  : -1;
  }
  if (SW) {
#pragma unroll
    for (int f = 0; f < FM; f++) {
      const int p = at.row[f] >> 16, q = at.row[f] & 0xffff;
      wrow[f] = (r0 + f) * 16 + l16 < n2 ? p + (cl == 0 ? no : n2) * q : -1;
    }
  }
#pragma unroll
  for (int g = 0; g < FN; g++) {
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int i = OUT == 8 ? 4 * r + kk : 4 * kk + r;
      const int col = SW ? __shfl(wcol[g], i, 64) : wcol[g];
#pragma unroll
      for (int f = 0; f < FM; f++) {
        const int m = (r0 + f) * 16 + i;
        const int row = SW ? wrow[f] : m < n2 ? no * m : -1;
        if (row >= 0 && col >= 0) {
          const double v = (double)acc[f][g][r];
          if (cl > 0)
            unsafeAtomicAdd(Gwin + row + col, v);
          else
            Gwin[row + col] = v;
        }
      }
    }
  }
}

// One wave tile: row fragments r0 .. of the No^2 (p,q) rows, column fragments
// c0 .. of an A-pair's columns.  W of window slot s sits at Gwin + s*No^3 in the
// order i + No j + No^2 k.
template <bool SW, int FM, int FN>
__device__ __forceinline__ void wave_tile(const BSys &S, const Sub &u, int cl,
                                          int r0, int c0, double *Gwin,
                                          int lane) {
  const int64_t No = S.No, Nv = S.Nv, N2 = No * No, Kv = S.Kv, Ko = S.Ko;
  const int kk = lane >> 4, l16 = lane & 15;
  TileAt<FM, FN> at;
  at.set((int)No, u, r0, c0, l16);

  d4 acc[FM][FN];
#pragma unroll
  for (int f = 0; f < FM; f++)
#pragma unroll
    for (int g = 0; g < FN; g++) acc[f][g] = d4{0.0, 0.0, 0.0, 0.0};
  uint32_t ao[FM], bo[FN];  // byte offsets from the uniform bases ap, bp
  d2 a0[FM], b0[FN], a1[FM], b1[FN];
#define LOAD(AV, BV, C)                                                 \
  {                                                                     \
    const char *ac_ = ap + (int64_t)1024 * (C);                         \
    const char *bc_ = bp + (int64_t)1024 * (C);                         \
    _Pragma("unroll") for (int f = 0; f < FM; f++) AV[f] =              \
        *(const d2 *)(ac_ + ao[f]);                                     \
    _Pragma("unroll") for (int g = 0; g < FN; g++) BV[g] =              \
        *(const d2 *)(bc_ + bo[g]);                                     \
    __builtin_amdgcn_sched_barrier(0);                                  \
  }
#define COMPUTE(AV, BV)                                                   \
  {                                                                       \
    _Pragma("unroll") for (int s = 0; s < 2; s++)                         \
        _Pragma("unroll") for (int f = 0; f < FM; f++)                    \
            _Pragma("unroll") for (int g = 0; g < FN; g++) acc[f][g] =    \
                __builtin_amdgcn_mfma_f64_16x16x4f64(                     \
                    SW ? BV[g][s] : AV[f][s], SW ? AV[f][s] : BV[g][s],   \
                    acc[f][g], 0, 0, 0);                                  \
  }
  // segments: 0 T3[x1] straight, 1 T3[x2] swapped, 2 H3[x2] straight,
  //           3 H3[x1] swapped, in 8-deep chunks (one operand tile each).
  // Each segment has its own two-stage pipeline: one pipeline through all
  // four keeps the next segment's pointers live as well and costs the kernel
  // its second wave per SIMD.
  const int64_t N2p = pad16(N2);
#pragma unroll 1
  for (int sg = 0; sg < 4; sg++) {
    const int64_t K_ = sg < 2 ? Kv : Ko;
    const double *As = sg < 2 ? S.T3s : S.H3s;  // null: the straight array
    const bool sw = (sg & 1) && As;
    const double *Ab = sw ? As : sg < 2 ? S.T3 : S.H3;
    const int64_t xr = (sg == 0 || sg == 3 ? u.x1 : u.x2) * N2p;
    const char *ap = (const char *)(Ab + f64_row(xr, K_));
#pragma unroll
    for (int f = 0; f < FM; f++) {
      const uint32_t p = at.row[f] >> 16, q = at.row[f] & 0xffff;
      const uint32_t m = (sg & 1) && !sw ? q + (uint32_t)No * p : p + (uint32_t)No * q;
      ao[f] = 8 * (uint32_t)f64_row(m, K_) + 256 * kk;
    }
    // the columns' rows lie within seven third indices of the first one's, so
    // 32 bits hold the offsets for any system that fits the device
    int which;
    const int64_t row0 = b_row(cl, sg, u.x1, u.x2, u.y0, 0, Nv, No, which);
    const int64_t rstep =
        b_row(cl, sg, u.x1, u.x2, u.y0 + 1, 0, Nv, No, which) - row0;
    const char *bp =
        (const char *)((which == 0 ? S.V3 : which == 1 ? S.T2N : S.T2TN) +
                       f64_row(row0 & ~15LL, K_));
#pragma unroll
    for (int g = 0; g < FN; g++) {
      const uint32_t r = (uint32_t)(row0 & 15) +
                         (at.col[g] >> 16) * (uint32_t)rstep +
                         (at.col[g] & 0xffff);
      bo[g] = (r >> 4) * (128 * (uint32_t)K_) + 16 * (r & 15) + 256 * kk;
    }
    const int last = (int)(((sg < 2 ? Nv : No) + 7) / 8) - 1;
    LOAD(a0, b0, 0);
    for (int c = 0;; c += 2) {
      LOAD(a1, b1, c + 1 < last ? c + 1 : last);
      COMPUTE(a0, b0);
      if (c + 1 > last) break;
      LOAD(a0, b0, c + 2 < last ? c + 2 : last);
      COMPUTE(a1, b1);
      if (c + 2 > last) break;
    }
  }
#undef LOAD
#undef COMPUTE
  store_tile<SW, 8>(acc, at, u, cl, r0, c0, (int)No, Gwin, lane);
}

// The same wave tile with FP32 products (mixed forms): hi*hi on
// v_mfma_f32_16x16x4f32 and, when CORR, hi*lo + lo*hi in one
// v_mfma_f32_16x16x32_bf16 per 16-deep chunk (each lane group pairs
// [bf16(hi_a), lo_a] with [lo_b, bf16(hi_b)] over its four kappa), FP32
// accumulation; the tile is widened to FP64 when it is added into W.
template <bool SW, int FM, int FN, bool CORR>
__device__ __forceinline__ void wave_tile_split(const BSys &S, const BSplit &X,
                                                const Sub &u, int cl, int r0,
                                                int c0, double *Gwin, int lane) {
  const int64_t No = S.No, Nv = S.Nv, N2 = No * No, Kv = S.Kv, Ko = S.Ko;
  const int kk = lane >> 4, l16 = lane & 15;
  TileAt<FM, FN> at;
  at.set((int)No, u, r0, c0, l16);
  f4 acc[FM][FN];
#pragma unroll
  for (int f = 0; f < FM; f++)
#pragma unroll
    for (int g = 0; g < FN; g++) acc[f][g] = f4{0.f, 0.f, 0.f, 0.f};
  uint32_t ao[FM], bo[FN];  // element offsets from the uniform bases
  f4 ah0[FM], bh0[FN], ah1[FM], bh1[FN];
  bf4 ac0[FM], bc0[FN], ac1[FM], bc1[FN];
#define LOAD(AH, AC, BH, BC, KOFF)                                          \
  {                                                                         \
    _Pragma("unroll") for (int f = 0; f < FM; f++) {                        \
      AH[f] = *(const f4 *)(aph + (KOFF) + ao[f]);                          \
      if constexpr (CORR) AC[f] = *(const bf4 *)(apc + (KOFF) + ao[f]);     \
    }                                                                       \
    _Pragma("unroll") for (int g = 0; g < FN; g++) {                        \
      BH[g] = *(const f4 *)(bph + (KOFF) + bo[g]);                          \
      if constexpr (CORR) BC[g] = *(const bf4 *)(bpc + (KOFF) + bo[g]);     \
    }                                                                       \
    __builtin_amdgcn_sched_barrier(0);                                      \
  }
#define COMPUTE(AH, AC, BH, BC)                                             \
  {                                                                         \
    _Pragma("unroll") for (int s = 0; s < 4; s++)                           \
        _Pragma("unroll") for (int f = 0; f < FM; f++)                      \
            _Pragma("unroll") for (int g = 0; g < FN; g++) acc[f][g] =      \
                __builtin_amdgcn_mfma_f32_16x16x4f32(                       \
                    SW ? BH[g][s] : AH[f][s], SW ? AH[f][s] : BH[g][s],     \
                    acc[f][g], 0, 0, 0);                                    \
    if constexpr (CORR) {                                                   \
      bf8 ca_[FM], cb_[FN];                                                 \
      _Pragma("unroll") for (int f = 0; f < FM; f++) ca_[f] =               \
          corr_a(AH[f], AC[f]);                                             \
      _Pragma("unroll") for (int g = 0; g < FN; g++) cb_[g] =               \
          corr_b(BH[g], BC[g]);                                             \
      _Pragma("unroll") for (int f = 0; f < FM; f++)                        \
          _Pragma("unroll") for (int g = 0; g < FN; g++) acc[f][g] =        \
              __builtin_amdgcn_mfma_f32_16x16x32_bf16(                      \
                  SW ? cb_[g] : ca_[f], SW ? ca_[f] : cb_[g], acc[f][g], 0, \
                  0, 0);                                                    \
    }                                                                       \
  }
  // per-segment pipelines: one pipeline across the segments (as in
  // wave_tile) keeps more pointers live and costs this tile its second wave
  // per SIMD
#pragma unroll 1
  for (int sg = 0; sg < 4; sg++) {
    const int64_t K_ = sg < 2 ? Kv : Ko;
    const int64_t abase = ((sg == 0 || sg == 3) ? u.x1 : u.x2) * N2 * K_;
    const float *aph = (sg < 2 ? X.T3h : X.H3h) + abase;
    const __bf16 *apc = (const __bf16 *)(sg < 2 ? X.T3l : X.H3l) + abase;
#pragma unroll
    for (int f = 0; f < FM; f++) {
      const uint32_t p = at.row[f] >> 16, q = at.row[f] & 0xffff;
      ao[f] = (sg & 1 ? q + (uint32_t)No * p : p + (uint32_t)No * q) * (uint32_t)K_ + 4 * kk;
    }
    int which;
    const int64_t row0 = b_row(cl, sg, u.x1, u.x2, u.y0, 0, Nv, No, which);
    const int64_t rstep =
        b_row(cl, sg, u.x1, u.x2, u.y0 + 1, 0, Nv, No, which) - row0;
    const float *bph =
        (which == 0 ? X.V3h : which == 1 ? X.T2Nh : X.T2TNh) + row0 * K_;
    const __bf16 *bpc =
        (const __bf16 *)(which == 0 ? X.V3l : which == 1 ? X.T2Nl : X.T2TNl) +
        row0 * K_;
#pragma unroll
    for (int g = 0; g < FN; g++)
      bo[g] = ((at.col[g] >> 16) * (uint32_t)rstep + (at.col[g] & 0xffff)) *
                  (uint32_t)K_ +
              4 * kk;
    const int64_t last = K_ - KCHUNK;
    LOAD(ah0, ac0, bh0, bc0, 0);
    for (int64_t k0 = 0;; k0 += 2 * KCHUNK) {
      LOAD(ah1, ac1, bh1, bc1, k0 + KCHUNK < last ? k0 + KCHUNK : last);
      COMPUTE(ah0, ac0, bh0, bc0);
      if (k0 + KCHUNK > last) break;
      LOAD(ah0, ac0, bh0, bc0, k0 + 2 * KCHUNK < last ? k0 + 2 * KCHUNK : last);
      COMPUTE(ah1, ac1, bh1, bc1);
      if (k0 + 2 * KCHUNK > last) break;
    }
  }
#undef LOAD
#undef COMPUTE

  store_tile<SW, 4>(acc, at, u, cl, r0, c0, (int)No, Gwin, lane);
}

// Energy of tuple (a,b,c) from its W (order i + No j + No^2 k), by one
// wave; tA/tB/tC hold Tai at (a,x), (b,x), (c,x).
__device__ __forceinline__ double tuple_energy(const BSys &S, const double *W, int64_t a,
                               int64_t b, int64_t c, const double *tA,
                               const double *tB, const double *tC, int lane) {
  const int64_t No = S.No, Nv = S.Nv, N2 = No * No;
  int distinct = 0;
  if (a == b) distinct++;
  if (b == c) distinct--;
  const double epsabc = (S.ea[a] + S.ea[b]) + S.ea[c];
  const double *Vbc = S.VHH + (b + Nv * c) * N2;
  const double *Vac = S.VHH + (a + Nv * c) * N2;
  const double *Vab = S.VHH + (a + Nv * b) * N2;
  const int no = (int)No;
  auto Wv = [&](int x, int y, int z) { return W[x + no * (y + no * z)]; };
  // singles at a permutation (x,y,z): t_a[x] V^bc_yz + t_b[y] V^ac_xz
  // + t_c[z] V^ab_xy
  auto Z = [&](double wv, int x, int y, int z) {
    double zz = wv + tA[x] * Vbc[y + no * z];
    zz = zz + tB[y] * Vac[x + no * z];
    zz = zz + tC[z] * Vab[x + no * y];
    return zz;
  };
  double acc = 0.0;
#pragma unroll 1
  for (int64_t pt = lane; pt < S.npoints; pt += 64) {
    const uint32_t pk = S.points[pt];
    const int i = pk & 1023, j = (pk >> 10) & 1023, k = pk >> 20;
    const double facjk = j == k ? 0.5 : 1.0;
    const double facij = i == j ? 0.5 : 1.0;
    const double eijk = (S.ei[i] + S.ei[j]) + S.ei[k];
    const double denominator = epsabc - eijk;
    if (distinct == 0) {
      const double A = Wv(i, j, k), B = Wv(i, k, j), C = Wv(j, i, k),
                   D = Wv(j, k, i), E = Wv(k, i, j), F = Wv(k, j, i);
      const double U = Z(A, i, j, k), V = Z(B, i, k, j), W_ = Z(C, j, i, k),
                   X = Z(D, j, k, i), Y = Z(E, k, i, j), Zz = Z(F, k, j, i);
      const double UXY = U + (X + Y), VWZ = V + (W_ + Zz);
      const double first =
          A * U + (B * V + (C * W_ + (D * X + (E * Y + F * Zz))));
      const double second = (UXY - 2.0 * VWZ) * (A + (D + E));
      const double third = (VWZ - 2.0 * UXY) * (B + (C + F));
      const double value = 3.0 * first + (second + third);
      acc += ((2.0 * value) / denominator) * (facjk * facij);
    } else {
      const double A = Wv(i, j, k), B = Wv(j, k, i), C = Wv(k, i, j);
      const double U = Z(A, i, j, k), V = Z(B, j, k, i), W_ = Z(C, k, i, j);
      const double UVW = U + (V + W_);
      const double value =
          3.0 * ((A * U + B * V) + C * W_) - (A + (B + C)) * UVW;
      acc += ((2.0 * value) / denominator) * (facjk * facij);
    }
  }
  return wave_sum(acc);
}

constexpr int BMAX_NO = 64;  // singles tables in LDS

// Load a descriptor the whole workgroup shares and make every 32-bit word
// wave-uniform, so it lives in scalar registers.
template <typename T>
__device__ __forceinline__ T uniform_load(const T *p) {
  static_assert(sizeof(T) % 4 == 0, "descriptor size");
  T v = *p;
  uint32_t w[sizeof(T) / 4];
  __builtin_memcpy(w, &v, sizeof(T));
#pragma unroll
  for (unsigned i = 0; i < sizeof(T) / 4; i++)
    w[i] = __builtin_amdgcn_readfirstlane(w[i]);
  __builtin_memcpy(&v, w, sizeof(T));
  return v;
}

template <int PREC>
__global__ __launch_bounds__(256, 2) void batched_kernel(BatchedLaunch P) {
  __shared__ int task_sh;
  __shared__ double etup[512];
  __shared__ double tsing[4][3][BMAX_NO];
  const int tid = threadIdx.x, lane = tid & 63;
  // uniform, so that a wave tile's place is worked out in scalar registers
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  double *Gwin = P.scratch + (int64_t)blockIdx.x * P.scratch_stride;
#pragma unroll 1
  for (;;) {
    if (tid == 0) task_sh = (int)atomicAdd(P.counter, 1u);
    __syncthreads();
    // uniform: the work item's descriptors then load into scalar registers
    const int q = __builtin_amdgcn_readfirstlane(task_sh);
    __syncthreads();
    if (q >= P.ntasks) break;
    const int tix = uniform_load(P.order + q);
    const BTask T = uniform_load(P.tasks + tix);
    const BSys S = uniform_load(P.sys + T.sys);
    BSplit X{};
    if constexpr (PREC != ATRIP_FP64) X = uniform_load(P.split + T.sys);
    const int nb = S.nb, nb3 = nb * nb * nb;
    const int64_t No = S.No, N2 = No * No;
    const int fm = bfm(S.tile), fn = bfn(S.tile);
    const int rfrags = (int)((N2 + 15) / 16);
    const int mtiles = (rfrags + fm - 1) / fm;
    const int ntiles = (int)((nb * No + 16 * fn - 1) / (16 * fn));
    const int nsub = nb * nb * mtiles * ntiles;

#pragma unroll 1
    for (int cl = 0; cl < 3; cl++) {
#pragma unroll 1
      for (int q = wave; q < nsub; q += 4) {
        const int nt = q % ntiles, mt = (q / ntiles) % mtiles;
        const int pair = q / (ntiles * mtiles);
        const Sub u = sub_work(S, T, cl, pair / nb, pair % nb);
        const int r0 = mt * fm, c0 = nt * fn;
        const int nc = (u.ncols + 15) / 16 - c0;
        if (nc <= 0) continue;
        const int v = fitting_tile(S.tile, min(fm, rfrags - r0), min(fn, nc));
        // classes w and v with the MFMA's operands swapped (see store_tile)
        switch (v + (cl == 2 ? N_BTILES : 0)) {
#define TILE_CASE1(V, SW)                                                    \
  case V + (SW ? 0 : N_BTILES):                                              \
    if constexpr (PREC == ATRIP_FP64)                                        \
      wave_tile<SW, bfm(V), bfn(V)>(S, u, cl, r0, c0, Gwin, lane);           \
    else                                                                     \
      wave_tile_split<SW, bfm(V), bfn(V), PREC == ATRIP_SPLIT_FP32>(         \
          S, X, u, cl, r0, c0, Gwin, lane);                                  \
    break;
#define TILE_CASE(V) TILE_CASE1(V, true) TILE_CASE1(V, false)
          TILE_CASE(0)
          TILE_CASE(1)
          TILE_CASE(2)
          TILE_CASE(3)
          TILE_CASE(4)
          TILE_CASE(5)
          TILE_CASE(6)
          TILE_CASE(7)
          TILE_CASE(8)
          TILE_CASE(9)
#undef TILE_CASE
#undef TILE_CASE1
          default:
            break;
        }
      }
      // the class is in memory before the next adds to it
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
    }

    // energies, one tuple per wave, each wave through its own slots: the
    // singles table tsing[wave] is the wave's own, so its LDS writes need
    // only to complete before the same wave reads them
#pragma unroll 1
    for (int slot = wave; slot < nb3; slot += 4) {
      const int64_t a = (int64_t)T.al * nb + slot / (nb * nb);
      const int64_t b = (int64_t)T.be * nb + (slot / nb) % nb;
      const int64_t c = (int64_t)T.ga * nb + slot % nb;
      const bool ok = tuple_ok(S.Nv, a, b, c);
      double e = 0.0;
      if (ok) {
        if (lane < No) {
          tsing[wave][0][lane] = S.Tai[a + S.Nv * lane];
          tsing[wave][1][lane] = S.Tai[b + S.Nv * lane];
          tsing[wave][2][lane] = S.Tai[c + S.Nv * lane];
        }
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): LDS writes done
        __builtin_amdgcn_wave_barrier();
        e = tuple_energy(S, Gwin + (int64_t)slot * N2 * No, a, b, c,
                         tsing[wave][0], tsing[wave][1], tsing[wave][2],
                         lane);
        __builtin_amdgcn_wave_barrier();  // reads done before the next writes
      }
      if (lane == 0) etup[slot] = e;
    }
    __syncthreads();  // every slot's energy is in etup
    if (P.tuple_e)
      for (int s = tid; s < nb3; s += 256) P.tuple_e[T.tuple_off + s] = etup[s];
    if (tid == 0) {
      // Neumaier over the slots in order
      double sum = 0.0, comp = 0.0;
      for (int s = 0; s < nb3; s++) {
        const double x = etup[s];
        const double t = sum + x;
        comp += (fabs(sum) >= fabs(x)) ? (sum - t) + x : (x - t) + sum;
        sum = t;
      }
      P.task_e[2 * tix] = sum;
      P.task_e[2 * tix + 1] = comp;
    }
    // the next window overwrites W and etup only after the barriers at the
    // top of the loop
  }
}

}  // namespace

hipError_t launch_batched(const BatchedLaunch &L, hipStream_t st) {
  if (L.ntasks <= 0 || L.grid <= 0) return hipSuccess;
  if (L.precision == ATRIP_FP64)
    hipLaunchKernelGGL(batched_kernel<ATRIP_FP64>, dim3(L.grid), dim3(256), 0,
                       st, L);
  else if (L.precision == ATRIP_SPLIT_FP32)
    hipLaunchKernelGGL(batched_kernel<ATRIP_SPLIT_FP32>, dim3(L.grid),
                       dim3(256), 0, st, L);
  else if (L.precision == ATRIP_FP32)
    hipLaunchKernelGGL(batched_kernel<ATRIP_FP32>, dim3(L.grid), dim3(256), 0,
                       st, L);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

int batched_blocks_per_cu(int precision) {
  int n = 0;
  hipError_t e;
  if (precision == ATRIP_SPLIT_FP32)
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(
        &n, batched_kernel<ATRIP_SPLIT_FP32>, 256, 0);
  else if (precision == ATRIP_FP32)
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(
        &n, batched_kernel<ATRIP_FP32>, 256, 0);
  else
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(
        &n, batched_kernel<ATRIP_FP64>, 256, 0);
  if (e != hipSuccess) return 1;
  return n > 0 ? n : 1;
}

}  // namespace atrip_amd
