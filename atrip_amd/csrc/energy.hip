// Singles + energy epilogue of the (T) hot path, from the three class buffers
// the doubles kernels wrote (see internal.hpp for their layout; FP64, or FP32
// for the forms with FP32 or bf16 products).
//
// energy_fused_kernel (a workgroup per block triple of a tuple) and
// energy_small_kernel (small No: a wave or workgroup per tuple) sum the classes
// to W in FP64 in LDS, (w + v) + u, and form the energies there; W is never
// written to memory.  wsum_kernel and energy_kernel do it in two steps, W as
// 8x8x8 cubes in between (w_cube); complex systems take their class sums from
// the first.
//
// Z = W + singles is formed in registers (reference
// src/atrip/Equations.cxx:387-426, with Z copied from W as in
// src/atrip/Atrip.cxx:899-906), and the energy of the tuple follows
// get_energy_distinct / get_energy_same (src/atrip/Equations.cxx:101-238)
// selected as src/atrip/Atrip.cxx:636-670 does.  The i>=j>=k points are
// spread over the workgroup; each thread sums its points in a fixed order
// and a fixed shuffle/LDS tree combines the threads, so the per-tuple energy
// does not depend on which other tuples share the launch.
#include <type_traits>

#include "internal.hpp"

namespace atrip_amd {
namespace {

struct EnergyParams {
  const double *W, *WJ;  // W (and the (cT) pass's W) as cubes, [slot][W3]
  const double *Tai, *VHH, *ei, *ea;
  WindowArgs win;
  double *e_slot;
  int64_t No, Nv, N2, W3, nbk, slots;  // nbk: cubes per index, W3 = (8 nbk)^3
  double tai_sign;
};

__device__ inline double wave_sum(double v) {
  // fixed xor butterfly over the 64 lanes
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// Thread's pair of elements e = 2 tid, 2 tid + 1 of an 8^3 block in class
// order: class cls of W block (bx, by, bz); the pair runs along the class's
// own fastest index.  `at` is its offset in the slot's class buffer, pos the
// place of its first element in an LDS block x + CY y + CZ z and step that of
// the second after it, in0, in1 whether the elements exist (No: W edge).
struct PairAt {
  uint32_t at;
  int pos, step;
  bool in0, in1;
};
// (FULL: every block the caller reads lies inside the occupied range.)
template <int CY, int CZ, bool FULL>
__device__ __forceinline__ PairAt pair_at(int cls, int bx, int by, int bz,
                                          int nbk, int no, int tid) {
  const int e = 2 * tid, r = e & 7, p = (e >> 3) & 7, q = e >> 6;
  // (p, q, r) in W indices: w (x,y,z), v (x,z,y), u (y,z,x)
  const int bp = cls == 2 ? by : bx, bq = cls == 0 ? by : bz,
            br = cls == 0 ? bz : cls == 1 ? by : bx;
  const int x = cls == 2 ? r : p, y = cls == 0 ? q : cls == 1 ? r : p,
            z = cls == 0 ? r : q;
  PairAt a;
  const bool in = FULL || ((8 * bp + p < no) & (8 * bq + q < no));
  a.in0 = FULL || (in & (8 * br + r < no));
  a.in1 = FULL || (in & (8 * br + r + 1 < no));
  const uint32_t blk = (uint32_t)((bq * nbk + bp) * nbk + br) << 9;
  a.at = blk + (a.in0 ? (uint32_t)e : 0u);  // always inside the buffer
  a.pos = x + CY * y + CZ * z;
  a.step = cls == 0 ? CZ : cls == 1 ? CY : 1;
  return a;
}

// Class sums of one 8^3 block of W for every slot of the batch: out = (Aw +
// Av) + Au, written as cubes.
template <typename GT>
__global__ __launch_bounds__(256) void wsum_kernel(const GT *A, double *out,
                                                   int no, int64_t W3g,
                                                   int64_t slots, int nbk) {
  typedef GT g2 __attribute__((ext_vector_type(2)));
  constexpr int CZ = 69;
  __shared__ double br[7 * CZ + 64];
  const uint32_t n3 = (uint32_t)(nbk * nbk * nbk), bid = blockIdx.x;
  const int64_t slot = bid / n3;
  const int blk = (int)(bid - (uint32_t)slot * n3);
  const int bx = blk % nbk, by = (blk / nbk) % nbk, bz = blk / (nbk * nbk);
  const int tid = threadIdx.x;
  PairAt a[3];
  g2 v[3];
#pragma unroll
  for (int cls = 0; cls < 3; cls++) {
    a[cls] = pair_at<8, CZ, false>(cls, bx, by, bz, nbk, no, tid);
    v[cls] = *(const g2 *)(A + (cls * slots + slot) * W3g + a[cls].at);
  }
#pragma unroll
  for (int cls = 0; cls < 3; cls++) {
    const double v0 = a[cls].in0 ? (double)v[cls][0] : 0.0,
                 v1 = a[cls].in1 ? (double)v[cls][1] : 0.0;
    double *b0 = br + a[cls].pos, *b1 = b0 + a[cls].step;
    if (cls == 0) {
      *b0 = v0;
      *b1 = v1;
    } else {
      *b0 += v0;
      *b1 += v1;
    }
    __syncthreads();
  }
  double *o = out + slot * (int64_t)(512 * n3) +
              ((int64_t)((bz * nbk + by) * nbk + bx) << 9);
#pragma unroll
  for (int e = tid; e < 512; e += 256) o[e] = br[(e & 63) + CZ * (e >> 6)];
}

// Energy of one tuple per workgroup.  The i>=j>=k points are visited per
// block triple (B1>=B2>=B3) of edge 8: the (up to) six distinct cubes that
// hold W at the six index permutations of those points are copied into LDS
// with coalesced 4 KiB reads, then every point reads its twelve W/Z values
// from LDS.
// The orbit of block triple (B1, B2, B3) under the six index permutations
// (ijk ikj jik jki kij kji): base offsets cb[s] of its nc distinct cubes and
// the slot al[p] of the cube of each permutation.
__device__ __forceinline__ void orbit(int B1, int B2, int B3, int nbk,
                                      int (&cb)[6], int &nc, int (&al)[6]) {
  const int cx[6] = {B1, B1, B2, B2, B3, B3};
  const int cy[6] = {B2, B3, B1, B3, B1, B2};
  const int cz[6] = {B3, B2, B3, B1, B2, B1};
  nc = 0;
#pragma unroll
  for (int p = 0; p < 6; p++) {
    int q0 = p;
#pragma unroll
    for (int q = 0; q < p; q++)
      if (q0 == p && cx[q] == cx[p] && cy[q] == cy[p] && cz[q] == cz[p]) q0 = q;
    if (q0 == p) {
      al[p] = nc;
      cb[nc < 6 ? nc : 5] = ((cz[p] * nbk + cy[p]) * nbk + cx[p]) << 9;
      nc++;
    } else {
      al[p] = al[q0];
    }
  }
}

// A point's energy term from W at its permutations (A ijk, B ikj, C jik, D
// jki, E kij, F kji; three of them, ijk, jki, kij, when two of a, b, c are
// equal) and Z = W + singles there: get_energy_distinct / get_energy_same in
// the reference's expression order.
__device__ __forceinline__ double term_distinct(
    double A, double B, double C, double D, double E, double F, double U,
    double V, double W, double X, double Y, double Z, double denominator,
    double fac) {
  const double UXY = U + (X + Y), VWZ = V + (W + Z);
  const double first = A * U + (B * V + (C * W + (D * X + (E * Y + F * Z))));
  const double second = (UXY - 2.0 * VWZ) * (A + (D + E));
  const double third = (VWZ - 2.0 * UXY) * (B + (C + F));
  const double value = 3.0 * first + (second + third);
  return ((2.0 * value) / denominator) * fac;
}
__device__ __forceinline__ double term_same(double A, double B, double C,
                                            double U, double V, double W,
                                            double denominator, double fac) {
  const double UVW = U + (V + W);
  const double value = 3.0 * ((A * U + B * V) + C * W) - (A + (B + C)) * UVW;
  return ((2.0 * value) / denominator) * fac;
}

// Energy terms of the i>=j>=k points of block triple (B1, B2, B3) (edge 8)
// of one tuple, two points per thread, added to e_acc (and, with the (cT)
// W, to ect_acc).  The six permuted W cubes of the triple's orbit sit in
// LDS (cube[alias[p]] holds W at permutation p, element x + CY y + CZ z), as
// do the singles tables tA/tB/tC (Tai at (a,x), (b,x), (c,x), slot 8 * position
// + local index), the eps_i table sE and the V^bc, V^ac, V^ab 8x8 block pairs
// sV.  Z = W + singles (reference src/atrip/Equations.cxx:387-426) and the
// get_energy_distinct / get_energy_same formulas (:101-238) in the
// reference's expression order.
// sV holds the 8x8 V blocks of the triple, [slice][block pair][ly + 8 lz]:
// all nine ordered position pairs (V6 false) or only the six with two
// different positions (V6 true), the only ones a point reads, then with
// rows 9 apart (a point reads V at (j, i) and (k, i) too, lanes along i: rows
// 8 apart met in two banks).  ALL: every point of the triple is an ordered
// triple i > j > k inside the range.
constexpr int V6_BLOCK = 72;  // doubles of an 8 x 8 V block with rows 9 apart
template <bool HJ, int CY, int CZ, int CSZ, bool V6, bool ALL>
__device__ __forceinline__ void triple_points(
    int B1, int B2, int B3, int no, int distinct, double epsabc,
    const int (&alias)[6], const double (*cube)[CSZ], const double *cubeJ,
    const double *tA, const double *tB, const double *tC, const double *sE,
    const double *sV, int tid, double &e_acc, double &ect_acc) {
  auto vb = [](int v, int r, int s2, int ly, int lz) {
    return V6 ? (v * 6 + 2 * r + s2 - (s2 > r ? 1 : 0)) * V6_BLOCK + ly + 9 * lz
              : ((v * 3 + r) * 3 + s2) * 64 + ly + 8 * lz;
  };
  // both points of a thread in one body, so their LDS reads and FP64
  // chains interleave
#pragma unroll
  for (int pt = tid; pt < 512; pt += 256) {
    const int li = pt & 7, lj = (pt >> 3) & 7, lk = pt >> 6;
    const int i = B1 * 8 + li, j = B2 * 8 + lj, k = B3 * 8 + lk;
    if (!ALL && (i >= no || j >= no || k >= no || i < j || j < k)) continue;
    const double ei = sE[li], ej = sE[8 + lj], ek = sE[16 + lk];
    const double facjk = !ALL && j == k ? 0.5 : 1.0;
    const double facij = !ALL && i == j ? 0.5 : 1.0;
    const double eijk = (ei + ej) + ek;
    const double denominator = epsabc - eijk;
    // local offsets of the permutations inside their cubes
    const int o_ijk = li + CY * lj + CZ * lk, o_ikj = li + CY * lk + CZ * lj,
              o_jik = lj + CY * li + CZ * lk, o_jki = lj + CY * lk + CZ * li,
              o_kij = lk + CY * li + CZ * lj, o_kji = lk + CY * lj + CZ * li;
    // singles at a permutation (x,y,z): t_a[x] V^bc_yz + t_b[y] V^ac_xz
    // + t_c[z] V^ab_xy; slot s = 8 * position + local index (position 0:
    // i, 1: j, 2: k)
    auto Z = [&](double wv, int sx, int sy, int sz) {
      const int px = sx >> 3, py = sy >> 3, pz = sz >> 3;
      const int lx = sx & 7, ly = sy & 7, lz = sz & 7;
      double zz = wv + tA[sx] * sV[vb(0, py, pz, ly, lz)];
      zz = zz + tB[sy] * sV[vb(1, px, pz, lx, lz)];
      zz = zz + tC[sz] * sV[vb(2, px, py, lx, ly)];
      return zz;
    };
    auto J = [&](int p, int o) { return cubeJ[alias[p] * CSZ + o]; };
    const int si = li, sj = 8 + lj, sk = 16 + lk;
    if (distinct == 0) {
      const double A = cube[alias[0]][o_ijk], B = cube[alias[1]][o_ikj],
                   C = cube[alias[2]][o_jik], D = cube[alias[3]][o_jki],
                   E = cube[alias[4]][o_kij], F = cube[alias[5]][o_kji];
      const double U = Z(A, si, sj, sk), V = Z(B, si, sk, sj),
                   W = Z(C, sj, si, sk), X = Z(D, sj, sk, si),
                   Y = Z(E, sk, si, sj), Zz = Z(F, sk, sj, si);
      e_acc += term_distinct(A, B, C, D, E, F, U, V, W, X, Y, Zz, denominator,
                             facjk * facij);
      if constexpr (HJ)
        ect_acc += term_distinct(J(0, o_ijk), J(1, o_ikj), J(2, o_jik),
                                 J(3, o_jki), J(4, o_kij), J(5, o_kji), U, V, W,
                                 X, Y, Zz, denominator, facjk * facij);
    } else {
      const double A = cube[alias[0]][o_ijk], B = cube[alias[3]][o_jki],
                   C = cube[alias[4]][o_kij];
      const double U = Z(A, si, sj, sk), V = Z(B, sj, sk, si),
                   W = Z(C, sk, si, sj);
      e_acc += term_same(A, B, C, U, V, W, denominator, facjk * facij);
      if constexpr (HJ)
        ect_acc += term_same(J(0, o_ijk), J(3, o_jki), J(4, o_kij), U, V, W,
                             denominator, facjk * facij);
    }
  }
}

template <bool HJ>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 8)))
void energy_kernel(EnergyParams P) {
  const int64_t gslot = blockIdx.x;
  const int64_t No = P.No, Nv = P.Nv, N2 = P.N2;
  int64_t a, b, c;
  if (!slot_tuple(P.win, (uint64_t)Nv, blockIdx.x, a, b, c)) {
    if (threadIdx.x == 0) {
      P.e_slot[2 * gslot] = 0.0;
      P.e_slot[2 * gslot + 1] = 0.0;
    }
    return;
  }
  constexpr bool have_j = HJ;

  // cube element x + 8 y + 64 z at x + 8 y + CZ z: the six permutation
  // reads of a wave (lanes over two of x, y, z) are then at most 2-way bank
  // conflicts instead of 8-way
  constexpr int CZ = 69, CSZ = 7 * CZ + 64;
  __shared__ double cube[6][CSZ];
  __shared__ double cubeJ[HJ ? 6 : 1][HJ ? CSZ : 1];
  __shared__ double tA[64], tB[64], tC[64];  // No <= 64 handled in tiles below
  __shared__ double sE[24];                  // eps_i at the triple's blocks
  // V^bc, V^ac, V^ab on the 8x8 block pairs (r, s) of the current triple
  // (positions r != s of blocks B1, B2, B3): sV[slice][r][s][ly + 8 lz]
  __shared__ double sV[3][3][3][64];
  __shared__ double red[2][4];

  const double *Vbc = P.VHH + (b + Nv * c) * N2;
  const double *Vac = P.VHH + (a + Nv * c) * N2;
  const double *Vab = P.VHH + (a + Nv * b) * N2;
  const double *Ws = P.W + gslot * P.W3;
  const double *Js = have_j ? P.WJ + gslot * P.W3 : Ws;

  int distinct = 0;
  if (a == b) distinct++;
  if (b == c) distinct--;
  const double epsabc = (P.ea[a] + P.ea[b]) + P.ea[c];
  const int nbk = (int)P.nbk;
  const int no = (int)No;
  const int tid = threadIdx.x;

  double e_acc = 0.0, ect_acc = 0.0;
  // Block triples B1 >= B2 >= B3 in nested order (B1 fastest).  The loads
  // of the next triple (cubes, V blocks, t and eps_i tables) are issued into
  // registers before the points of the current one are computed and written
  // to LDS after them, so each triple's memory latency hides behind the
  // previous triple's arithmetic.  Loads are unconditional (the last triple
  // fetches itself again) so none waits behind a branch, and the point loop
  // reads LDS only.
  double tt[12];             // t at (a,x), (b,x), (c,x) and eps_i, x in B1,B2,B3
  double vv[7];              // V^bc, V^ac, V^ab block pairs
  double vw[12];             // cubes of the orbit (2 elements per cube)
  double vwJ[HJ ? 12 : 1];
  int ncur = 0, nnext = 0;
#define FETCH(F1, F2, F3, NC)                                                  \
  {                                                                            \
    const int t_ = tid & 7;                                                    \
    const int xi_ = (F1) * 8 + t_, xj_ = (F2) * 8 + t_, xk_ = (F3) * 8 + t_;   \
    const int ci_ = xi_ < no ? xi_ : 0, cj_ = xj_ < no ? xj_ : 0,              \
              ck_ = xk_ < no ? xk_ : 0;                                        \
    tt[0] = P.Tai[a + Nv * ci_]; tt[1] = P.Tai[a + Nv * cj_];                  \
    tt[2] = P.Tai[a + Nv * ck_]; tt[3] = P.Tai[b + Nv * ci_];                  \
    tt[4] = P.Tai[b + Nv * cj_]; tt[5] = P.Tai[b + Nv * ck_];                  \
    tt[6] = P.Tai[c + Nv * ci_]; tt[7] = P.Tai[c + Nv * cj_];                  \
    tt[8] = P.Tai[c + Nv * ck_]; tt[9] = P.ei[ci_];                            \
    tt[10] = P.ei[cj_]; tt[11] = P.ei[ck_];                                    \
    const int Bp_[3] = {(F1), (F2), (F3)};                                     \
    _Pragma("unroll") for (int it = 0; it < 7; it++) {                         \
      const int e = tid + 256 * it;                                            \
      const int v = e / 576, rs = (e / 64) % 9, l = e & 63;                    \
      const int r = rs / 3, sp = rs % 3;                                       \
      const int y = Bp_[r] * 8 + (l & 7), z = Bp_[sp] * 8 + (l >> 3);          \
      const double *V = v == 0 ? Vbc : v == 1 ? Vac : Vab;                     \
      const bool ok_ = e < 3 * 9 * 64 && r != sp && y < No && z < No;          \
      const double val_ = V[ok_ ? y + No * z : 0];                             \
      vv[it] = ok_ ? val_ : 0.0;                                               \
    }                                                                          \
    int cb_[6], al_[6];                                                        \
    orbit((F1), (F2), (F3), nbk, cb_, NC, al_);                                \
    _Pragma("unroll") for (int it = 0; it < 12; it++) {                        \
      const int p_ = it >> 1, q_ = tid + 256 * (it & 1);                       \
      vw[it] = Ws[cb_[p_ < (NC) ? p_ : 0] + q_];                               \
      if constexpr (HJ) vwJ[it] = Js[cb_[p_ < (NC) ? p_ : 0] + q_];            \
    }                                                                          \
  }
#define COMMIT(C1, C2, C3, NC)                                                 \
  {                                                                            \
    if (tid < 8) {                                                             \
      const int ii_ = (C1) * 8 + tid, jj_ = (C2) * 8 + tid,                    \
                kk_ = (C3) * 8 + tid;                                          \
      tA[tid] = ii_ < No ? P.tai_sign * tt[0] : 0.0;                           \
      tA[8 + tid] = jj_ < No ? P.tai_sign * tt[1] : 0.0;                       \
      tA[16 + tid] = kk_ < No ? P.tai_sign * tt[2] : 0.0;                      \
      tB[tid] = ii_ < No ? P.tai_sign * tt[3] : 0.0;                           \
      tB[8 + tid] = jj_ < No ? P.tai_sign * tt[4] : 0.0;                       \
      tB[16 + tid] = kk_ < No ? P.tai_sign * tt[5] : 0.0;                      \
      tC[tid] = ii_ < No ? P.tai_sign * tt[6] : 0.0;                           \
      tC[8 + tid] = jj_ < No ? P.tai_sign * tt[7] : 0.0;                       \
      tC[16 + tid] = kk_ < No ? P.tai_sign * tt[8] : 0.0;                      \
      sE[tid] = tt[9];                                                         \
      sE[8 + tid] = tt[10];                                                    \
      sE[16 + tid] = tt[11];                                                   \
    }                                                                          \
    _Pragma("unroll") for (int it = 0; it < 7; it++) {                         \
      const int e = tid + 256 * it;                                            \
      if (e < 3 * 9 * 64) (&sV[0][0][0][0])[e] = vv[it];                       \
    }                                                                          \
    _Pragma("unroll") for (int it = 0; it < 12; it++) {                        \
      const int p_ = it >> 1, q_ = tid + 256 * (it & 1);                       \
      if (p_ < (NC)) {                                                         \
        const int at_ = (q_ & 63) + CZ * (q_ >> 6);                            \
        cube[p_][at_] = vw[it];                                                \
        if constexpr (HJ) cubeJ[p_][at_] = vwJ[it];                            \
      }                                                                        \
    }                                                                          \
  }
  int B1 = 0, B2 = 0, B3 = 0;
  FETCH(0, 0, 0, ncur);
#pragma unroll 1
  for (;;) {
    __syncthreads();  // the previous triple's points are done with the LDS
    COMMIT(B1, B2, B3, ncur);
    __syncthreads();
    int N1 = B1 + 1, N2b = B2, N3 = B3;
    if (N1 == nbk) {
      N2b++;
      if (N2b == nbk) {
        N3++;
        N2b = N3;
      }
      N1 = N2b;
    }
    const bool more = N3 < nbk;
    if (!more) {
      N1 = B1;
      N2b = B2;
      N3 = B3;
    }
    FETCH(N1, N2b, N3, nnext);
    int alias[6];
    {
      int cb_[6], nc_;
      orbit(B1, B2, B3, nbk, cb_, nc_, alias);
    }
    triple_points<HJ, 8, CZ, CSZ, false, false>(B1, B2, B3, no, distinct, epsabc,
                                      alias, cube, &cubeJ[0][0], tA, tB, tC,
                                      sE, &sV[0][0][0][0], tid, e_acc,
                                      ect_acc);
    if (!more) break;
    B1 = N1;
    B2 = N2b;
    B3 = N3;
    ncur = nnext;
  }
#undef FETCH
#undef COMMIT

  e_acc = wave_sum(e_acc);
  ect_acc = wave_sum(ect_acc);
  const int wave = tid >> 6, lane = tid & 63;
  if (lane == 0) {
    red[0][wave] = e_acc;
    red[1][wave] = ect_acc;
  }
  __syncthreads();
  if (tid == 0) {
    const double e = (red[0][0] + red[0][1]) + (red[0][2] + red[0][3]);
    const double ect = (red[1][0] + red[1][1]) + (red[1][2] + red[1][3]);
    P.e_slot[2 * gslot] = e;
    P.e_slot[2 * gslot + 1] = have_j ? ect : e;
  }
}

// Fused class sums + singles + energy: one workgroup per (tuple slot, block
// triple B1 >= B2 >= B3 of edge 8).  The workgroup reads the (up to) six
// permuted W cubes of the triple's orbit straight from the three class
// buffers the doubles kernel wrote (4 KiB runs, two elements per lane) and
// sums them in LDS in the fixed order (w + v) + u, the order of wsum_kernel,
// so W is the same bits as in the cube path; then the triple's points follow
// triple_points, and the workgroup's energy (a fixed shuffle/LDS tree) goes
// to its own entry of e_part.  slot_sum_kernel adds a tuple's triples in
// order.  Nothing about W leaves the chip: no cube is written to memory and
// read back.
// Bound by HBM with FP64 buffers (5.8 TB/s read at No=40), by LDS and VALU
// with FP32 ones.  For 155,248 tuples at No=40, Nv=400, FP64 / bf16x3 in ms:
// 57.1 / 55.7 from GEMM-ordered buffers, 53.7 / 47.4 from 8^3 blocks, 41.5 /
// 39.8 with one instance per orbit type and for triples inside the range,
// 40.8 / 36.8 with the LDS strides below; No=60, Nv=240 131 / 119 -> 95 / 83.
struct FusedParams {
  const void *G, *GJ;  // class buffers [3][slots][g_elems(No)] (FP64 or FP32)
  const double *Tai, *VHH, *ei, *ea;
  const uint32_t *points;
  WindowArgs win;
  double *e_part;  // [triple][slot][2]
  int64_t No, Nv, N2, W3g, slots, ntri, npoints;
  int nbk;
  double tai_sign;
};

// Triple t of the nested order B3 outer, B2 = B3.., B1 = B2.. innermost
// (the order the per-tuple kernel walks).
__device__ __forceinline__ void triple_of(int t, int nbk, int &B1, int &B2,
                                          int &B3) {
  int r = t;
  B3 = 0;
  for (;;) {
    const int m = nbk - B3, cnt = m * (m + 1) / 2;
    if (r < cnt) break;
    r -= cnt;
    B3++;
  }
  B2 = B3;
  for (;;) {
    const int cnt = nbk - B2;
    if (r < cnt) break;
    r -= cnt;
    B2++;
  }
  B1 = B2 + r;
}

// The orbit of a block triple B1 >= B2 >= B3 under the six index
// permutations (ijk ikj jik jki kij kji), by type: 0 all different, 1 B1 =
// B2, 2 B2 = B3, 3 all equal.  NC: its distinct cubes; CUBE: their block
// coordinates as positions in (B1, B2, B3); ALIAS: cube of each permutation.
template <int TYPE> struct Orbit;
template <> struct Orbit<0> {
  static constexpr int NC = 6, ALIAS[6] = {0, 1, 2, 3, 4, 5};
  static constexpr int CUBE[6][3] = {{0, 1, 2}, {0, 2, 1}, {1, 0, 2},
                                     {1, 2, 0}, {2, 0, 1}, {2, 1, 0}};
};
template <> struct Orbit<1> {
  static constexpr int NC = 3, ALIAS[6] = {0, 1, 0, 1, 2, 2};
  static constexpr int CUBE[3][3] = {{0, 0, 2}, {0, 2, 0}, {2, 0, 0}};
};
template <> struct Orbit<2> {
  static constexpr int NC = 3, ALIAS[6] = {0, 0, 1, 2, 1, 2};
  static constexpr int CUBE[3][3] = {{0, 1, 1}, {1, 0, 1}, {1, 1, 0}};
};
template <> struct Orbit<3> {
  static constexpr int NC = 1, ALIAS[6] = {0, 0, 0, 0, 0, 0};
  static constexpr int CUBE[1][3] = {{0, 0, 0}};
};

// The loads, class phases and points of one block triple of orbit TYPE: one
// compile-time instance per type, and per triple whose blocks lie inside the
// occupied range (FULL), so every load of an instance is issued before any is
// waited on, none is spent on a repeated cube, and its addresses and LDS
// places are constants next to one per-thread offset (with run-time cube
// codes and range checks 692 VALU instructions per wave, of which about 150
// were the points' arithmetic).
template <typename GT, bool HJ, int TYPE, bool FULL, int CY, int CZ, int CSZ>
__device__ __forceinline__ void fused_orbit(
    const FusedParams &P, int64_t gid, int64_t gslot, int tid, int no,
    int64_t a, int64_t b, int64_t c, int B1, int B2, int B3, int distinct,
    double epsabc, double (*cube)[CSZ], double (*cubeJ)[HJ ? CSZ : 1], double *tA,
    double *tB, double *tC, double *sE, double *sV, double (*red)[4]) {
  const int64_t No = P.No, Nv = P.Nv, N2 = P.N2;
  const int64_t W3g = P.W3g, slots = P.slots;
  const GT *Gs = (const GT *)P.G + gslot * W3g;
  const GT *GJs = (const GT *)P.GJ + gslot * W3g;
  typedef GT g2 __attribute__((ext_vector_type(2)));
  constexpr int NC = Orbit<TYPE>::NC;
  const int alias[6] = {Orbit<TYPE>::ALIAS[0], Orbit<TYPE>::ALIAS[1],
                        Orbit<TYPE>::ALIAS[2], Orbit<TYPE>::ALIAS[3],
                        Orbit<TYPE>::ALIAS[4], Orbit<TYPE>::ALIAS[5]};
  auto pair = [&](int q, int cls) {
    const int *c = Orbit<TYPE>::CUBE[q];
    auto B = [&](int x) { return x == 0 ? B1 : x == 1 ? B2 : B3; };
    return pair_at<CY, CZ, FULL>(cls, B(c[0]), B(c[1]), B(c[2]), P.nbk, no, tid);
  };
  // Every global load of the workgroup is issued before any is waited on
  // (a load behind a branch is waited on before the branch joins, which
  // serialised the first version's loads): W and the (cT) W of the orbit's
  // cubes, the V^bc, V^ac, V^ab blocks of the triple, and (wave 0) t at
  // (a,x), (b,x), (c,x) and eps_i for x in the blocks B1, B2, B3.
  g2 vals[HJ ? 2 : 1][3][NC];
#pragma unroll
  for (int set = 0; set < (HJ ? 2 : 1); set++)
#pragma unroll
    for (int cls = 0; cls < 3; cls++)
#pragma unroll
      for (int q = 0; q < NC; q++)
        vals[set][cls][q] =
            *(const g2 *)((set ? GJs : Gs) + cls * slots * W3g + pair(q, cls).at);
  double vv[5];
  {
    const double *Vbc = P.VHH + (b + Nv * c) * N2;
    const double *Vac = P.VHH + (a + Nv * c) * N2;
    const double *Vab = P.VHH + (a + Nv * b) * N2;
#pragma unroll
    for (int it = 0; it < 5; it++) {
      // entry e: slice v, block pair ps = 2 r + (s - [s > r]) of positions
      // r != s, element l = ly + 8 lz
      const int e = tid + 256 * it;
      const int v = e / 384, ps = (e / 64) % 6, l = e & 63;
      const int r = ps >> 1, s2 = (ps & 1) < r ? (ps & 1) : (ps & 1) + 1;
      // (selects, not an array: a run-time-indexed array lives in
      // scratch, and its loads count in vmcnt behind the gathers)
      const int Br = r == 0 ? B1 : r == 1 ? B2 : B3;
      const int Bs = s2 == 0 ? B1 : s2 == 1 ? B2 : B3;
      const int y = Br * 8 + (l & 7), z = Bs * 8 + (l >> 3);
      const double *V = v == 0 ? Vbc : v == 1 ? Vac : Vab;
      const bool ok_ = (it < 4 || e < 3 * 6 * 64) & (FULL || ((y < No) & (z < No)));
      const double val = V[ok_ ? y + No * z : 0];
      vv[it] = ok_ ? val : 0.0;
    }
  }
  if (tid < 64) {  // wave 0
    const int l = tid < 24 ? tid : 0;
    const int blk = l >> 3 == 0 ? B1 : l >> 3 == 1 ? B2 : B3;
    const int x = blk * 8 + (l & 7);
    const bool in = tid < 24 && x < no;
    const int cx = x < no ? x : 0;
    const double ta = P.Tai[a + Nv * cx], tb = P.Tai[b + Nv * cx],
                 tc = P.Tai[c + Nv * cx], ex = P.ei[cx];
    tA[tid] = in ? P.tai_sign * ta : 0.0;
    tB[tid] = in ? P.tai_sign * tb : 0.0;
    tC[tid] = in ? P.tai_sign * tc : 0.0;
    sE[tid] = ex;
  }
#pragma unroll
  for (int it = 0; it < 5; it++) {
    const int e = tid + 256 * it;
    if (it < 4 || e < 3 * 6 * 64)
      sV[(e >> 6) * V6_BLOCK + (e & 7) + 9 * ((e >> 3) & 7)] = vv[it];
  }
  // the three class phases into LDS in the order w, v, u
#pragma unroll
  for (int cls = 0; cls < 3; cls++) {
#pragma unroll
    for (int q = 0; q < NC; q++) {
      const PairAt a = pair(q, cls);
#pragma unroll
      for (int set = 0; set < (HJ ? 2 : 1); set++) {
        const g2 v = vals[set][cls][q];
        const double v0 = a.in0 ? (double)v[0] : 0.0,
                     v1 = a.in1 ? (double)v[1] : 0.0;
        double *b0 = set ? &cubeJ[q][a.pos] : &cube[q][a.pos], *b1 = b0 + a.step;
        if (cls == 0) {
          *b0 = v0;
          *b1 = v1;
        } else {
          *b0 += v0;
          *b1 += v1;
        }
      }
    }
    __syncthreads();
  }

  double e_acc = 0.0, ect_acc = 0.0;
  triple_points<HJ, CY, CZ, CSZ, true, TYPE == 0 && FULL>(B1, B2, B3, no, distinct, epsabc, alias,
                                   cube, &cubeJ[0][0], tA, tB, tC, sE, sV,
                                   tid, e_acc, ect_acc);
  e_acc = wave_sum(e_acc);
  ect_acc = wave_sum(ect_acc);
  const int wave = tid >> 6, lane = tid & 63;
  if (lane == 0) {
    red[0][wave] = e_acc;
    red[1][wave] = ect_acc;
  }
  __syncthreads();
  if (tid == 0) {
    const double e = (red[0][0] + red[0][1]) + (red[0][2] + red[0][3]);
    const double ect = (red[1][0] + red[1][1]) + (red[1][2] + red[1][3]);
    P.e_part[2 * gid] = e;
    P.e_part[2 * gid + 1] = HJ ? ect : e;
  }
}

template <typename GT, bool HJ>
__global__ __launch_bounds__(256, HJ ? 2 : 4) void energy_fused_kernel(
    FusedParams P) {
  // workgroups go to the 8 XCDs round-robin: XCD x runs the triples of
  // slots x, x + 8, x + 16, ... one slot after the other, so the triples of
  // a slot (whose row pieces share 128-byte lines) meet in one L2, and the
  // slots stay spread over the XCDs
  // (all of the decode in 32-bit unsigned arithmetic: a 64-bit division is
  // ~130 scalar instructions, and the scalar unit, shared by the CU's
  // waves, was the kernel's bound)
  const uint32_t bid = blockIdx.x, r = bid >> 3, ntri = (uint32_t)P.ntri;
  const uint32_t rq = r / ntri;
  const uint32_t gs = 8 * rq + (bid & 7);
  // each slot starts one triple further on: with 4, 20 or 120 triples a fixed
  // order brings the triples of one cube to the same shader engine every time
  uint32_t tr = r - rq * ntri + rq % ntri;
  if (tr >= ntri) tr -= ntri;
  const int tri = (int)tr;
  if ((int64_t)gs >= P.slots) return;
  const int64_t gslot = gs;
  const int64_t gid = tri * P.slots + gslot;
  const int64_t No = P.No, Nv = P.Nv;
  const int tid = threadIdx.x;
  int64_t a, b, c;
  if (!slot_tuple(P.win, (uint64_t)Nv, gs, a, b, c)) {
    if (tid == 0) {
      P.e_part[2 * gid] = 0.0;
      P.e_part[2 * gid + 1] = 0.0;
    }
    return;
  }
  // element x + 9 y + 74 z of a cube: of the 16 lanes that share an LDS cycle
  // at most two meet in a bank, in the class phases (lanes along a pair of
  // x, y or z and the class's second index) and in the points' six reads
  // (lanes along i and j); with x + 8 y + 69 z four did in half of them
  constexpr int CY = 9, CZ = 74, CSZ = 7 * (CY + CZ) + 8;
  __shared__ double cube[6][CSZ];
  __shared__ double cubeJ[HJ ? 6 : 1][HJ ? CSZ : 1];
  // singles tables (entries 0..23 used; wave 0 writes all 64) and the V
  // blocks of the six block pairs of different positions
  __shared__ double tA[64], tB[64], tC[64], sE[64];
  __shared__ double sV[3 * 6 * V6_BLOCK];
  __shared__ double red[2][4];

  int distinct = 0;
  if (a == b) distinct++;
  if (b == c) distinct--;
  const double epsabc = (P.ea[a] + P.ea[b]) + P.ea[c];
  const int no = (int)No;
  int B1, B2, B3;
  triple_of(tri, P.nbk, B1, B2, B3);
  // wave-uniform choice of the instance: only the last block of the range can
  // be partly empty, and B1 is the largest
  const bool full = 8 * (B1 + 1) <= no;
#define ORBIT(T, F)                                                           \
  fused_orbit<GT, HJ, T, F, CY, CZ, CSZ>(P, gid, gslot, tid, no, a, b, c, B1, B2, \
                                     B3, distinct, epsabc, cube, cubeJ, tA,   \
                                     tB, tC, sE, sV, red)
  if (B1 > B2 && B2 > B3) {
    if (full) ORBIT(0, true); else ORBIT(0, false);
  } else if (B1 > B2) {
    if (full) ORBIT(2, true); else ORBIT(2, false);
  } else if (B2 > B3) {
    if (full) ORBIT(1, true); else ORBIT(1, false);
  } else {
    ORBIT(3, false);
  }
#undef ORBIT
}

// The same for small No: T threads do a whole tuple, a wave up to No = 8, four
// up to 14 and eight up to 20, NI pairs of elements of each class per thread.
// By block triples such a tuple took 1 to 10 workgroups of a few points each,
// whose time was their setup, barriers and latencies, and half or more of the
// elements they covered lay outside No; here every thread holds pairs that
// exist and W is read once.  W sits in LDS at x + SY y + SZ z with odd strides, V
// and t whole.  Bound by HBM from No = 9 on: No=10, Nv=90 8.5 ns a tuple for 38
// KB of touched lines, No=16, Nv=80 21 ns for 98 KB; times before and after are
// at small_energy, which chooses.  (No=14, 15, 16 in FP64 with four / eight
// waves: 1.42 / 1.51, 2.0 / 1.83 ms at 14 and 16.)
template <typename GT, bool HJ, int T, int NI>
__global__ __launch_bounds__(T < 256 ? 256 : T, HJ ? 2 : 4) void energy_small_kernel(
    FusedParams P) {
  extern __shared__ double lds[];
  constexpr int S = T < 256 ? 256 / T : 1;  // tuples of a workgroup
  const int tid = threadIdx.x, tl = tid % T;
  const int sub = __builtin_amdgcn_readfirstlane(tid / T);
  const int64_t gslot = (int64_t)blockIdx.x * S + sub;
  if (gslot >= P.slots) return;
  const int64_t Nv = P.Nv;
  int64_t a, b, c;
  if (!slot_tuple(P.win, (uint64_t)Nv, gslot, a, b, c)) {
    if (tl < 2) P.e_part[2 * gslot + tl] = 0.0;
    return;
  }
  // a tuple's threads are one wave, whose LDS accesses are in order, or the
  // workgroup
  auto sync = [] {
    if constexpr (T == 64) {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    } else {
      __syncthreads();
    }
  };
  const int no = (int)P.No, n2 = no * no;
  const int SY = no | 1, SZ = (SY * no) | 1, CS = SZ * no;
  double *cube = lds + sub * ((HJ ? 2 : 1) * CS + 3 * n2 + 4 * no);
  double *cubeJ = cube + CS, *sV = cube + (HJ ? 2 : 1) * CS, *sT = sV + 3 * n2;

  // element pairs (p, q, r), (p, q, r + 1) of the class buffers
  const int H = (no + 1) / 2, count = n2 * H;
  const float rH = 1.0f / (float)H, rN = 1.0f / (float)no;
  uint32_t at[NI];
  int pqr[NI];
#pragma unroll
  for (int it = 0; it < NI; it++) {
    const int e = tl + T * it, x = e < count ? e : 0;
    // (both quotients exact: they lie at least 1 / 40 from a whole number)
    const int m = (int)(((float)x + 0.5f) * rH), r = 2 * (x - m * H);
    const int q = (int)(((float)m + 0.5f) * rN), p = m - q * no;
    at[it] = ((uint32_t)(((q >> 3) * P.nbk + (p >> 3)) * P.nbk + (r >> 3)) << 9) +
             ((q & 7) << 6) + ((p & 7) << 3) + (r & 7);
    pqr[it] = e < count ? p | q << 8 | r << 16 : -1;
  }
  typedef GT g2 __attribute__((ext_vector_type(2)));
#pragma unroll
  for (int set = 0; set < (HJ ? 2 : 1); set++) {
    const GT *Gs = (const GT *)(set ? P.GJ : P.G) + gslot * P.W3g;
    g2 vals[3][NI];
#pragma unroll
    for (int cls = 0; cls < 3; cls++)
#pragma unroll
      for (int it = 0; it < NI; it++)
        vals[cls][it] = *(const g2 *)(Gs + cls * P.slots * P.W3g + at[it]);
    if (set == 0) {
      const int v0 = tl < n2 ? tl : 0, x0 = tl < no ? tl : 0;
      const double vbc = P.VHH[(b + Nv * c) * P.N2 + v0],
                   vac = P.VHH[(a + Nv * c) * P.N2 + v0],
                   vab = P.VHH[(a + Nv * b) * P.N2 + v0];
      const double ta = P.Tai[a + Nv * x0], tb = P.Tai[b + Nv * x0],
                   tc = P.Tai[c + Nv * x0], ex = P.ei[x0];
      if (tl < n2) {
        sV[tl] = vbc;
        sV[n2 + tl] = vac;
        sV[2 * n2 + tl] = vab;
      }
      if (tl < no) {
        sT[tl] = P.tai_sign * ta;
        sT[no + tl] = P.tai_sign * tb;
        sT[2 * no + tl] = P.tai_sign * tc;
        sT[3 * no + tl] = ex;
      }
    }
    double *W = set ? cubeJ : cube;
#pragma unroll
    for (int cls = 0; cls < 3; cls++) {
#pragma unroll
      for (int it = 0; it < NI; it++) {
        if (pqr[it] < 0) continue;
        const int p = pqr[it] & 255, q = (pqr[it] >> 8) & 255, r = pqr[it] >> 16;
        // (p, q, r) in W indices: w (i,j,k), v (i,k,j), u (j,k,i)
        double *w = W + (cls == 0   ? p + SY * q + SZ * r
                         : cls == 1 ? p + SY * r + SZ * q
                                    : r + SY * p + SZ * q);
        const int step = cls == 0 ? SZ : cls == 1 ? SY : 1;
        const double x0 = (double)vals[cls][it][0], x1 = (double)vals[cls][it][1];
        if (cls == 0) {
          w[0] = x0;
          if (r + 1 < no) w[step] = x1;
        } else {
          w[0] += x0;
          if (r + 1 < no) w[step] += x1;
        }
      }
      sync();
    }
  }

  int distinct = 0;
  if (a == b) distinct++;
  if (b == c) distinct--;
  const double epsabc = (P.ea[a] + P.ea[b]) + P.ea[c];
  double e_acc = 0.0, ect_acc = 0.0;
#pragma unroll 1
  for (int pt = tl; pt < (int)P.npoints; pt += T) {
    const uint32_t pk = P.points[pt];
    const int i = pk & 1023, j = (pk >> 10) & 1023, k = pk >> 20;
    const double *tA = sT, *tB = sT + no, *tC = sT + 2 * no, *sE = sT + 3 * no;
    const double fac = (j == k ? 0.5 : 1.0) * (i == j ? 0.5 : 1.0);
    const double denominator = epsabc - ((sE[i] + sE[j]) + sE[k]);
    const int o_ijk = i + SY * j + SZ * k, o_ikj = i + SY * k + SZ * j,
              o_jik = j + SY * i + SZ * k, o_jki = j + SY * k + SZ * i,
              o_kij = k + SY * i + SZ * j, o_kji = k + SY * j + SZ * i;
    // singles at a permutation (x,y,z): t_a[x] V^bc_yz + t_b[y] V^ac_xz
    // + t_c[z] V^ab_xy
    auto Z = [&](double wv, int x, int y, int z) {
      double zz = wv + tA[x] * sV[y + no * z];
      zz = zz + tB[y] * sV[n2 + x + no * z];
      zz = zz + tC[z] * sV[2 * n2 + x + no * y];
      return zz;
    };
    if (distinct == 0) {
      const double A = cube[o_ijk], B = cube[o_ikj], C = cube[o_jik],
                   D = cube[o_jki], E = cube[o_kij], F = cube[o_kji];
      const double U = Z(A, i, j, k), V = Z(B, i, k, j), W = Z(C, j, i, k),
                   X = Z(D, j, k, i), Y = Z(E, k, i, j), Zz = Z(F, k, j, i);
      e_acc += term_distinct(A, B, C, D, E, F, U, V, W, X, Y, Zz, denominator, fac);
      if constexpr (HJ)
        ect_acc += term_distinct(cubeJ[o_ijk], cubeJ[o_ikj], cubeJ[o_jik],
                                 cubeJ[o_jki], cubeJ[o_kij], cubeJ[o_kji], U, V,
                                 W, X, Y, Zz, denominator, fac);
    } else {
      const double A = cube[o_ijk], B = cube[o_jki], C = cube[o_kij];
      const double U = Z(A, i, j, k), V = Z(B, j, k, i), W = Z(C, k, i, j);
      e_acc += term_same(A, B, C, U, V, W, denominator, fac);
      if constexpr (HJ)
        ect_acc += term_same(cubeJ[o_ijk], cubeJ[o_jki], cubeJ[o_kij], U, V, W,
                             denominator, fac);
    }
  }
  e_acc = wave_sum(e_acc);
  ect_acc = wave_sum(ect_acc);
  if constexpr (T > 64) {
    __shared__ double red[2][T / 64];
    if ((tid & 63) == 0) {
      red[0][tid >> 6] = e_acc;
      red[1][tid >> 6] = ect_acc;
    }
    __syncthreads();
    e_acc = ect_acc = 0.0;
    for (int w = 0; w < T / 64; w++) {
      e_acc += red[0][w];
      ect_acc += red[1][w];
    }
  }
  if (tl == 0) {
    P.e_part[2 * gslot] = e_acc;
    P.e_part[2 * gslot + 1] = HJ ? ect_acc : e_acc;
  }
}

template <typename GT, bool HJ>
hipError_t launch_small(const FusedParams &P, hipStream_t st) {
  const int no = (int)P.No, n2 = no * no, SZ = ((no | 1) * no) | 1;
  const int T = no <= 8 ? 64 : no <= 14 ? 256 : 512, S = T < 256 ? 256 / T : 1;
  const size_t lds = sizeof(double) * S * ((HJ ? 2 : 1) * SZ * no + 3 * n2 + 4 * no);
  const int ni = (n2 * ((no + 1) / 2) + T - 1) / T;  // pairs per thread
  const dim3 grid((unsigned)((P.slots + S - 1) / S));
#define SMALL(TT, NI)                                                       \
  if (T == TT && ni <= NI) {                                                \
    /* beyond the 64 KB every launch may have */                            \
    hipError_t e = hipFuncSetAttribute(                                     \
        (const void *)energy_small_kernel<GT, HJ, TT, NI>,                  \
        hipFuncAttributeMaxDynamicSharedMemorySize, MAX_LDS);              \
    if (e != hipSuccess) return e;                                          \
    hipLaunchKernelGGL((energy_small_kernel<GT, HJ, TT, NI>), grid,         \
                       TT < 256 ? 256 : TT, lds, st, P);                    \
    return hipGetLastError();                                               \
  }
  SMALL(64, 1) SMALL(64, 2) SMALL(64, 4)
  SMALL(256, 2) SMALL(256, 4) SMALL(256, 6)
  SMALL(512, 4) SMALL(512, 6)
  // (No = 19, 20: with (cT) or FP32 buffers only, see small_energy)
  if constexpr (HJ || std::is_same_v<GT, float>) SMALL(512, 8)
#undef SMALL
  return hipErrorInvalidConfiguration;
}

// Neumaier step on a (sum, compensation) pair.
__device__ inline void nadd(double &s, double &c, double x) {
  const double t = s + x;
  c += (fabs(s) >= fabs(x)) ? (s - t) + x : (x - t) + s;
  s = t;
}

// Compensated sum of the workgroup's 256 (sum, compensation) pairs of e and
// e_ct by a fixed pairwise tree; thread 0 writes out[0 .. 3].
__device__ inline void pair_tree(double s0, double c0, double s1, double c1,
                                 double (*sh)[256], double *out) {
  const int tid = threadIdx.x;
  sh[0][tid] = s0; sh[1][tid] = c0; sh[2][tid] = s1; sh[3][tid] = c1;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if (tid < h) {
      for (int k = 0; k < 4; k += 2) {
        double s = sh[k][tid], c = sh[k + 1][tid] + sh[k + 1][tid + h];
        nadd(s, c, sh[k][tid + h]);
        sh[k][tid] = s;
        sh[k + 1][tid] = c;
      }
    }
    __syncthreads();
  }
  if (tid < 4) out[tid] = sh[tid][0];
}

// Energy of each tuple slot (with e_part: its triples' partials added in
// triple order, read across the slots), and per 256 slots a compensated sum
// of them to partials[4 * workgroup + {sum, comp, sum_ct, comp_ct}], which
// the host adds in order.  (One workgroup summing a launch's slots by itself
// was a chain of slots / 256 dependent loads: 4.7-8.6 us per launch of 2048
// slots behind a 4.7 us kernel for the triples; both together now 5 us, and
// longer launches cost no more per slot.)
__global__ __launch_bounds__(256) void slot_sum_kernel(const double *e_part,
                                                       int64_t slots,
                                                       int64_t ntri,
                                                       double *e_slot,
                                                       double *partials) {
  __shared__ double sh[4][256];
  const int64_t slot = (int64_t)blockIdx.x * 256 + threadIdx.x;
  double e = 0.0, ect = 0.0;
  if (slot < slots) {
    if (e_part) {
      for (int64_t t = 0; t < ntri; t++) {
        const double *p = e_part + 2 * (t * slots + slot);
        e += p[0];
        ect += p[1];
      }
      e_slot[2 * slot] = e;
      e_slot[2 * slot + 1] = ect;
    } else {
      e = e_slot[2 * slot];
      ect = e_slot[2 * slot + 1];
    }
  }
  pair_tree(e, 0.0, ect, 0.0, sh, partials + 4 * (int64_t)blockIdx.x);
}

// Per window of a batch, a compensated sum of its `per` slot energies: each
// thread over a fixed strided subset, then the fixed tree; (sum, comp) to
// out[2 w], out[2 w + 1].  One workgroup per window (one thread per window
// walked its slots alone: 42 us per launch, 17 % of a served step).
__global__ __launch_bounds__(256) void window_sum_kernel(const double *e_slot,
                                                         int64_t per,
                                                         double *out) {
  __shared__ double sh[4][256];
  __shared__ double res[4];
  const double *e = e_slot + 2 * blockIdx.x * per;
  double sum = 0.0, comp = 0.0;
  for (int64_t q = threadIdx.x; q < per; q += 256) nadd(sum, comp, e[2 * q]);
  pair_tree(sum, comp, 0.0, 0.0, sh, res);
  __syncthreads();
  if (threadIdx.x < 2) out[2 * (int64_t)blockIdx.x + threadIdx.x] = res[threadIdx.x];
}

}  // namespace

hipError_t launch_wsum(const DevSystem &s, const BatchArgs &b, const void *A,
                       bool g32, double *out, hipStream_t st) {
  const int nbk = (int)w_blocks(s.No);
  const int64_t grid = b.slots * (int64_t)nbk * nbk * nbk;
  if (grid <= 0) return hipSuccess;
  if (grid > MAX_GRID) return hipErrorInvalidConfiguration;
  const int64_t W3g = g_elems(s.No);
  if (g32)
    hipLaunchKernelGGL(wsum_kernel<float>, dim3((unsigned)grid), dim3(256), 0,
                       st, (const float *)A, out, (int)s.No, W3g, b.slots,
                       nbk);
  else
    hipLaunchKernelGGL(wsum_kernel<double>, dim3((unsigned)grid), dim3(256),
                       0, st, (const double *)A, out, (int)s.No, W3g, b.slots,
                       nbk);
  return hipGetLastError();
}

hipError_t launch_energy(const DevSystem &s, const BatchArgs &b,
                         const void *G, const void *GJ, bool g32,
                         double tai_sign, double *e_slot, double *scratch,
                         bool fused, hipStream_t st) {
  if (fused) {
    const int64_t nbk = w_blocks(s.No), ntri = energy_parts(s.No, GJ, g32);
    FusedParams P;
    P.points = s.points;
    P.npoints = s.npoints;
    P.G = G;
    P.GJ = GJ;
    P.Tai = s.Tai;
    P.VHH = s.VHH;
    P.ei = s.ei;
    P.ea = s.ea;
    P.win = b;
    P.e_part = scratch;
    P.No = s.No;
    P.Nv = s.Nv;
    P.N2 = s.No * s.No;
    P.W3g = g_elems(s.No);
    P.slots = b.slots;
    P.ntri = ntri;
    P.nbk = (int)nbk;
    P.tai_sign = tai_sign;
    const int64_t grid = (b.slots + 7) / 8 * 8 * ntri;
    if (grid <= 0) return hipSuccess;
    if (small_energy(s.No, GJ, g32)) {
      if (grid > MAX_GRID) return hipErrorInvalidConfiguration;
      if (g32)
        return GJ ? launch_small<float, true>(P, st)
                  : launch_small<float, false>(P, st);
      return GJ ? launch_small<double, true>(P, st)
                : launch_small<double, false>(P, st);
    }
    // (the kernel decodes its block id and class-buffer offsets in 32 bits)
    if (grid > MAX_GRID || g_elems(s.No) >= (int64_t(1) << 31))
      return hipErrorInvalidConfiguration;
    if (g32 && GJ)
      hipLaunchKernelGGL((energy_fused_kernel<float, true>), dim3((unsigned)grid),
                         dim3(256), 0, st, P);
    else if (g32)
      hipLaunchKernelGGL((energy_fused_kernel<float, false>), dim3((unsigned)grid),
                         dim3(256), 0, st, P);
    else if (GJ)
      hipLaunchKernelGGL((energy_fused_kernel<double, true>), dim3((unsigned)grid),
                         dim3(256), 0, st, P);
    else
      hipLaunchKernelGGL((energy_fused_kernel<double, false>), dim3((unsigned)grid),
                         dim3(256), 0, st, P);
    return hipGetLastError();
  }
  const int64_t W3c = w_cube(s.No);
  double *W = scratch, *WJ = GJ ? scratch + b.slots * W3c : nullptr;
  hipError_t e = launch_wsum(s, b, G, g32, W, st);
  if (e != hipSuccess) return e;
  if (GJ && (e = launch_wsum(s, b, GJ, g32, WJ, st)) != hipSuccess)
    return e;
  EnergyParams P;
  P.W = W;
  P.WJ = WJ;
  P.Tai = s.Tai;
  P.VHH = s.VHH;
  P.ei = s.ei;
  P.ea = s.ea;
  P.win = b;
  P.e_slot = e_slot;
  P.No = s.No;
  P.Nv = s.Nv;
  P.N2 = s.No * s.No;
  P.nbk = w_blocks(s.No);
  P.W3 = W3c;
  P.slots = b.slots;
  P.tai_sign = tai_sign;
  const dim3 grid((unsigned)b.slots), block(256);
  if (GJ)
    hipLaunchKernelGGL(energy_kernel<true>, grid, block, 0, st, P);
  else
    hipLaunchKernelGGL(energy_kernel<false>, grid, block, 0, st, P);
  return hipGetLastError();
}

hipError_t launch_window_sums(const double *e_slot, int nw, int64_t per,
                              double *out, hipStream_t st) {
  if (nw <= 0) return hipSuccess;
  hipLaunchKernelGGL(window_sum_kernel, dim3((unsigned)nw), dim3(256), 0, st,
                     e_slot, per, out);
  return hipGetLastError();
}

hipError_t launch_slot_sums(const double *e_part, int64_t slots, int64_t ntri,
                            double *e_slot, double *partials, hipStream_t st) {
  if (slots <= 0) return hipSuccess;
  hipLaunchKernelGGL(slot_sum_kernel, dim3((unsigned)slot_partials(slots)),
                     dim3(256), 0, st, e_part, slots, ntri, e_slot, partials);
  return hipGetLastError();
}

}  // namespace atrip_amd
