// Singles + energy epilogue of complex (T) (atrip::Atrip::run<Complex>).
//
// The doubles of a complex system run as real class GEMMs on real/imaginary
// operand planes (see the run loop), so W = Wr + i Wi arrives as two sets of
// class buffers.  Up to No = 20 (16 with (cT)) energy_z_small_kernel takes a
// tuple straight from them; beyond, they are summed into cubes by launch_wsum
// and energy_z_kernel (one workgroup per tuple) reads, for each block triple of
// edge 8, the cubes holding W at the six index permutations into LDS.
// Z = W + singles is formed with complex products (reference
// src/atrip/Equations.cxx:387-426), and the energy follows
// get_energy_distinct / get_energy_same (:101-238) with F = Complex:
// A..F = conj(W) (maybe_conjugate_scalar), U..Z = Z, complex denominators,
// real part of the tuple's sum (:176-178).  Fixed per-thread order and a
// fixed reduction tree, as the real epilogue.
#include "internal.hpp"

namespace atrip_amd {
namespace {

struct cplx {
  double r, i;
};
__device__ inline cplx operator+(cplx a, cplx b) { return {a.r + b.r, a.i + b.i}; }
__device__ inline cplx operator-(cplx a, cplx b) { return {a.r - b.r, a.i - b.i}; }
__device__ inline cplx operator*(cplx a, cplx b) {
  return {a.r * b.r - a.i * b.i, a.r * b.i + a.i * b.r};
}
__device__ inline cplx operator*(double s, cplx a) { return {s * a.r, s * a.i}; }
__device__ inline cplx conj(cplx a) { return {a.r, -a.i}; }
// Real part of a / b (Smith's scaling, exact for real b).
__device__ inline double re_div(cplx a, cplx b) {
  if (b.i == 0.0) return a.r / b.r;
  if (fabs(b.r) >= fabs(b.i)) {
    const double t = b.i / b.r, d = b.r + b.i * t;
    return (a.r + a.i * t) / d;
  }
  const double t = b.r / b.i, d = b.r * t + b.i;
  return (a.r * t + a.i) / d;
}

struct EnergyZParams {
  const double *Wr, *Wi, *WJr, *WJi;  // cubes [slot][W3], or class buffers
  const uint32_t *points;
  int64_t npoints;
  const double *Tair, *Taii, *VHHr, *VHHi, *eir, *eii, *ear;
  WindowArgs win;
  double *e_slot;
  int64_t No, Nv, N2, W3, nbk, slots;  // nbk: cubes per index, W3 = (8 nbk)^3
  double tai_sign;
};

__device__ inline double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// A point's energy term from W and Z at its six permutations.
__device__ __forceinline__ double z_term(const cplx (&Wq)[6], const cplx (&Zp)[6],
                                         int distinct, cplx den, double fac) {
  cplx value;
  if (distinct == 0) {
    const cplx A = conj(Wq[0]), B = conj(Wq[1]), C = conj(Wq[2]),
               D = conj(Wq[3]), E = conj(Wq[4]), F = conj(Wq[5]);
    const cplx U = Zp[0], V = Zp[1], W = Zp[2], X = Zp[3], Y = Zp[4],
               Z = Zp[5];
    const cplx UXY = U + (X + Y), VWZ = V + (W + Z);
    const cplx first = A * U + (B * V + (C * W + (D * X + (E * Y + F * Z))));
    value = 3.0 * first + ((UXY - 2.0 * VWZ) * (A + (D + E)) +
                           (VWZ - 2.0 * UXY) * (B + (C + F)));
  } else {
    const cplx A = conj(Wq[0]), B = conj(Wq[3]), C = conj(Wq[4]);
    const cplx U = Zp[0], V = Zp[3], W = Zp[4];
    value = 3.0 * ((A * U + B * V) + C * W) - (A + (B + C)) * (U + (V + W));
  }
  return re_div(2.0 * value, den) * fac;
}

template <bool HJ>
__global__ __launch_bounds__(256) void energy_z_kernel(EnergyZParams P) {
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
  __shared__ double cr[6][512], ci[6][512];
  __shared__ double jr[HJ ? 6 : 1][HJ ? 512 : 1], ji[HJ ? 6 : 1][HJ ? 512 : 1];
  __shared__ double red[2][4];

  const int64_t pbc = (b + Nv * c) * N2, pac = (a + Nv * c) * N2,
                pab = (a + Nv * b) * N2;
  int distinct = 0;
  if (a == b) distinct++;
  if (b == c) distinct--;
  // the reference keeps only the real part of the virtual-orbital sum
  // (std::real, src/atrip/Atrip.cxx:643-644); the occupied energies of the
  // denominator stay complex
  const cplx epsabc = cplx{(P.ear[a] + P.ear[b]) + P.ear[c], 0.0};
  const int nbk = (int)P.nbk, no = (int)No, tid = threadIdx.x;
  auto tai = [&](int64_t x, int occ) {
    return cplx{P.tai_sign * P.Tair[x + Nv * occ], P.tai_sign * P.Taii[x + Nv * occ]};
  };
  auto vhh = [&](int64_t base, int p, int q) {
    return cplx{P.VHHr[base + p + no * q], P.VHHi[base + p + no * q]};
  };
  const int64_t off = gslot * P.W3;

  double e_acc = 0.0, ect_acc = 0.0;
#pragma unroll 1
  for (int B3 = 0; B3 < nbk; B3++)
#pragma unroll 1
    for (int B2 = B3; B2 < nbk; B2++)
#pragma unroll 1
      for (int B1 = B2; B1 < nbk; B1++) {
        // cubes of the permutations ijk ikj jik jki kij kji
        const int cx[6] = {B1, B1, B2, B2, B3, B3};
        const int cy[6] = {B2, B3, B1, B3, B1, B2};
        const int cz[6] = {B3, B2, B3, B1, B2, B1};
        __syncthreads();
        for (int p = 0; p < 6; p++) {
          const int64_t base = off + (((int64_t)(cz[p] * nbk + cy[p]) * nbk + cx[p]) << 9);
          for (int q = tid; q < 512; q += 256) {
            cr[p][q] = P.Wr[base + q];
            ci[p][q] = P.Wi[base + q];
            if constexpr (HJ) {
              jr[p][q] = P.WJr[base + q];
              ji[p][q] = P.WJi[base + q];
            }
          }
        }
        __syncthreads();
#pragma unroll 1
        for (int pt = tid; pt < 512; pt += 256) {
          const int li = pt & 7, lj = (pt >> 3) & 7, lk = pt >> 6;
          const int i = B1 * 8 + li, j = B2 * 8 + lj, k = B3 * 8 + lk;
          if (i >= no || j >= no || k >= no || i < j || j < k) continue;
          const double facjk = j == k ? 0.5 : 1.0, facij = i == j ? 0.5 : 1.0;
          const cplx den = epsabc - ((cplx{P.eir[i], P.eii[i]} + cplx{P.eir[j], P.eii[j]}) +
                                     cplx{P.eir[k], P.eii[k]});
          const int o[6] = {li + 8 * lj + 64 * lk, li + 8 * lk + 64 * lj,
                            lj + 8 * li + 64 * lk, lj + 8 * lk + 64 * li,
                            lk + 8 * li + 64 * lj, lk + 8 * lj + 64 * li};
          const int px[6] = {i, i, j, j, k, k}, py[6] = {j, k, i, k, i, j},
                    pz[6] = {k, j, k, i, j, i};
          cplx Wp[6], Zp[6];
#pragma unroll
          for (int p = 0; p < 6; p++) {
            Wp[p] = cplx{cr[p][o[p]], ci[p][o[p]]};
            // Z = W + t_a[x] V^bc_yz + t_b[y] V^ac_xz + t_c[z] V^ab_xy
            cplx z = Wp[p] + tai(a, px[p]) * vhh(pbc, py[p], pz[p]);
            z = z + tai(b, py[p]) * vhh(pac, px[p], pz[p]);
            z = z + tai(c, pz[p]) * vhh(pab, px[p], py[p]);
            Zp[p] = z;
          }
          e_acc += z_term(Wp, Zp, distinct, den, facjk * facij);
          if constexpr (HJ) {
            cplx Jp[6];
#pragma unroll
            for (int p = 0; p < 6; p++) Jp[p] = cplx{jr[p][o[p]], ji[p][o[p]]};
            ect_acc += z_term(Jp, Zp, distinct, den, facjk * facij);
          }
        }
      }
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
    P.e_slot[2 * gslot + 1] = HJ ? ect : e;
  }
}

// The same for small No straight from the class buffers, the planes' classes
// summed in LDS as the real kernel for small No does: T threads do a whole tuple,
// a wave up to No = 8 and eight beyond, NI pairs of elements per thread, class
// and plane; W, V and t of both planes sit in LDS.  By cubes the sums went
// through memory twice and every point read 36 values of V from there.
// No=14, Nv=90 20.6 -> 4.9 ms (18.8 GB of touched lines: 3.9 TB/s), No=4, Nv=50
// 0.59 -> 0.05, No=20, Nv=60 15.4 -> 4.6 (one workgroup a CU), (cT) No=16, Nv=60
// 12.8 -> 4.3.
template <bool HJ, int T, int NI>
__global__ __launch_bounds__(T < 256 ? 256 : T) void energy_z_small_kernel(
    EnergyZParams P) {
  extern __shared__ double lds[];
  constexpr int S = T < 256 ? 256 / T : 1, PL = HJ ? 4 : 2;
  const int tid = threadIdx.x, tl = tid % T;
  const int sub = __builtin_amdgcn_readfirstlane(tid / T);
  const int64_t gslot = (int64_t)blockIdx.x * S + sub;
  if (gslot >= P.slots) return;
  const int64_t Nv = P.Nv;
  int64_t a, b, c;
  if (!slot_tuple(P.win, (uint64_t)Nv, gslot, a, b, c)) {
    if (tl < 2) P.e_slot[2 * gslot + tl] = 0.0;
    return;
  }
  auto sync = [] {
    if constexpr (T == 64) {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    } else {
      __syncthreads();
    }
  };
  const int no = (int)P.No, n2 = no * no, nbk = (int)P.nbk;
  const int SY = no | 1, SZ = (SY * no) | 1, CS = SZ * no;
  double *cube = lds + sub * (PL * CS + 6 * n2 + 8 * no);
  double *sV = cube + PL * CS, *sT = sV + 6 * n2;

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
    at[it] = ((uint32_t)(((q >> 3) * nbk + (p >> 3)) * nbk + (r >> 3)) << 9) +
             ((q & 7) << 6) + ((p & 7) << 3) + (r & 7);
    pqr[it] = e < count ? p | q << 8 | r << 16 : -1;
  }
  typedef double d2 __attribute__((ext_vector_type(2)));
#pragma unroll
  for (int pl = 0; pl < PL; pl++) {
    const double *G = pl == 0 ? P.Wr : pl == 1 ? P.Wi : pl == 2 ? P.WJr : P.WJi;
    G += gslot * P.W3;
    d2 vals[3][NI];
#pragma unroll
    for (int cls = 0; cls < 3; cls++)
#pragma unroll
      for (int it = 0; it < NI; it++)
        vals[cls][it] = *(const d2 *)(G + cls * P.slots * P.W3 + at[it]);
    if (pl < 2) {  // V and t of the plane
      const double *V = pl ? P.VHHi : P.VHHr, *t = pl ? P.Taii : P.Tair;
      const int v0 = tl < n2 ? tl : 0, x0 = tl < no ? tl : 0;
      const double vbc = V[(b + Nv * c) * P.N2 + v0],
                   vac = V[(a + Nv * c) * P.N2 + v0],
                   vab = V[(a + Nv * b) * P.N2 + v0];
      const double ta = t[a + Nv * x0], tb = t[b + Nv * x0], tc = t[c + Nv * x0],
                   ex = (pl ? P.eii : P.eir)[x0];
      if (tl < n2) {
        sV[3 * n2 * pl + tl] = vbc;
        sV[3 * n2 * pl + n2 + tl] = vac;
        sV[3 * n2 * pl + 2 * n2 + tl] = vab;
      }
      if (tl < no) {
        sT[4 * no * pl + tl] = P.tai_sign * ta;
        sT[4 * no * pl + no + tl] = P.tai_sign * tb;
        sT[4 * no * pl + 2 * no + tl] = P.tai_sign * tc;
        sT[4 * no * pl + 3 * no + tl] = ex;
      }
    }
    double *W = cube + pl * CS;
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
        if (cls == 0) {
          w[0] = vals[cls][it][0];
          if (r + 1 < no) w[step] = vals[cls][it][1];
        } else {
          w[0] += vals[cls][it][0];
          if (r + 1 < no) w[step] += vals[cls][it][1];
        }
      }
      sync();
    }
  }

  int distinct = 0;
  if (a == b) distinct++;
  if (b == c) distinct--;
  const cplx epsabc = cplx{(P.ear[a] + P.ear[b]) + P.ear[c], 0.0};
  double e_acc = 0.0, ect_acc = 0.0;
#pragma unroll 1
  for (int pt = tl; pt < (int)P.npoints; pt += T) {
    const uint32_t pk = P.points[pt];
    const int i = pk & 1023, j = (pk >> 10) & 1023, k = pk >> 20;
    const double fac = (j == k ? 0.5 : 1.0) * (i == j ? 0.5 : 1.0);
    auto tab = [&](int t, int x) {
      return cplx{sT[t * no + x], sT[4 * no + t * no + x]};
    };
    auto vhh = [&](int v, int x, int y) {
      return cplx{sV[v * n2 + x + no * y], sV[3 * n2 + v * n2 + x + no * y]};
    };
    const cplx den = epsabc - ((tab(3, i) + tab(3, j)) + tab(3, k));
    const int px[6] = {i, i, j, j, k, k}, py[6] = {j, k, i, k, i, j},
              pz[6] = {k, j, k, i, j, i};
    cplx Wp[6], Zp[6];
#pragma unroll
    for (int p = 0; p < 6; p++) {
      const int o = px[p] + SY * py[p] + SZ * pz[p];
      Wp[p] = cplx{cube[o], cube[CS + o]};
      // Z = W + t_a[x] V^bc_yz + t_b[y] V^ac_xz + t_c[z] V^ab_xy
      cplx z = Wp[p] + tab(0, px[p]) * vhh(0, py[p], pz[p]);
      z = z + tab(1, py[p]) * vhh(1, px[p], pz[p]);
      z = z + tab(2, pz[p]) * vhh(2, px[p], py[p]);
      Zp[p] = z;
    }
    e_acc += z_term(Wp, Zp, distinct, den, fac);
    if constexpr (HJ) {
#pragma unroll
      for (int p = 0; p < 6; p++) {
        const int o = px[p] + SY * py[p] + SZ * pz[p];
        Wp[p] = cplx{cube[2 * CS + o], cube[3 * CS + o]};
      }
      ect_acc += z_term(Wp, Zp, distinct, den, fac);
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
    P.e_slot[2 * gslot] = e_acc;
    P.e_slot[2 * gslot + 1] = HJ ? ect_acc : e_acc;
  }
}

template <bool HJ>
hipError_t launch_z_small(const EnergyZParams &P, hipStream_t st) {
  const int no = (int)P.No, n2 = no * no, SZ = ((no | 1) * no) | 1;
  const int T = no <= 8 ? 64 : 512, S = T < 256 ? 256 / T : 1;
  const size_t lds =
      sizeof(double) * S * ((HJ ? 4 : 2) * SZ * no + 6 * n2 + 8 * no);
  const int ni = (n2 * ((no + 1) / 2) + T - 1) / T;  // pairs per thread
  const dim3 grid((unsigned)((P.slots + S - 1) / S));
#define SMALL(TT, NI)                                                         \
  if (T == TT && ni <= NI) {                                                  \
    /* beyond the 64 KB every launch may have */                              \
    hipError_t e = hipFuncSetAttribute(                                       \
        (const void *)energy_z_small_kernel<HJ, TT, NI>,                      \
        hipFuncAttributeMaxDynamicSharedMemorySize, MAX_LDS);                \
    if (e != hipSuccess) return e;                                            \
    hipLaunchKernelGGL((energy_z_small_kernel<HJ, TT, NI>), grid,             \
                       TT < 256 ? 256 : TT, lds, st, P);                      \
    return hipGetLastError();                                                 \
  }
  SMALL(64, 1) SMALL(64, 4) SMALL(512, 2) SMALL(512, 4)
  // (No = 17..20: without (cT) only, see small_energy_z)
  if constexpr (!HJ) SMALL(512, 8)
#undef SMALL
  return hipErrorInvalidConfiguration;
}

}  // namespace

hipError_t launch_energy_z(const DevSystem &s, const BatchArgs &b,
                           double *const G[2], double *const GJ[2],
                           double tai_sign, double *e_slot, double *wcube,
                           bool fused, hipStream_t st) {
  const bool small = fused && small_energy_z(s.No, GJ);
  const int64_t W3c = small ? g_elems(s.No) : w_cube(s.No), n = b.slots * W3c;
  EnergyZParams P;
  P.points = s.points;
  P.npoints = s.npoints;
  P.Wr = wcube;
  P.Wi = wcube + n;
  P.WJr = GJ ? wcube + 2 * n : nullptr;
  P.WJi = GJ ? wcube + 3 * n : nullptr;
  if (small) {
    P.Wr = G[0];
    P.Wi = G[1];
    P.WJr = GJ ? GJ[0] : nullptr;
    P.WJi = GJ ? GJ[1] : nullptr;
  }
  hipError_t e;
  if (small) {
    // (nothing to sum first)
  } else if ((e = launch_wsum(s, b, G[0], false, (double *)P.Wr, st)) != hipSuccess ||
      (e = launch_wsum(s, b, G[1], false, (double *)P.Wi, st)) != hipSuccess)
    return e;
  if (!small && GJ &&
      ((e = launch_wsum(s, b, GJ[0], false, (double *)P.WJr, st)) != hipSuccess ||
       (e = launch_wsum(s, b, GJ[1], false, (double *)P.WJi, st)) != hipSuccess))
    return e;
  P.Tair = s.Tai;
  P.Taii = s.Taii;
  P.VHHr = s.VHH;
  P.VHHi = s.VHHi;
  P.eir = s.ei;
  P.eii = s.eii;
  P.ear = s.ea;
  P.win = b;
  P.e_slot = e_slot;
  P.No = s.No;
  P.Nv = s.Nv;
  P.N2 = s.No * s.No;
  P.nbk = w_blocks(s.No);
  P.W3 = W3c;
  P.slots = b.slots;
  P.tai_sign = tai_sign;
  if (small)
    return b.slots <= 0 ? hipSuccess
           : GJ         ? launch_z_small<true>(P, st)
                        : launch_z_small<false>(P, st);
  const dim3 grid((unsigned)b.slots), block(256);
  if (GJ)
    hipLaunchKernelGGL(energy_z_kernel<true>, grid, block, 0, st, P);
  else
    hipLaunchKernelGGL(energy_z_kernel<false>, grid, block, 0, st, P);
  return hipGetLastError();
}

}  // namespace atrip_amd
