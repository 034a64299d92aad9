// Device re-layout of CTF tensors and on-device synthetic generation.
//
// The reference cuts slices out of the CTF tensors with Tensor::slice into
// contiguous buffers once per run (src/atrip/Unions.hpp:22-75) and then
// ships them per tuple.  Here every tensor is re-laid out once, on the
// device, into the layouts documented on DevSystem (internal.hpp), and stays
// resident.  The same layouts can also be filled straight from the
// counter-based generator, which avoids host generation and PCIe traffic for
// large synthetic systems.
#include "../../include/atrip_synth.h"
#include "internal.hpp"

#include <algorithm>

namespace atrip_amd {
namespace {

constexpr int TT = 32;  // transpose tile edge

// dst[o*dst_o + a*dst_a + b*dst_b] = scale * src[o*src_o + a*src_a + b*src_b]
// b is the contiguous source index, a the contiguous destination index.
__global__ __launch_bounds__(256) void transpose_kernel(
    const double *__restrict__ src, double *__restrict__ dst, int64_t n_a,
    int64_t n_b, int64_t tiles_a, int64_t src_o, int64_t src_a, int64_t src_b,
    int64_t dst_o, int64_t dst_a, int64_t dst_b, double scale) {
  __shared__ double tile[TT][TT + 1];
  const int64_t o = blockIdx.y;
  const int64_t ta = blockIdx.x % tiles_a, tb = blockIdx.x / tiles_a;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const double *s = src + o * src_o;
  double *d = dst + o * dst_o;
#pragma unroll
  for (int r = 0; r < TT; r += 8) {
    const int64_t a = ta * TT + ty + r, b = tb * TT + tx;
    if (a < n_a && b < n_b) tile[ty + r][tx] = s[a * src_a + b * src_b];
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < TT; r += 8) {
    const int64_t b = tb * TT + ty + r, a = ta * TT + tx;
    if (a < n_a && b < n_b) d[a * dst_a + b * dst_b] = scale * tile[tx][ty + r];
  }
}

// The same through the tile addresses of an FP64 operand (f64_at).  A row's
// consecutive k are 16-byte pairs 256 bytes apart, so the writes are 16-byte
// pieces; uploads are bound by the host link, not by them.
__global__ __launch_bounds__(256) void transpose_tiled_kernel(
    const double *__restrict__ src, double *__restrict__ dst, int64_t n_a,
    int64_t n_b, int64_t tiles_a, int64_t o_first, int64_t src_o,
    int64_t src_a, int64_t src_b, TileMap m, double scale) {
  __shared__ double tile[TT][TT + 1];
  const int64_t o = blockIdx.y + o_first;
  const int64_t ta = blockIdx.x % tiles_a, tb = blockIdx.x / tiles_a;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const double *s = src + o * src_o;
#pragma unroll
  for (int r = 0; r < TT; r += 8) {
    const int64_t a = ta * TT + ty + r, b = tb * TT + tx;
    if (a < n_a && b < n_b) tile[ty + r][tx] = s[a * src_a + b * src_b];
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < TT; r += 8) {
    const int64_t b = tb * TT + ty + r, a = ta * TT + tx;
    if (a >= n_a || b >= n_b) continue;
    int64_t R = m.R0 + o * m.Ro + a * m.Ra + b * m.Rb;
    if (m.swap) {
      const int64_t row = m.swap == 1 ? m.row0 + o : b;
      R += row / m.No + m.No * (row % m.No);
    }
    dst[f64_at(R, m.k0 + o * m.ko + a * m.ka, m.K)] = scale * tile[tx][ty + r];
  }
}

enum SynthTarget { S_T3, S_V3, S_H3, S_T2N, S_T2TN };

// Fill the forms `out` of a doubles operand of geometry g from the generator,
// one octet (eight k of a row) per thread, consecutive threads on the
// consecutive rows of a 16-row tile, so FP64 and bf16x3 tiles are written in
// whole lines and the index divisions are paid once per eight values.  Bound
// by the generator's FP64 arithmetic; at No=40, Nv=400 all operands take 30 ms
// in bf16x3 (48 ms with one element per thread and scattered 2-byte stores)
// and 30 ms in FP64 with the row-swapped copies (32 ms without them before).
// swapped: row p + No q holds the values of row q + No p.
__global__ __launch_bounds__(256) void synth_operand_kernel(
    OpSink out, TriGeom g, int64_t n, int target, int tensor, uint64_t stream,
    int64_t No, int64_t Nv, bool swapped, double scale) {
  const int64_t N2 = No * No, Nv2 = Nv * Nv, K8 = g.K >> 3;
  for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < n;
       q += (int64_t)gridDim.x * blockDim.x) {
    const int64_t t = q >> 4, R = t / K8 * 16 + (q & 15), k8 = t % K8 * 8;
    const int64_t o = R / g.nrp;
    int64_t r = R - o * g.nrp, base = 0, step = 0, kmax = 0;
    const int64_t row = r;
    double v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    if (o < g.no && r < g.nr) {
      if (swapped) r = r / No + No * (r % No);
      double sign = 1.0;
      switch (target) {
      case S_T3:  // [x][row][E] = Tpphh[x,E,row]
        base = o + Nv2 * r; step = Nv; kmax = Nv;
        break;
      case S_V3:  // [pair][r][E] = Vppph[pair,E,r]
        base = o + Nv2 * Nv * r; step = Nv2; kmax = Nv;
        break;
      case S_H3:  // [x][row][L] = Vhhhp[row,L,x]
        base = r + N2 * No * o; step = N2; kmax = No;
        break;
      case S_T2N:  // [pair][n][L] = -Tpphh[pair,L,n]
        base = o + Nv2 * No * r; step = Nv2; kmax = No; sign = -1.0;
        break;
      default:  // S_T2TN: [pair][n][L] = -Tpphh[pair,n,L]
        base = o + Nv2 * r; step = Nv2 * No; kmax = No; sign = -1.0;
      }
#pragma unroll 1
      for (int e = 0; e < 8; e++) {
        const int64_t k = k8 + e;
        if (k >= kmax) break;
        const double x = sign * atrip_synth_value(stream, tensor, (uint64_t)No,
                                                  (uint64_t)Nv,
                                                  (uint64_t)(base + k * step)) *
                         scale;
        // a run-time index into v would put it in scratch memory
#pragma unroll
        for (int z = 0; z < 8; z++)
          if (z == e) v[z] = x;
      }
    }
    sink_put8(v, out, g, o, row, k8);
  }
}

// Fill a plain array of n elements: element q is the tensor's element q, or
// with nij > 0 (VHH) [pair][ij] = Vpphh[pair,ij], nij = No^2.
__global__ __launch_bounds__(256) void synth_plain_kernel(
    double *dst, int64_t n, int64_t nij, int tensor, uint64_t stream,
    int64_t No, int64_t Nv, double scale) {
  for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < n;
       q += (int64_t)gridDim.x * blockDim.x) {
    const int64_t idx = nij ? q / nij + Nv * Nv * (q % nij) : q;
    dst[q] = atrip_synth_value(stream, tensor, (uint64_t)No, (uint64_t)Nv,
                               (uint64_t)idx) * scale;
  }
}

// FP64 operand to another form, one octet per thread in the order of the
// destination's tiles.
__global__ __launch_bounds__(256) void convert_kernel(const double *x,
                                                      TriGeom gx, OpSink out,
                                                      TriGeom g, bool swapped,
                                                      int64_t No, int64_t n) {
  typedef double d2 __attribute__((ext_vector_type(2)));
  const int64_t K8 = g.K >> 3;
  for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < n;
       q += (int64_t)gridDim.x * blockDim.x) {
    const int64_t t = q >> 4, R = t / K8 * 16 + (q & 15), k8 = t % K8 * 8;
    const int64_t o = R / g.nrp, r = R - o * g.nrp;
    double v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    if (o < g.no && r < g.nr) {
      const int64_t rs = swapped ? r / No + No * (r % No) : r;
      const double *at = x + f64_at(o * gx.nrp + rs, k8, gx.K);
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const d2 y = *(const d2 *)(at + 32 * e);
        v[2 * e] = y[0];
        v[2 * e + 1] = y[1];
      }
    }
    sink_put8(v, out, g, o, r, k8);
  }
}

unsigned fill_blocks(int64_t n) {
  return (unsigned)std::min<int64_t>((n + 255) / 256, 65536L * 16);
}

// Rows of a form's arrays, whole tiles of 32 (bf16x3) or 16 rows.
int64_t fill_rows(const OpSink &out, const TriGeom &g) {
  return out.t ? pad32(g.no * g.nrp) : pad16(g.no * g.nrp);
}

hipError_t synth_operand(const OpSink &out, const TriGeom &g,
                         SynthTarget target, int tensor, uint64_t seed,
                         const DevSystem &s, bool swapped, double scale,
                         hipStream_t st) {
  const int64_t n = fill_rows(out, g) * (g.K >> 3);
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(synth_operand_kernel, dim3(fill_blocks(n)), dim3(256), 0,
                     st, out, g, n, (int)target, tensor,
                     atrip_synth_stream(seed, tensor), s.No, s.Nv, swapped,
                     scale);
  return hipGetLastError();
}

hipError_t synth_plain(double *dst, int64_t n, int64_t nij, int tensor,
                       uint64_t seed, const DevSystem &s, double scale,
                       hipStream_t st) {
  if (n <= 0) return hipSuccess;
  // amplitudes and integrals carry the scale, orbital energies do not
  const int base = tensor & 15;
  if (base == ATRIP_SYN_EI || base == ATRIP_SYN_EA) scale = 1.0;
  hipLaunchKernelGGL(synth_plain_kernel, dim3(fill_blocks(n)), dim3(256), 0,
                     st, dst, n, nij, tensor, atrip_synth_stream(seed, tensor),
                     s.No, s.Nv, scale);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_transpose(const double *src, double *dst, int64_t n_outer,
                            int64_t n_a, int64_t n_b, int64_t src_o,
                            int64_t src_a, int64_t src_b, int64_t dst_o,
                            int64_t dst_a, int64_t dst_b, double scale,
                            hipStream_t st) {
  if (n_outer <= 0 || n_a <= 0 || n_b <= 0) return hipSuccess;
  const int64_t tiles_a = (n_a + TT - 1) / TT, tiles_b = (n_b + TT - 1) / TT;
  // blockIdx.y carries the outer index (<= 65535 per launch)
  for (int64_t o0 = 0; o0 < n_outer; o0 += 65535) {
    const int64_t no = n_outer - o0 < 65535 ? n_outer - o0 : 65535;
    hipLaunchKernelGGL(transpose_kernel, dim3((unsigned)(tiles_a * tiles_b),
                                              (unsigned)no),
                       dim3(256), 0, st, src + o0 * src_o, dst + o0 * dst_o,
                       n_a, n_b, tiles_a, src_o, src_a, src_b, dst_o, dst_a,
                       dst_b, scale);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_transpose_tiled(const double *src, double *dst,
                                  int64_t n_outer, int64_t n_a, int64_t n_b,
                                  int64_t src_o, int64_t src_a, int64_t src_b,
                                  const TileMap &m, double scale,
                                  hipStream_t st) {
  if (n_outer <= 0 || n_a <= 0 || n_b <= 0) return hipSuccess;
  const int64_t tiles_a = (n_a + TT - 1) / TT, tiles_b = (n_b + TT - 1) / TT;
  for (int64_t o0 = 0; o0 < n_outer; o0 += 65535) {
    const int64_t no = n_outer - o0 < 65535 ? n_outer - o0 : 65535;
    hipLaunchKernelGGL(transpose_tiled_kernel,
                       dim3((unsigned)(tiles_a * tiles_b), (unsigned)no),
                       dim3(256), 0, st, src, dst, n_a, n_b, tiles_a, o0,
                       src_o, src_a, src_b, m, scale);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_convert(const double *x, const TriGeom &gx,
                          const OpSink &out, const TriGeom &g, bool swapped,
                          int64_t No, hipStream_t st) {
  const int64_t n = fill_rows(out, g) * (g.K >> 3);
  if (n <= 0) return hipSuccess;
  if (g.K % 16 || g.K != gx.K || (swapped && g.nr != No * No))
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(convert_kernel, dim3(fill_blocks(n)), dim3(256), 0, st, x,
                     gx, out, g, swapped, No, n);
  return hipGetLastError();
}

hipError_t launch_synth(DevSystem &s, uint64_t seed, bool with_j,
                        hipStream_t st, int tensor_flag, double scale) {
  const int64_t No = s.No, Nv = s.Nv, N2 = No * No, Nv2 = Nv * Nv;
  hipError_t e = hipSuccess;
  // a doubles operand in the form the system keeps, with its row-swapped
  // copy (xs, tp.sw)
  auto op = [&](double *x, double *xs, const DevSystem::Split &sp,
                const TriOp &tp, bool a, int64_t K, SynthTarget target,
                int tensor) {
    const TriGeom g = s.store == 3 ? (a ? tri_geom_a(No, Nv, K) : tri_geom_b(No, Nv, K))
                                   : (a ? f64_geom_a(No, Nv, K) : f64_geom_b(No, Nv, K));
    for (int sw = 0; sw < 2 && e == hipSuccess; sw++) {
      OpSink k;
      if (s.store == 0) k.d = sw ? xs : x;
      else if (s.store == 3) k.t = sw ? tp.sw : tp.p;
      else if (!sw) { k.h = sp.h; k.l = sp.l; }
      if (!k.d && !k.h && !k.t) continue;
      e = synth_operand(k, g, target, tensor | tensor_flag, seed, s, sw, scale, st);
    }
  };
  auto plain = [&](double *x, int64_t n, int64_t nij, int tensor) {
    if (e == hipSuccess)
      e = synth_plain(x, n, nij, tensor | tensor_flag, seed, s, scale, st);
  };
  op(s.T3, s.T3s, s.sT3, s.tT3, true, s.Kv, S_T3, ATRIP_SYN_TABIJ);
  op(s.V3, nullptr, s.sV3, s.tV3, false, s.Kv, S_V3, ATRIP_SYN_VABCI);
  op(s.H3, s.H3s, s.sH3, s.tH3, true, s.Ko, S_H3, ATRIP_SYN_VIJKA);
  op(s.T2N, nullptr, s.sT2N, s.tT2N, false, s.Ko, S_T2N, ATRIP_SYN_TABIJ);
  op(s.T2TN, nullptr, s.sT2TN, s.tT2TN, false, s.Ko, S_T2TN, ATRIP_SYN_TABIJ);
  plain(s.VHH, Nv2 * N2, N2, ATRIP_SYN_VABIJ);
  plain(s.Tai, Nv * No, 0, ATRIP_SYN_TAI);
  plain(s.ei, No, 0, ATRIP_SYN_EI);
  plain(s.ea, Nv, 0, ATRIP_SYN_EA);
  if (with_j) {
    op(s.V3J, nullptr, s.sV3J, s.tV3J, false, s.Kv, S_V3, ATRIP_SYN_JABCI);
    op(s.H3J, s.H3Js, s.sH3J, s.tH3J, true, s.Ko, S_H3, ATRIP_SYN_JIJKA);
  }
  return e;
}

__global__ __launch_bounds__(256) void scale_kernel(const double *src,
                                                    double *dst, int64_t n,
                                                    double scale) {
  for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < n;
       q += (int64_t)gridDim.x * blockDim.x)
    dst[q] = scale * src[q];
}

hipError_t launch_scale(const double *src, double *dst, int64_t n,
                        double scale, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  int64_t blocks = (n + 255) / 256;
  if (blocks > 65536L * 16) blocks = 65536L * 16;
  hipLaunchKernelGGL(scale_kernel, dim3((unsigned)blocks), dim3(256), 0, st,
                     src, dst, n, scale);
  return hipGetLastError();
}

// One thread per row (k, j) of points and per prefix entry.
__global__ __launch_bounds__(256) void tables_kernel(uint32_t *points,
                                                     uint64_t *prefix,
                                                     int64_t No, int64_t Nv) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  auto tri = [](int64_t n) { return n * (n + 1) * (n + 2) / 6; };
  if (t < No * No) {
    const int64_t k = t / No, j = t % No, m = No - k, d = j - k;
    if (d >= 0) {
      // rows of smaller k, then rows k .. j - 1 of this k (m, m - 1, ... points)
      uint32_t *at = points + (tri(No) - tri(m)) + d * m - d * (d - 1) / 2;
      for (int64_t i = j; i < No; i++)
        at[i - j] = (uint32_t)(i | (j << 10) | (k << 20));
    }
  }
  if (t <= Nv) prefix[t] = (uint64_t)(tri(Nv) - tri(Nv - t) - t);
}

hipError_t launch_tables(const DevSystem &s, hipStream_t st) {
  const int64_t n = std::max(s.No * s.No, s.Nv + 1);
  hipLaunchKernelGGL(tables_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256),
                     0, st, s.points, s.aprefix, s.No, s.Nv);
  return hipGetLastError();
}

}  // namespace atrip_amd
