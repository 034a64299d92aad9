// Internal declarations shared by the HIP translation units of libatrip_hip.
#pragma once

#include <hip/hip_runtime.h>

#include <array>
#include <cstdint>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/atrip_hip.h"

namespace atrip_amd {

// Largest pinned host buffer of a reader upload (bytes).
constexpr int64_t PINNED_MAX = (int64_t)256 << 20;

// Contraction-index padding of the device layouts: every K run of the
// doubles GEMMs is a multiple of the 16-element K chunk of the kernels.
constexpr int KCHUNK = 16;
__host__ __device__ inline int64_t pad16(int64_t n) { return (n + 15) / 16 * 16; }

// bf16x3 operands.  An FP64 operand [o][r < nr][k < K] is held as three
// bf16 parts per element (x ~ b0 + b1 + b2) in tiles of 32 rows x 16 k,
// R = o * nrp + r (nrp: nr, or nr padded to 32 so that every o starts a
// tile row).  Tile (R / 32, k / 16) sits at ((R / 32) (K / 16) + k / 16)
// * 1536 parts; inside it part p of (R, k) sits at 512 p + 8 L + k % 8 with
// L = R % 32 + 32 ((k % 16) / 8), the lane that feeds (R, k) to a 32x32x16
// MFMA, so each part of a 32 x 16 fragment chunk is 1 KiB contiguous in
// lane order (one 16-byte load per lane).  The A operands (nr = No^2 rows
// (p, q)) also keep a row-swapped copy whose row p + No q holds row
// q + No p.
__host__ __device__ inline int64_t pad32(int64_t n) { return (n + 31) / 32 * 32; }
struct TriGeom {
  int64_t no, nr, nrp, K;
  bool swapped;  // keeps a row-swapped copy (A operands)
};
struct TriOp {
  uint16_t *p = nullptr, *sw = nullptr;
};
__host__ __device__ inline int64_t tri_parts(const TriGeom &g) {
  return 3 * pad32(g.no * g.nrp) * g.K;
}
// Start of tile (R / 32, k / 16) and the lane slot of (R, k).
__host__ __device__ inline int64_t tri_tile(int64_t R, int64_t k, int64_t K) {
  return ((R >> 5) * (K >> 4) + (k >> 4)) * 1536;
}
__host__ __device__ inline int tri_lane(int64_t R, int64_t k) {
  return (int)((R & 31) + 32 * ((k & 15) >> 3));
}

// FP64 operands: the same rows R and contraction index k in tiles of 16 rows
// x 8 k, 128 doubles (1 KiB) each, tile (R / 16, k / 8) at
// ((R / 16) (K / 8) + k / 8) * 128; inside it (R, k) sits at
// 32 ((k % 8) / 2) + 2 (R % 16) + k % 2: lane (R % 16) + 16 ((k % 8) / 2) of
// a 16x16x4 MFMA fragment owns the two k of its 16 bytes, so a fragment's
// 8-deep K step is one 16-byte load per lane over 1 KiB of consecutive
// addresses (8 lines of 128 bytes; rows K apart cost 64 lines).  The A
// operands (rows (p, q), padded to whole tiles per o) keep a row-swapped
// copy like the bf16x3 ones.
__host__ __device__ inline int64_t f64_row(int64_t R, int64_t K) {
  return (R >> 4) * (K >> 3) * 128 + 2 * (R & 15);
}
__host__ __device__ inline int64_t f64_at(int64_t R, int64_t k, int64_t K) {
  return f64_row(R, K) + (k >> 3) * 128 + 32 * ((k & 7) >> 1) + (k & 1);
}
__host__ __device__ inline int64_t f64_elems(const TriGeom &g) {
  return pad16(g.no * g.nrp) * g.K;
}

// Layout of the per-tuple class buffers written by the doubles kernels and
// read by the energy kernels: blocks of 8 x 8 x 8 elements of the GEMM output
// (row m = p + No q, column r), element (p, q, r) at block
// ((q / 8) nbk + p / 8) nbk + r / 8, inside it 64 (q % 8) + 8 (p % 8) + r % 8;
// in W indices
//   class w: (p, q, r) = (i, j, k)
//   class v: (p, q, r) = (i, k, j)
//   class u: (p, q, r) = (j, k, i)
// so the 8^3 block of W an epilogue workgroup needs is one run of 4 KiB (FP64;
// 2 KiB FP32) in each class, where a GEMM-ordered buffer held it in 64 pieces
// of 64 bytes, one request each.  Elements past No are neither written nor
// read.
// Edge of the blocks (of the class buffers, and of W in LDS).
constexpr int WCUBE = 8;
__host__ __device__ inline int64_t w_blocks(int64_t No) {
  return (No + WCUBE - 1) / WCUBE;
}
// Elements of one tuple's class buffer.
__host__ __device__ inline int64_t g_elems(int64_t No) {
  const int64_t n = w_blocks(No) * WCUBE;
  return n * n * n;
}
// Elements of it in GEMM order, each row padded to a 64-byte line: what the
// allocation-free region is counted in.
inline int64_t g_row_elems(int64_t No, bool g32) {
  const int64_t q = g32 ? 16 : 8;
  return No * No * ((No + q - 1) / q * q);
}
// Offset of a GEMM row and of a GEMM column in it.
struct GLayout {
  uint32_t No, nbk, magic;  // magic: ceil(2^32 / No), exact for rows < No^2
};
inline GLayout g_layout(int64_t No) {
  return {(uint32_t)No, (uint32_t)w_blocks(No),
          No == 1 ? 0u : (uint32_t)((((uint64_t)1 << 32) + No - 1) / No)};
}
__device__ __forceinline__ uint32_t g_row(const GLayout &L, uint32_t m) {
  const uint32_t q = L.No == 1 ? m : __umulhi(m, L.magic), p = m - q * L.No;
  return (((q >> 3) * L.nbk + (p >> 3)) * L.nbk << 9) + ((q & 7) << 6) +
         ((p & 7) << 3);
}
__device__ __forceinline__ uint32_t g_col(uint32_t r) {
  return ((r >> 3) << 9) + (r & 7);
}
// Largest one-dimensional grid a launch takes (workgroups); launchers
// refuse larger ones instead of truncating the count.
constexpr int64_t MAX_GRID = 0xFFFFFFFFLL;
// Doubles of one tuple's W in the cube layout the energy kernels read: the
// occupied range padded to whole cubes, cube (bx, by, bz) at
// ((bz nbk + by) nbk + bx) * 512, element x + 8 y + 64 z inside.
__host__ __device__ inline int64_t w_cube(int64_t No) {
  const int64_t n = w_blocks(No) * WCUBE;
  return n * n * n;
}
// Block triples B1 >= B2 >= B3 over nbk blocks per index.
__host__ __device__ inline int64_t n_triples(int64_t nbk) {
  return nbk * (nbk + 1) * (nbk + 2) / 6;
}

// Whether the fused epilogue does a tuple in one wave or workgroup: up to the No
// whose W (two with (cT)) fits 160 KB of LDS, from FP64 buffers alone up to 18.
// Energies by block triples -> by tuples, ms: FP64 No=4, Nv=36 .052 -> .015,
// 10/90 2.55 -> 1.06, 16/80 2.32 -> 1.83, 18/80 5.58 -> 3.87, 20/80 5.82 -> 5.99
// (one workgroup a CU, or spills); (cT) 20/60 4.93 -> 4.38; bf16x3 16/80 2.03
// -> 1.48, 20/80 5.34 -> 3.06.
__host__ __device__ inline bool small_energy(int64_t No, bool use_j, bool g32) {
  return No <= (use_j || g32 ? 20 : 18);
}
// Dynamic LDS those kernels are allowed (the same for every launch, so that
// threads do not undo each other's); the largest use is 155,200 bytes.
constexpr int MAX_LDS = 156 * 1024;
// The same for complex systems, whose two planes of W (four with (cT)) fit 160 KB.
__host__ __device__ inline bool small_energy_z(int64_t No, bool use_j) {
  return No <= (use_j ? 16 : 20);
}
// Partial energies of a real tuple in it: one, or one per block triple.
__host__ __device__ inline int64_t energy_parts(int64_t No, bool use_j,
                                                bool g32) {
  return small_energy(No, use_j, g32) ? 1 : n_triples(w_blocks(No));
}

// Device-resident system.  Pair-indexed arrays use the CTF pair order
// p(x,y) = x + Nv*y.  The doubles operands, as rows times contraction index:
//   T3  [x][p + No q][E < Kv]    = Tpphh[x,E,p,q]          (T(x) slices)
//   V3  [p(x,y)][r][E < Kv]      = Vppph[x,y,E,r]          (V(xy) slices)
//   H3  [x][p + No q][L < Ko]    = Vhhhp[p,q,L,x]          (Vhhh(x) slices)
//   T2N [p(x,y)][n][L < Ko]      = -Tpphh[x,y,L,n]         (-T(xy)[L,n])
//   T2TN[p(x,y)][n][L < Ko]      = -Tpphh[x,y,n,L]         (-T(xy)[n,L])
// in FP64 as 16 x 8 tiles (f64_at); T3s, H3s hold row q + No p in row
// p + No q (null when they found no memory: the kernels then read the
// swapped rows from T3, H3).  The other arrays, last index fastest:
//   VHH [p(x,y)][i + No j]       = Vpphh[x,y,i,j]          (V(xy)ij)
//   Tai [a + Nv i], ei[i], ea[a] as in CTF.
// Padding entries (E >= Nv, L >= No, rows past No^2) are zero.
struct DevSystem {
  int64_t No = 0, Nv = 0, Kv = 0, Ko = 0;
  double *T3 = nullptr, *V3 = nullptr, *H3 = nullptr, *T2N = nullptr,
         *T2TN = nullptr, *VHH = nullptr, *Tai = nullptr, *ei = nullptr,
         *ea = nullptr;
  double *T3s = nullptr, *H3s = nullptr;  // row-swapped copies of T3, H3
  double *V3J = nullptr, *H3J = nullptr;  // (cT) integrals, may be null
  double *H3Js = nullptr;
  bool has_j = false;                     // (cT) integrals present
  // Complex systems: the arrays above hold the real parts, these the
  // imaginary parts (same layouts), and the *n arrays the negated imaginary
  // parts of T3 and the hole integrals (operands of the real-GEMM passes).
  bool cplx = false;
  double *T3i = nullptr, *V3i = nullptr, *H3i = nullptr, *T2Ni = nullptr,
         *T2TNi = nullptr, *VHHi = nullptr, *Taii = nullptr, *eii = nullptr,
         *eai = nullptr, *V3Ji = nullptr, *H3Ji = nullptr;
  double *T3is = nullptr, *H3is = nullptr, *H3Jis = nullptr;
  double *T3in = nullptr, *H3in = nullptr, *H3Jin = nullptr;
  double *T3ins = nullptr, *H3ins = nullptr, *H3Jins = nullptr;
  // Split-FP32 copies of the GEMM operands, made on the first mixed run:
  // h = (float)x and l = bf16(x - h), same layouts as above (bf16(h), the
  // other factor of the correction products, is formed in registers).
  struct Split {
    float *h = nullptr;
    uint16_t *l = nullptr;
  };
  Split sT3, sV3, sH3, sT2N, sT2TN, sV3J, sH3J;
  bool split_ready = false;
  // bf16x3 copies in the tiled layout (TriGeom): T3 and H3 rows padded to
  // 32 per slice with row-swapped copies, the pair-indexed arrays unpadded.
  TriOp tT3, tV3, tH3, tT2N, tT2TN, tV3J, tH3J;
  bool tri_ready = false;
  // Operand store: 0 FP64 (split or bf16x3 copies made on the first mixed
  // run of that form), 1 split FP32 only (h + l, 6 bytes per element), 2
  // FP32 (h) only, 3 bf16x3 only (6 bytes per element).  Modes 1-3 keep no
  // FP64 copy of the doubles operands (T3, V3, H3, T2N, T2TN and the J
  // arrays).
  int store = 0;
  uint32_t *points = nullptr;             // packed (i>=j>=k) triples
  int64_t npoints = 0;
  uint64_t *aprefix = nullptr;            // tuples with first index < a
  uint64_t bytes = 0;
  std::vector<void *> allocations;
  void *block = nullptr, *swaps = nullptr;  // all arrays; the swapped copies
  size_t block_bytes = 0, swap_bytes = 0;
  enum { NONE, COUNT, PLACE } laying = NONE;  // (see dev_bytes)
};

// bf16 of a float, round to nearest even (finite inputs).
__device__ inline uint16_t to_bf16(float v) {
  uint32_t u = __float_as_uint(v);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

// A conversion works on octets: the eight k of one row that share an FP64
// tile (and one lane slot of a bf16x3 tile).
//
// bf16x3 parts of the octet v into row R, k = k8 of a tiled copy:
// b0 = bf16(x), b1 = bf16(x - b0), b2 = bf16(x - b0 - b1), each residual
// formed in FP64, so b0 + b1 + b2 is x within 2^-27 |x|.
__device__ inline void tri_put8(const double (&v)[8], uint16_t *out, int64_t R,
                                int64_t k8, int64_t K) {
  typedef uint16_t u8 __attribute__((ext_vector_type(8)));
  u8 p0, p1, p2;
#pragma unroll
  for (int e = 0; e < 8; e++) {
    p0[e] = to_bf16((float)v[e]);
    const double r1 = v[e] - (double)__uint_as_float((uint32_t)p0[e] << 16);
    p1[e] = to_bf16((float)r1);
    const double r2 = r1 - (double)__uint_as_float((uint32_t)p1[e] << 16);
    p2[e] = to_bf16((float)r2);
  }
  uint16_t *at = out + tri_tile(R, k8, K) + 8 * tri_lane(R, k8);
  *(u8 *)at = p0;
  *(u8 *)(at + 512) = p1;
  *(u8 *)(at + 1024) = p2;
}

// Split-FP32 octet: h = (float)x, l = bf16(x - h), row-major at element q;
// l may be null (FP32-only store).
__device__ inline void split_put8(const double (&v)[8], float *h, uint16_t *l,
                                  int64_t q) {
  typedef uint16_t u8 __attribute__((ext_vector_type(8)));
  typedef float f8 __attribute__((ext_vector_type(8)));
  f8 hi;
  u8 lo;
#pragma unroll
  for (int e = 0; e < 8; e++) {
    hi[e] = (float)v[e];
    lo[e] = to_bf16((float)(v[e] - (double)hi[e]));
  }
  *(f8 *)(h + q) = hi;
  if (l) *(u8 *)(l + q) = lo;
}

// FP64 octet into row R, k = k8 of a tiled operand.
__device__ inline void f64_put8(const double (&v)[8], double *out, int64_t R,
                                int64_t k8, int64_t K) {
  typedef double d2 __attribute__((ext_vector_type(2)));
  double *at = out + f64_at(R, k8, K);
#pragma unroll
  for (int q = 0; q < 4; q++) *(d2 *)(at + 32 * q) = d2{v[2 * q], v[2 * q + 1]};
}

// One form of a doubles operand being filled: FP64 tiles, split FP32 rows
// and / or bf16x3 tiles (null: not kept).
struct OpSink {
  double *d = nullptr;
  float *h = nullptr;
  uint16_t *l = nullptr, *t = nullptr;
};
__device__ inline void sink_put8(const double (&v)[8], const OpSink &s,
                                 const TriGeom &g, int64_t o, int64_t r,
                                 int64_t k8) {
  const int64_t R = o * g.nrp + r;
  if (s.d) f64_put8(v, s.d, R, k8, g.K);
  if (s.h && r < g.nr && o < g.no)
    split_put8(v, s.h, s.l, (o * g.nr + r) * g.K + k8);
  if (s.t) tri_put8(v, s.t, R, k8, g.K);
}

// Tuple windows of a system: block triples (alpha <= beta <= gamma) of edge
// nb in lexicographic order.
struct WindowPlan {
  int nb = 0;
  std::vector<int32_t> origin;   // (a0, b0, c0) per window
  std::vector<uint64_t> wcount;  // tuples per window
};

struct KernelStat {
  uint64_t launches = 0;
  double ms = 0.0;
  double flop = 0.0;
};

struct Batch;

// Tuned plan of the batched form for one system shape.
struct BatchTune {
  int nb = 1, tile = 0;
  double sec_window = 0.0;  // measured (or modelled) time of a full window
  bool measured = false;
};

}  // namespace atrip_amd

struct atrip_hip_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  std::string err;
  std::map<int, atrip_amd::DevSystem> systems;
  std::map<int, atrip_amd::WindowPlan> plans;  // keyed by system
  int next_sys = 1;
  // options
  int window = 0;  // window edge; 0: automatic per system (auto_window)
  int batch = 0;   // windows per launch; 0: automatic (auto_batch)
  int timing = 0;
  int tile = -1;  // -1: chosen per system shape
  int operand_store = 0;  // store mode of the next uploads (DevSystem::store)
  bool operand_swaps = true;  // uploads keep row-swapped copies (FP64 store)
  int epilogue = 0;  // 0: fused class sums + energy, 1: W cubes first
  int serve_plain_no = 16;  // served requests with No >= this: plain path
  int64_t stage_kb = 4 << 20;  // device staging of host uploads (KiB)
  // Held while device work of a call uses the systems' arrays and the scratch
  // below, so that a call of another context may give back what this one can
  // do without (give_back); never while a callback of the caller runs.
  std::mutex in_use;
  // scratch, grown on demand
  double *G = nullptr;       // class buffers [ncls][slots][g_elems(No)]
  size_t G_bytes = 0;
  double *wcube = nullptr;   // W as cubes for the energy kernels
  size_t wcube_bytes = 0;
  double *e_slot = nullptr;  // per-slot energies (2 per slot: e, e_ct)
  size_t e_slot_bytes = 0;
  double *partials = nullptr;  // (sum, comp) x 2 per 256 slots of a run
  size_t partials_bytes = 0;
  void *sel = nullptr;  // a run's window list (and per-window sums)
  size_t sel_bytes = 0;
  // batched form: tuned plans keyed by (No, padded Nv, precision),
  // workgroup scratch
  std::map<std::array<int64_t, 3>, atrip_amd::BatchTune> btune;
  double *bscratch = nullptr;
  size_t bscratch_bytes = 0;
  int64_t batch_scratch_mb = 8192;
  int batch_grid = 0;   // 0: occupancy x CUs
  int batch_order = 0;  // 0: longest window first, 1: canonical
  int batch_nb = 0;     // forced window edge of the batched form (0: tuned)
  int batch_tile = -1;  // forced tile variant of the batched form (-1: tuned)
  std::map<std::string, atrip_amd::KernelStat> stats;
  std::vector<std::pair<hipEvent_t, hipEvent_t>> pending_events;
  std::vector<std::string> pending_names;
  std::vector<double> pending_flop;
};

namespace atrip_amd {

// ---- launch wrappers (one translation unit each) -----------------------

// Batch of consecutive windows handed to the hot kernels: window w holds the
// tuples (a0 + ta, b0 + tb, c0 + tc), ta < ea, tb < eb, tc < ec, from its
// origin (a0, b0, c0) at windows[3 w]; slot (ta eb + tb) ec + tc of window w
// is slot w ea eb ec + that of the batch.
struct WindowArgs {
  const int32_t *windows;   // device, 3 per window of this batch
  const uint64_t *aprefix;  // of the system (tuple_index)
  uint64_t first, last;     // canonical tuple range [first, last)
  int nw;                   // windows in the batch
  int ea, eb, ec;           // window edges, at most 32
  int mtiles, ntiles;       // tiles of a pair's GEMM (set by the launchers)
};
struct BatchArgs : WindowArgs {
  int64_t slots;  // nw * ea * eb * ec
};
// Tuple of batch slot gs, false outside the range or the ordered tuples.
__device__ __forceinline__ bool slot_tuple(const WindowArgs &W, uint64_t Nv,
                                           uint32_t gs, int64_t &a, int64_t &b,
                                           int64_t &c);

// Doubles contractions in FP64 MFMA: class buffers G[3][slots][g_elems(No)].
// With s2 its four products are added to those of s (same shape) in the same
// GEMM: one plane of a complex product.
hipError_t launch_doubles_f64(const DevSystem &s, const DevSystem *s2,
                              const BatchArgs &b, bool use_j, double *G,
                              int tile, hipStream_t st);

// Doubles contractions with FP32 products (class buffers in FP32): split FP32
// (with the hi*lo + lo*hi corrections), and FP32 only.
hipError_t launch_doubles_split(const DevSystem &s, const BatchArgs &b,
                                bool use_j, float *G, int tile, hipStream_t st);
hipError_t launch_doubles_fp32(const DevSystem &s, const BatchArgs &b,
                               bool use_j, float *G, int tile, hipStream_t st);

// Doubles contractions in bf16x3 (six part products on bf16 MFMA, FP32
// accumulation, class buffers in FP32).
hipError_t launch_doubles_tri(const DevSystem &s, const BatchArgs &b,
                              bool use_j, float *G, int tile, hipStream_t st);

// Class sums: out[slot] = sum(A) as cubes (w_cube per slot), for class-buffer
// set A (FP64, or FP32 when g32).
hipError_t launch_wsum(const DevSystem &s, const BatchArgs &b, const void *A,
                       bool g32, double *out, hipStream_t st);

// Class sums and singles + energy epilogue.  fused: one kernel gathers each
// block triple's W straight from the class buffers and writes the triple's
// energies to scratch ([triple][slot][2], slots * energy_parts * 2 doubles),
// which launch_slot_sums adds up (small No: a whole tuple at once); otherwise the class-sum kernel writes W as
// cubes first (scratch: (GJ ? 2 : 1) * slots * w_cube(No) doubles) and
// e_slot[2*slot + {0,1}] is written here.  Same W bits either way.
hipError_t launch_energy(const DevSystem &s, const BatchArgs &b,
                         const void *G, const void *GJ, bool g32,
                         double tai_sign, double *e_slot, double *scratch,
                         bool fused, hipStream_t st);
// Doubles of energy scratch per tuple slot (see launch_energy).
inline int64_t energy_scratch_per_slot(int64_t No, bool use_j, bool g32,
                                       bool cplx, bool fused) {
  if (fused && !cplx) return 2 * energy_parts(No, use_j, g32);
  if (fused && small_energy_z(No, use_j)) return 1;  // none needed
  return (use_j ? 2 : 1) * (cplx ? 2 : 1) * w_cube(No);
}

// Singles + energy of complex systems from the class-buffer sets of W's real
// and imaginary plane; GJ null without (cT).
// fused: straight from the buffers where small_energy_z holds; otherwise by
// cubes, wcube: scratch of (GJ ? 4 : 2) * slots * w_cube(No) doubles.
hipError_t launch_energy_z(const DevSystem &s, const BatchArgs &b,
                           double *const G[2], double *const GJ[2],
                           double tai_sign, double *e_slot, double *wcube,
                           bool fused, hipStream_t st);

// The points table of a system (i >= j >= k, packed 10 bits per index, k
// slowest) and its prefix table (tuples with a smaller first index).
hipError_t launch_tables(const DevSystem &s, hipStream_t st);
// Per window of a batch (nw windows of `per` slots), a compensated sum of
// its slot energies in a fixed order: out[2 w] = sum, out[2 w + 1] =
// compensation.
hipError_t launch_window_sums(const double *e_slot, int nw, int64_t per,
                              double *out, hipStream_t st);

// Slot energies from the triples' partials (e_part null: e_slot holds them)
// and their compensated sums, one quadruple {sum, comp, sum_ct, comp_ct} of
// partials per 256 slots.
hipError_t launch_slot_sums(const double *e_part, int64_t slots, int64_t ntri,
                            double *e_slot, double *partials, hipStream_t st);
inline int64_t slot_partials(int64_t slots) { return (slots + 255) / 256; }

// Upload helpers.
hipError_t launch_transpose(const double *src, double *dst, int64_t n_outer,
                            int64_t n_a, int64_t n_b, int64_t src_o,
                            int64_t src_a, int64_t src_b, int64_t dst_o,
                            int64_t dst_a, int64_t dst_b, double scale,
                            hipStream_t st);
// The same copy into an FP64 operand's tiles: element (o, a, b) goes to row
// R0 + o Ro + a Ra + b Rb at contraction index k0 + o ko + a ka.  swap 1:
// the row part of R is row0 + o, swap 2: it is b, and the element goes to
// the swapped row q + No p instead of p + No q (R: the other parts).
struct TileMap {
  int64_t R0 = 0, Ro = 0, Ra = 0, Rb = 0, k0 = 0, ko = 0, ka = 0, K = 0;
  int swap = 0;
  int64_t row0 = 0, No = 1;
};
hipError_t launch_transpose_tiled(const double *src, double *dst,
                                  int64_t n_outer, int64_t n_a, int64_t n_b,
                                  int64_t src_o, int64_t src_a, int64_t src_b,
                                  const TileMap &m, double scale,
                                  hipStream_t st);
// Generate a synthetic system in place; tensor_flag is or-ed into every
// tensor id (ATRIP_SYN_IMAG fills the imaginary parts of a complex system,
// given a DevSystem whose arrays are its imaginary planes).
// Every amplitude and integral value is multiplied by `scale` (orbital
// energies are not).
hipError_t launch_synth(DevSystem &s, uint64_t seed, bool with_j,
                        hipStream_t st, int tensor_flag = 0,
                        double scale = 1.0);
// dst[q] = scale * src[q], q < n.
hipError_t launch_scale(const double *src, double *dst, int64_t n,
                        double scale, hipStream_t st);
// Fill another form of FP64 operand x (geometry gx) of geometry g, in g's
// row order or, swapped, with row q + No p in row p + No q.
hipError_t launch_convert(const double *x, const TriGeom &gx,
                          const OpSink &out, const TriGeom &g, bool swapped,
                          int64_t No, hipStream_t st);
// Geometry of a system's FP64 operands: A (T3, H3 and H3J, rows padded to
// whole tiles) and the pair-indexed B arrays (V3, T2N, T2TN, V3J).
inline TriGeom f64_geom_a(int64_t No, int64_t Nv, int64_t K) {
  return TriGeom{Nv, No * No, pad16(No * No), K, true};
}
inline TriGeom f64_geom_b(int64_t No, int64_t Nv, int64_t K) {
  return TriGeom{Nv * Nv, No, No, K, false};
}
// Geometry of a system's bf16x3 operands: A (T3, H3 and H3J) and the
// pair-indexed B arrays (V3, T2N, T2TN, V3J), for contraction length K.
inline TriGeom tri_geom_a(int64_t No, int64_t Nv, int64_t K) {
  return TriGeom{Nv, No * No, pad32(No * No), K, true};
}
inline TriGeom tri_geom_b(int64_t No, int64_t Nv, int64_t K) {
  return TriGeom{Nv * Nv, No, No, K, false};
}
inline uint64_t tri_bytes(const TriGeom &g) {
  return (uint64_t)tri_parts(g) * 2 * (g.swapped ? 2 : 1);
}

// ---- batched form: many small resident systems in one persistent launch --

// One system of a batched launch, with the window edge and tile variant
// chosen for it.  Tile variant v is the wave tile of (16*bfm(v)) x
// (16*bfn(v)) outputs.
struct BSys {
  const double *T3, *T3s, *V3, *H3, *H3s, *T2N, *T2TN, *VHH, *Tai, *ei, *ea;
  const uint32_t *points;
  int64_t No, Nv, Kv, Ko, npoints;
  int32_t nb, tile;
};
constexpr int N_BTILES = 10;
constexpr __host__ __device__ inline int bfm(int v) {
  constexpr int t[N_BTILES] = {1, 1, 2, 2, 1, 4, 2, 4, 3, 3};
  return t[v];
}
constexpr __host__ __device__ inline int bfn(int v) {
  constexpr int t[N_BTILES] = {1, 2, 1, 2, 4, 1, 4, 2, 2, 3};
  return t[v];
}

// The smallest tile variant within `tile` holding its nr x nc fragments inside
// the GEMM, for a tile at the edge.
__host__ __device__ inline int fitting_tile(int tile, int nr, int nc) {
  int best = bfm(tile) * bfn(tile), v = tile;
#pragma unroll
  for (int t = 0; t < N_BTILES; t++)
    if (bfm(t) >= nr && bfm(t) <= bfm(tile) && bfn(t) >= nc &&
        bfn(t) <= bfn(tile) && bfm(t) * bfn(t) < best) {
      best = bfm(t) * bfn(t);
      v = t;
    }
  return v;
}

// Split-FP32 operands of a system in a batched launch (h = FP32 values,
// l = bf16(x - h); l unused by the FP32-only form).
struct BSplit {
  const float *T3h, *V3h, *H3h, *T2Nh, *T2TNh;
  const uint16_t *T3l, *V3l, *H3l, *T2Nl, *T2TNl;
};

// One work item: a window (block triple of edge nb) of one system.
struct BTask {
  int32_t sys, al, be, ga;
  int64_t tuple_off;  // first entry of the task's slots in the per-tuple output
};

struct BatchedLaunch {
  int precision;            // ATRIP_FP64, ATRIP_SPLIT_FP32 or ATRIP_FP32
  const BSys *sys;          // device
  const BSplit *split;      // device, one per system (mixed forms only)
  const BTask *tasks;       // device, canonical order (system-major)
  const int32_t *order;     // device, dispatch order (a permutation)
  int ntasks;
  unsigned *counter;        // device, zero before the launch
  double *scratch;          // grid * scratch_stride doubles
  int64_t scratch_stride;
  double *task_e;           // 2 per task: (sum, compensation)
  double *tuple_e;          // optional per-slot energies
  int grid;
};

// Persistent launch: every workgroup takes windows from the dispatch order
// until none is left; doubles, singles and energy of a window stay in the
// workgroup.
hipError_t launch_batched(const BatchedLaunch &L, hipStream_t st);
// Workgroups per CU the persistent kernel of a precision can hold.
int batched_blocks_per_cu(int precision);
// Canonical (lexicographic) index of tuple (a,b,c), a<=b<=c, not all equal.
__host__ __device__ inline uint64_t tuple_index(const uint64_t *aprefix,
                                                uint64_t Nv, uint64_t a,
                                                uint64_t b, uint64_t c) {
  // tuples (a, b', c') with a <= b' < b: sum_{b'=a}^{b-1} (Nv - b')
  const uint64_t nb = b - a;
  const uint64_t before_b = nb * Nv - (nb * (a + b - 1)) / 2;
  return aprefix[a] + before_b - (b > a ? 1 : 0) + (c - b) - (a == b ? 1 : 0);
}

__host__ __device__ inline bool tuple_ok(uint64_t Nv, uint64_t a, uint64_t b,
                                         uint64_t c) {
  return a <= b && b <= c && c < Nv && !(a == b && b == c);
}

// (32-bit arithmetic: a 64-bit division is ~130 scalar instructions)
__device__ __forceinline__ bool slot_tuple(const WindowArgs &W, uint64_t Nv,
                                           uint32_t gs, int64_t &a, int64_t &b,
                                           int64_t &c) {
  const uint32_t ebc = (uint32_t)(W.eb * W.ec), per = ebc * (uint32_t)W.ea;
  const uint32_t w = gs / per, s = gs - w * per;
  const uint32_t ta = s / ebc, r = s - ta * ebc;
  const uint32_t tb = r / (uint32_t)W.ec, tc = r - tb * (uint32_t)W.ec;
  a = W.windows[3 * w] + (int64_t)ta;
  b = W.windows[3 * w + 1] + (int64_t)tb;
  c = W.windows[3 * w + 2] + (int64_t)tc;
  if (!tuple_ok(Nv, a, b, c)) return false;
  if (W.first == 0 && W.last == ~0ULL) return true;
  const uint64_t idx = tuple_index(W.aprefix, Nv, a, b, c);
  return idx >= W.first && idx < W.last;
}

}  // namespace atrip_amd
