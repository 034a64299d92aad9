// C-ABI of the MI355X (T) hot path: contexts, resident systems, the tuple
// window scheduler and the run loop.  See include/atrip_hip.h.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <string>
#include <type_traits>
#include <vector>

#include "doubles_common.hpp"
#include "host.hpp"
#include "../../include/atrip_synth.h"

using namespace atrip_amd;

DevSystem &atrip_amd::get_sys(atrip_hip_ctx *ctx, int sys) {
  auto it = ctx->systems.find(sys);
  if (it == ctx->systems.end()) throw Fail{"unknown system handle"};
  return it->second;
}

namespace {
void *dev_bytes(DevSystem &s, size_t bytes, const char *what);
// Tiled bf16x3 copy (and row-swapped copy) of geometry g; its fill writes
// every element, padding included.
void alloc_tri(DevSystem &s, TriOp &o, const TriGeom &g, const char *what) {
  const size_t bytes = (size_t)tri_parts(g) * 2;
  o.p = (uint16_t *)dev_bytes(s, bytes, what);
  if (g.swapped) o.sw = (uint16_t *)dev_bytes(s, bytes, what);
}

// Copies of a system's operands that a failure part-way gives back whole.
struct CopyGuard {
  DevSystem &s;
  size_t n;
  uint64_t bytes;
  bool done = false;
  explicit CopyGuard(DevSystem &s_)
      : s(s_), n(s_.allocations.size()), bytes(s_.bytes) {}
  ~CopyGuard() {
    if (done) return;
    for (size_t q = n; q < s.allocations.size(); q++)
      (void)hipFree(s.allocations[q]);
    s.allocations.resize(n);
    s.bytes = bytes;
  }
};

// FP64 operand x of a system in its split form, or its bf16x3 form with the
// row-swapped copy.
void convert_split(const DevSystem &s, const double *x, const TriGeom &g,
                   const DevSystem::Split &o, hipStream_t st) {
  OpSink k;
  k.h = o.h;
  k.l = o.l;
  check(launch_convert(x, g, k, g, false, s.No, st), "split conversion");
}
void convert_tri(const DevSystem &s, const double *x, const TriGeom &gx,
                 const TriOp &o, const TriGeom &g, hipStream_t st) {
  for (uint16_t *p : {o.p, o.sw}) {
    if (!p) continue;
    OpSink k;
    k.t = p;
    check(launch_convert(x, gx, k, g, p == o.sw, s.No, st),
          "bf16x3 conversion");
  }
}
}

// Split-FP32 copies of the GEMM operands, made once per system on the first
// mixed-precision run.
void atrip_amd::ensure_split(atrip_hip_ctx *ctx, DevSystem &s) {
  if (s.split_ready) return;
  const int64_t No = s.No, Nv = s.Nv;
  const TriGeom ga = f64_geom_a(No, Nv, s.Kv), gb = f64_geom_b(No, Nv, s.Kv),
                gh = f64_geom_a(No, Nv, s.Ko), gt = f64_geom_b(No, Nv, s.Ko);
  CopyGuard guard(s);
  auto make = [&](const double *x, DevSystem::Split &o, const TriGeom &g) {
    if (!x) return;
    const size_t n = (size_t)(g.no * g.nr * g.K);
    o.h = (float *)dev_bytes(s, n * sizeof(float), "alloc split");
    o.l = (uint16_t *)dev_bytes(s, n * 2, "alloc split");
    convert_split(s, x, g, o, ctx->stream);
  };
  make(s.T3, s.sT3, ga);
  make(s.V3, s.sV3, gb);
  make(s.H3, s.sH3, gh);
  make(s.T2N, s.sT2N, gt);
  make(s.T2TN, s.sT2TN, gt);
  make(s.V3J, s.sV3J, gb);
  make(s.H3J, s.sH3J, gh);
  check(hipStreamSynchronize(ctx->stream), "split conversion");
  guard.done = true;
  s.split_ready = true;
}

void atrip_amd::check_precision(const DevSystem &s, int precision) {
  if (precision != ATRIP_FP64 && precision != ATRIP_SPLIT_FP32 &&
      precision != ATRIP_FP32 && precision != ATRIP_BF16X3)
    throw Fail{"unknown precision " + std::to_string(precision)};
  if (s.cplx && precision != ATRIP_FP64)
    throw Fail{"complex systems run in FP64 only"};
  if (precision == ATRIP_FP64 && s.store != 0)
    throw Fail{"system was uploaded without FP64 operands (operand_store)"};
  if (precision == ATRIP_SPLIT_FP32 && (s.store == 2 || s.store == 3))
    throw Fail{"system was uploaded without split operands (operand_store " +
               std::to_string(s.store) + ")"};
  if (precision == ATRIP_FP32 && s.store == 3)
    throw Fail{"system was uploaded with bf16x3 operands only (operand_store 3)"};
  if (precision == ATRIP_BF16X3 && s.store != 0 && s.store != 3)
    throw Fail{"system was uploaded without bf16x3 operands (operand_store " +
               std::to_string(s.store) + ")"};
}

// bf16x3 copies of the GEMM operands, made once per system on the first
// bf16x3 run.
void atrip_amd::ensure_tri(atrip_hip_ctx *ctx, DevSystem &s) {
  if (s.tri_ready) return;
  const int64_t No = s.No, Nv = s.Nv;
  CopyGuard guard(s);
  auto make = [&](const double *x, TriOp &o, bool a, int64_t K) {
    if (!x) return;
    const TriGeom g = a ? tri_geom_a(No, Nv, K) : tri_geom_b(No, Nv, K);
    alloc_tri(s, o, g, "alloc bf16x3");
    convert_tri(s, x, a ? f64_geom_a(No, Nv, K) : f64_geom_b(No, Nv, K), o, g,
                ctx->stream);
  };
  make(s.T3, s.tT3, true, s.Kv);
  make(s.V3, s.tV3, false, s.Kv);
  make(s.H3, s.tH3, true, s.Ko);
  make(s.T2N, s.tT2N, false, s.Ko);
  make(s.T2TN, s.tT2TN, false, s.Ko);
  make(s.V3J, s.tV3J, false, s.Kv);
  make(s.H3J, s.tH3J, true, s.Ko);
  check(hipStreamSynchronize(ctx->stream), "bf16x3 conversion");
  guard.done = true;
  s.tri_ready = true;
}

namespace {

double *dev_alloc(DevSystem &s, int64_t n, const char *what) {
  return (double *)dev_bytes(s, (size_t)std::max<int64_t>(n, 1) * sizeof(double),
                             what);
}

// The row-swapped copies of a system's FP64 A operands and the copies they
// belong to, with their contraction lengths.
struct SwapCopy {
  double **copy, *from;
  int64_t K;
};
std::vector<SwapCopy> swap_copies(DevSystem &s) {
  std::vector<SwapCopy> v;
  auto add = [&](double *&copy, double *from, int64_t K) {
    if (from) v.push_back({&copy, from, K});
  };
  add(s.T3s, s.T3, s.Kv);
  add(s.H3s, s.H3, s.Ko);
  add(s.H3Js, s.H3J, s.Ko);
  add(s.T3is, s.T3i, s.Kv);
  add(s.H3is, s.H3i, s.Ko);
  add(s.H3Jis, s.H3Ji, s.Ko);
  add(s.T3ins, s.T3in, s.Kv);
  add(s.H3ins, s.H3in, s.Ko);
  add(s.H3Jins, s.H3Jin, s.Ko);
  return v;
}

// Allocates the row-swapped copies as one block if it fits; without memory they
// stay null and the kernels read the swapped rows from the straight array.
void alloc_swaps(DevSystem &s) {
  const std::vector<SwapCopy> copies = swap_copies(s);
  size_t bytes = 0;
  for (const SwapCopy &c : copies)
    bytes += (size_t)f64_elems(f64_geom_a(s.No, s.Nv, c.K)) * sizeof(double);
  void *p = nullptr;
  if (hipMalloc(&p, bytes) != hipSuccess) {
    (void)hipGetLastError();
    return;
  }
  s.allocations.push_back(p);
  s.bytes += bytes;
  s.swaps = p;
  s.swap_bytes = bytes;
  char *at = (char *)p;
  for (const SwapCopy &c : copies) {  // (whole 2 KB tiles: aligned)
    *c.copy = (double *)at;
    at += (size_t)f64_elems(f64_geom_a(s.No, s.Nv, c.K)) * sizeof(double);
  }
}

// Zeroes the arrays of a system whose upload leaves the padding of its FP64
// operands unwritten.
void clear_operands(DevSystem &s, hipStream_t st) {
  if (s.store != 0) return;
  check(hipMemsetAsync(s.block, 0, s.block_bytes, st), "clear operands");
  if (s.swaps) check(hipMemsetAsync(s.swaps, 0, s.swap_bytes, st), "clear operands");
}

// Device memory of a system: while alloc_system lays it out a piece of its one
// block (first counted, then placed), later allocations of their own.
void *dev_bytes(DevSystem &s, size_t bytes, const char *what) {
  bytes = std::max<size_t>(bytes, 1);
  if (s.laying != DevSystem::NONE) {
    const size_t at = s.block_bytes;
    s.block_bytes += (bytes + 255) / 256 * 256;
    if (s.laying == DevSystem::COUNT) return nullptr;
    s.bytes += bytes;
    return (char *)s.block + at;
  }
  void *p = nullptr;
  check(hipMalloc(&p, bytes), what);
  s.allocations.push_back(p);
  s.bytes += bytes;
  return p;
}

void free_system(DevSystem &s) {
  for (void *p : s.allocations) (void)hipFree(p);
  s.allocations.clear();
}

}  // namespace

namespace {

// Gives back the buffers a plain run's launches grow (not its window list).
void drop_run_scratch(atrip_hip_ctx *ctx) {
  if (ctx->stream) (void)hipStreamSynchronize(ctx->stream);
  auto drop = [](double *&p, size_t &bytes) {
    if (p) (void)hipFree(p);
    p = nullptr;
    bytes = 0;
  };
  drop(ctx->G, ctx->G_bytes);
  drop(ctx->e_slot, ctx->e_slot_bytes);
  drop(ctx->wcube, ctx->wcube_bytes);
  drop(ctx->partials, ctx->partials_bytes);
}

// The contexts of the process.  Whoever holds the mutex may wait for a
// context's in_use; nobody takes it with an in_use held.
std::mutex contexts_mutex;
// (never destroyed: a context may be freed while the process ends)
std::vector<atrip_hip_ctx *> &contexts = *new std::vector<atrip_hip_ctx *>;

}  // namespace

void atrip_amd::give_back(atrip_hip_ctx *ctx) {
  std::lock_guard<std::mutex> use(ctx->in_use);
  drop_run_scratch(ctx);  // (waits for the stream)
  for (auto &kv : ctx->systems) {
    DevSystem &s = kv.second;
    if (!s.swaps) continue;
    for (const SwapCopy &c : swap_copies(s)) *c.copy = nullptr;
    s.allocations.erase(
        std::find(s.allocations.begin(), s.allocations.end(), s.swaps));
    (void)hipFree(s.swaps);
    s.swaps = nullptr;
    s.bytes -= s.swap_bytes;
  }
}

void atrip_amd::give_back_others(atrip_hip_ctx *ctx) {
  std::lock_guard<std::mutex> all(contexts_mutex);
  for (atrip_hip_ctx *c : contexts)
    if (c != ctx && c->device == ctx->device) give_back(c);
}

// Device bytes alloc_system takes for a system (the arrays below, the
// packed point table and the canonical-index prefix).
uint64_t atrip_amd::system_bytes(int64_t No, int64_t Nv, bool with_j,
                                 int store, bool swaps) {
  const uint64_t Kv = pad16(Nv), Ko = pad16(No), N2 = No * No, Nv2 = Nv * Nv;
  const auto d = [](uint64_t n) { return std::max<uint64_t>(n, 1) * 8; };
  // doubles operands: 8 bytes per element as FP64, 6 as split (4 + 2), 4
  // as FP32 only; bf16x3 copies by their tiled geometry
  const auto o = [&](uint64_t n) {
    return store == 2 ? n * 4 : store == 1 ? n * 6 : d(n);
  };
  uint64_t b = d(Nv2 * N2) + d(Nv * No) + d(No) + d(Nv);
  if (store == 3) {
    b += tri_bytes(tri_geom_a(No, Nv, Kv)) + tri_bytes(tri_geom_b(No, Nv, Kv)) +
         tri_bytes(tri_geom_a(No, Nv, Ko)) + 2 * tri_bytes(tri_geom_b(No, Nv, Ko));
    if (with_j)
      b += tri_bytes(tri_geom_b(No, Nv, Kv)) + tri_bytes(tri_geom_a(No, Nv, Ko));
  } else if (store == 0) {
    const auto f = [&](const TriGeom &g) { return d((uint64_t)f64_elems(g)); };
    const uint64_t t3 = f(f64_geom_a(No, Nv, Kv)), h3 = f(f64_geom_a(No, Nv, Ko)),
                   v3 = f(f64_geom_b(No, Nv, Kv));
    b += t3 + v3 + h3 + 2 * f(f64_geom_b(No, Nv, Ko)) + (swaps ? t3 + h3 : 0);
    if (with_j) b += v3 + h3 + (swaps ? h3 : 0);
  } else {
    b += o(Nv * N2 * Kv) + o(Nv2 * No * Kv) + o(Nv * N2 * Ko) +
         2 * o(Nv2 * No * Ko);
    if (with_j) b += o(Nv2 * No * Kv) + o(Nv * N2 * Ko);
  }
  b += (uint64_t)No * (No + 1) * (No + 2) / 6 * sizeof(uint32_t);
  b += (Nv + 1) * sizeof(uint64_t);
  return b;
}

namespace {

// The arrays of a system but its row-swapped copies.
void lay_out(DevSystem &s, bool with_j, bool cplx) {
  const int64_t No = s.No, Nv = s.Nv, N2 = No * No, Nv2 = Nv * Nv;
  // doubles operands: FP64, or only their split / FP32 / bf16x3 form
  auto operand = [&](double *&x, DevSystem::Split &sp, TriOp &tp,
                     const TriGeom &g, const char *what) {
    const int64_t n = g.no * g.nr * g.K;
    if (s.store == 0) {
      x = dev_alloc(s, f64_elems(g), what);
      return;
    }
    if (s.store == 3) {
      alloc_tri(s, tp, g.swapped ? tri_geom_a(No, Nv, g.K) : tri_geom_b(No, Nv, g.K),
                what);
      return;
    }
    sp.h = (float *)dev_bytes(s, (size_t)n * sizeof(float), what);
    if (s.store == 1) {
      sp.l = (uint16_t *)dev_bytes(s, (size_t)n * 2, what);
    }
  };
  const TriGeom ga = f64_geom_a(No, Nv, s.Kv), gb = f64_geom_b(No, Nv, s.Kv),
                gh = f64_geom_a(No, Nv, s.Ko), gt = f64_geom_b(No, Nv, s.Ko);
  operand(s.T3, s.sT3, s.tT3, ga, "alloc T3");
  operand(s.V3, s.sV3, s.tV3, gb, "alloc V3");
  operand(s.H3, s.sH3, s.tH3, gh, "alloc H3");
  operand(s.T2N, s.sT2N, s.tT2N, gt, "alloc T2N");
  operand(s.T2TN, s.sT2TN, s.tT2TN, gt, "alloc T2TN");
  s.split_ready = s.store == 1 || s.store == 2;
  s.tri_ready = s.store == 3;
  s.VHH = dev_alloc(s, Nv2 * N2, "alloc VHH");
  s.Tai = dev_alloc(s, Nv * No, "alloc Tai");
  s.ei = dev_alloc(s, No, "alloc ei");
  s.ea = dev_alloc(s, Nv, "alloc ea");
  s.has_j = with_j;
  if (with_j) {
    operand(s.V3J, s.sV3J, s.tV3J, gb, "alloc V3J");
    operand(s.H3J, s.sH3J, s.tH3J, gh, "alloc H3J");
  }
  s.cplx = cplx;
  if (cplx) {
    s.T3i = dev_alloc(s, f64_elems(ga), "alloc T3 (im)");
    s.V3i = dev_alloc(s, f64_elems(gb), "alloc V3 (im)");
    s.H3i = dev_alloc(s, f64_elems(gh), "alloc H3 (im)");
    s.T2Ni = dev_alloc(s, f64_elems(gt), "alloc T2N (im)");
    s.T2TNi = dev_alloc(s, f64_elems(gt), "alloc T2TN (im)");
    s.VHHi = dev_alloc(s, Nv2 * N2, "alloc VHH (im)");
    s.Taii = dev_alloc(s, Nv * No, "alloc Tai (im)");
    s.eii = dev_alloc(s, No, "alloc ei (im)");
    s.eai = dev_alloc(s, Nv, "alloc ea (im)");
    s.T3in = dev_alloc(s, f64_elems(ga), "alloc -T3 (im)");
    s.H3in = dev_alloc(s, f64_elems(gh), "alloc -H3 (im)");
    if (with_j) {
      s.V3Ji = dev_alloc(s, f64_elems(gb), "alloc V3J (im)");
      s.H3Ji = dev_alloc(s, f64_elems(gh), "alloc H3J (im)");
      s.H3Jin = dev_alloc(s, f64_elems(gh), "alloc -H3J (im)");
    }
  }
  s.npoints = No * (No + 1) * (No + 2) / 6;
  s.points = (uint32_t *)dev_bytes(s, (size_t)s.npoints * sizeof(uint32_t),
                                   "alloc points");
  s.aprefix = (uint64_t *)dev_bytes(s, (size_t)(Nv + 1) * sizeof(uint64_t),
                                    "alloc prefix");
}

// One block holds all of a system's arrays: an allocation for each, with its
// release, took a fifth of a small system's upload (No=10, Nv=50: upload and
// release 930 -> 730 us with the two tables made on the device and no wait
// between the tensors).
void alloc_system(atrip_hip_ctx *ctx, DevSystem &s, int64_t No, int64_t Nv,
                  bool with_j, bool cplx = false) {
  if (No < 1 || Nv < 1) throw Fail{"No and Nv must be positive"};
  if (cplx && ctx->operand_store != 0)
    throw Fail{"complex systems keep FP64 operands (operand_store 0)"};
  if (No > 1023) throw Fail{"No > 1023 is not supported"};
  s.No = No;
  s.Nv = Nv;
  s.Kv = pad16(Nv);
  s.Ko = pad16(No);
  s.store = ctx->operand_store;
  s.laying = DevSystem::COUNT;
  lay_out(s, with_j, cplx);
  check(hipMalloc(&s.block, s.block_bytes), "alloc system");
  s.allocations.push_back(s.block);
  s.block_bytes = 0;
  s.laying = DevSystem::PLACE;
  lay_out(s, with_j, cplx);
  s.laying = DevSystem::NONE;
  if (s.store == 0 && ctx->operand_swaps) alloc_swaps(s);
}

// The points and prefix tables (see launch_tables), after any clearing.
void fill_tables(const DevSystem &s, hipStream_t st) {
  check(launch_tables(s, st), "point and prefix tables");
}

// Where the values of a system's input tensors come from.  Values are in
// CTF linear (column-major) order; a value is `comp` doubles (1 real, 2 an
// interleaved (re, im) pair).  fetch() copies values [first, first + count)
// of tensor t (enum atrip_tensor) to device memory on stream st; host()
// reads them into host memory (the small tensors).
struct Source {
  int comp = 1;
  virtual ~Source() = default;
  virtual void fetch(int t, int64_t first, int64_t count, double *dst,
                     hipStream_t st) = 0;
  virtual void host(int t, int64_t first, int64_t count, double *out) = 0;
};

// Tensors in caller memory (the pointers of an atrip_sys_desc).
struct DescSource : Source {
  const double *p[9];
  DescSource(const atrip_sys_desc *d, int comp_) {
    comp = comp_;
    const double *q[9] = {d->ei,    d->ea,    d->Tai,   d->Tabij, d->Vabij,
                          d->Vijka, d->Vabci, d->Jijka, d->Jabci};
    std::copy(q, q + 9, p);
  }
  void fetch(int t, int64_t first, int64_t count, double *dst,
             hipStream_t st) override {
    check(hipMemcpyAsync(dst, p[t] + first * comp,
                         (size_t)(count * comp) * sizeof(double),
                         hipMemcpyHostToDevice, st),
          "upload chunk");
  }
  void host(int t, int64_t first, int64_t count, double *out) override {
    std::memcpy(out, p[t] + first * comp, (size_t)(count * comp) * sizeof(double));
  }
};

// Tensors read through the caller's reader, piece by piece into a pinned
// host buffer of bounded size (two halves: one is read into while the copy
// of the other is in flight), so the host holds no tensor whole.
struct ReaderSource : Source {
  atrip_read_fn fn;
  void *user;
  double *pinned = nullptr;
  int64_t half = 0;  // doubles per half
  hipEvent_t done[2] = {nullptr, nullptr};
  bool recorded[2] = {false, false};
  ReaderSource(atrip_read_fn f, void *u, int comp_, int64_t cap_bytes)
      : fn(f), user(u) {
    comp = comp_;
    half = std::max<int64_t>(comp, cap_bytes / (2 * (int64_t)sizeof(double)));
    half = half / comp * comp;
    try {
      check(hipHostMalloc((void **)&pinned,
                          (size_t)(2 * half) * sizeof(double),
                          hipHostMallocDefault),
            "alloc pinned staging");
      for (auto &e : done)
        check(hipEventCreateWithFlags(&e, hipEventDisableTiming), "event");
    } catch (...) {
      release();  // no destructor runs for a constructor that throws
      throw;
    }
  }
  ~ReaderSource() override { release(); }
  void release() {
    for (int h = 0; h < 2; h++)
      if (recorded[h]) (void)hipEventSynchronize(done[h]);  // copies done
    for (auto &e : done)
      if (e) (void)hipEventDestroy(e), e = nullptr;
    if (pinned) (void)hipHostFree(pinned), pinned = nullptr;
  }
  void read(int t, int64_t first, int64_t count, double *out) {
    if (fn(user, t, first, count, out) != 0)
      throw Fail{"tensor reader failed (tensor " + std::to_string(t) +
                 ", values " + std::to_string(first) + "+" +
                 std::to_string(count) + ")"};
  }
  void fetch(int t, int64_t first, int64_t count, double *dst,
             hipStream_t st) override {
    const int64_t per = half / comp;  // values per piece
    int h = 0;
    for (int64_t off = 0; off < count; off += per, h ^= 1) {
      const int64_t n = std::min(per, count - off);
      double *buf = pinned + h * half;
      if (recorded[h]) check(hipEventSynchronize(done[h]), "pinned staging");
      read(t, first + off, n, buf);
      check(hipMemcpyAsync(dst + off * comp, buf,
                           (size_t)(n * comp) * sizeof(double),
                           hipMemcpyHostToDevice, st),
            "upload chunk");
      check(hipEventRecord(done[h], st), "event");
      recorded[h] = true;
    }
  }
  void host(int t, int64_t first, int64_t count, double *out) override {
    read(t, first, count, out);
  }
};

// Device staging of an upload: one buffer, grown to the largest step of its
// tensors (at most stage_kb, or one slab), given back at the end.
struct Stage {
  hipStream_t st;
  void *p = nullptr;
  size_t bytes = 0;
  explicit Stage(hipStream_t s) : st(s) {}
  Stage(const Stage &) = delete;
  ~Stage() { drop(); }
  void drop() {
    if (!p) return;
    (void)hipStreamSynchronize(st);  // the kernels that read it
    (void)hipFree(p);
    p = nullptr;
    bytes = 0;
  }
  double *get(size_t need) {
    if (need > bytes) {
      drop();
      check(hipMalloc(&p, need), "alloc staging");
      bytes = need;
    }
    return (double *)p;
  }
};

// Stage tensor t through a bounded device buffer (the context's stage_kb),
// whole slabs of `slab` values of its slowest CTF index per step (n_slow
// slabs; at least one slab per step), and hand each staged chunk to
// `place(dev_chunk, first_slow, count_slow)`.  A step's copy follows the kernels
// that read the buffer before it on the stream.
int64_t stage_slabs(const atrip_hip_ctx *ctx, int comp, int64_t slab,
                    int64_t n_slow) {
  const int64_t budget = std::max<int64_t>(
      1, ctx->stage_kb * 1024 / (int64_t)(sizeof(double) * comp));
  return std::min(std::max<int64_t>(1, budget / std::max<int64_t>(slab, 1)),
                  n_slow);
}
template <typename P>
void staged(atrip_hip_ctx *ctx, Stage &stage, Source &src, int t, int64_t slab,
            int64_t n_slow, P &&place) {
  const int64_t per = stage_slabs(ctx, src.comp, slab, n_slow);
  double *buf = stage.get((size_t)(per * slab * src.comp) * sizeof(double));
  for (int64_t s0 = 0; s0 < n_slow; s0 += per) {
    const int64_t cnt = std::min(per, n_slow - s0);
    src.fetch(t, s0 * slab, cnt * slab, buf, ctx->stream);
    place((const double *)buf, s0, cnt);
  }
}

// A system that keeps only the split / FP32 / bf16x3 form of its doubles
// operands gets each FP64 operand in a temporary device array, converted
// and freed as soon as it is filled.
struct TempOperands {
  DevSystem &s;
  hipStream_t st;
  struct Item {
    double **x;
    DevSystem::Split *sp;
    TriOp *tp;
    TriGeom g;  // of the FP64 array
  };
  std::vector<Item> items;
  void add(double *&x, DevSystem::Split &sp, TriOp &tp, const TriGeom &g) {
    if (s.store == 0) return;
    const size_t bytes = (size_t)f64_elems(g) * sizeof(double);
    void *p = nullptr;
    check(hipMalloc(&p, bytes), "alloc temporary operand");
    x = (double *)p;
    items.push_back({&x, &sp, &tp, g});
    check(hipMemsetAsync(p, 0, bytes, st), "clear temporary operand");
  }
  void convert() {
    for (Item &it : items) {
      if (s.store == 3)
        convert_tri(s, *it.x, it.g, *it.tp,
                    it.g.swapped ? tri_geom_a(s.No, s.Nv, it.g.K)
                                 : tri_geom_b(s.No, s.Nv, it.g.K),
                    st);
      else
        convert_split(s, *it.x, it.g, *it.sp, st);
      check(hipStreamSynchronize(st), "operand conversion");
      (void)hipFree(*it.x);
      *it.x = nullptr;
    }
    items.clear();
  }
  ~TempOperands() {
    for (Item &it : items) {
      (void)hipFree(*it.x);
      *it.x = nullptr;
    }
  }
};

// Re-lays out every input tensor of `src` into the device arrays of s (and
// of im, the imaginary planes, for a complex source: src.comp == 2).  Each
// large tensor is streamed in slabs of its slowest CTF index through the
// staging buffer; every transpose reads one part of the interleaved values
// (stride comp).
void upload_tensors(atrip_hip_ctx *ctx, DevSystem &s, DevSystem *im,
                    Source &src) {
  const int64_t No = s.No, Nv = s.Nv, N2 = No * No, Nv2 = Nv * Nv;
  const int64_t Kv = s.Kv, Ko = s.Ko;
  const int m = src.comp;
  if ((m == 2) != (im != nullptr)) throw Fail{"internal: complex parts"};
  DevSystem *dst[2] = {&s, im};
  hipStream_t st = ctx->stream;
  clear_operands(s, st);
  fill_tables(s, st);
  TempOperands tmp{s, st, {}};
  Stage stage(st);
  if (s.store == 0) {  // (beside no temporary operands)
    auto need = [&](int64_t slab, int64_t n_slow) {
      return stage_slabs(ctx, m, slab, n_slow) * slab * m * sizeof(double);
    };
    stage.get(std::max({need(Nv2 * No, No), need(N2 * No, Nv), need(Nv2 * Nv, No)}));
  }
  tmp.add(s.T3, s.sT3, s.tT3, f64_geom_a(No, Nv, Kv));
  tmp.add(s.T2N, s.sT2N, s.tT2N, f64_geom_b(No, Nv, Ko));
  tmp.add(s.T2TN, s.sT2TN, s.tT2TN, f64_geom_b(No, Nv, Ko));
  const int64_t N2p = pad16(N2);
  // straight array, then its row-swapped copy when there is one
  auto both = [&](double *x, double *xs, const double *c, int64_t no,
                  int64_t na, int64_t nb, int64_t so, int64_t sa, int64_t sb,
                  TileMap straight, TileMap swapped, const char *what) {
    check(launch_transpose_tiled(c, x, no, na, nb, so, sa, sb, straight, 1.0, st),
          what);
    if (xs)
      check(launch_transpose_tiled(c, xs, no, na, nb, so, sa, sb, swapped, 1.0, st),
            what);
  };
  // Tabij {Nv,Nv,No,No}: slowest index j
  staged(ctx, stage, src, ATRIP_TENSOR_TABIJ, Nv2 * No, No,
         [&](const double *c, int64_t j0, int64_t cj) {
           for (int part = 0; part < m; part++) {
             DevSystem &d = *dst[part];
             // T3[x][p + No q][E] = T[x,E,p,q], rows of this chunk: q = j
             TileMap t, w;
             t.R0 = j0 * No; t.Ro = 1; t.Rb = N2p; t.ka = 1; t.K = Kv;
             w = t;
             w.R0 = w.Ro = 0; w.swap = 1; w.row0 = j0 * No; w.No = No;
             both(d.T3, d.T3s, c + part, No * cj, Nv, Nv, m * Nv2, m * Nv, m,
                  t, w, "relayout T3");
             // T2N[pair][n][L] = -T[pair,L,n], n = j
             TileMap n;
             n.R0 = j0; n.Ro = 1; n.Rb = No; n.ka = 1; n.K = Ko;
             check(launch_transpose_tiled(c + part, d.T2N, cj, No, Nv2,
                                          m * Nv2 * No, m * Nv2, m, n, -1.0, st),
                   "relayout T2N");
             // T2TN[pair][n][L] = -T[pair,n,L], L = j
             TileMap l;
             l.Ra = 1; l.Rb = No; l.k0 = j0; l.ko = 1; l.K = Ko;
             check(launch_transpose_tiled(c + part, d.T2TN, cj, No, Nv2,
                                          m * Nv2 * No, m * Nv2, m, l, -1.0, st),
                   "relayout T2TN");
           }
         });
  // Vabij {Nv,Nv,No,No}: VHH[pair][i + No j]
  staged(ctx, stage, src, ATRIP_TENSOR_VABIJ, Nv2 * No, No,
         [&](const double *c, int64_t j0, int64_t cj) {
           for (int part = 0; part < m; part++)
             check(launch_transpose(c + part, dst[part]->VHH + j0 * No, 1,
                                    No * cj, Nv2, 0, m * Nv2, m, 0, 1, N2, 1.0,
                                    st),
                   "relayout VHH");
         });
  // Vijka {No,No,No,Nv}: H3[x][row][L] = V[row,L,x]
  auto hhh = [&](int t, double *DevSystem::*arr, double *DevSystem::*arrs) {
    staged(ctx, stage, src, t, N2 * No, Nv,
           [&](const double *c, int64_t x0, int64_t cx) {
             for (int part = 0; part < m; part++) {
               TileMap t, w;
               t.R0 = x0 * N2p; t.Ro = N2p; t.Rb = 1; t.ka = 1; t.K = Ko;
               w = t;
               w.Rb = 0; w.swap = 2; w.No = No;
               both(dst[part]->*arr, dst[part]->*arrs, c + part, cx, No, N2,
                    m * N2 * No, m * N2, m, t, w, "relayout H3");
             }
           });
  };
  // Vabci {Nv,Nv,Nv,No}: V3[pair][r][E] = V[pair,E,r]
  auto ppph = [&](int t, double *DevSystem::*arr) {
    staged(ctx, stage, src, t, Nv2 * Nv, No,
           [&](const double *c, int64_t r0, int64_t cr) {
             for (int part = 0; part < m; part++) {
               TileMap t;
               t.R0 = r0; t.Ro = 1; t.Rb = No; t.ka = 1; t.K = Kv;
               check(launch_transpose_tiled(c + part, dst[part]->*arr, cr, Nv,
                                            Nv2, m * Nv2 * Nv, m * Nv2, m, t,
                                            1.0, st),
                     "relayout V3");
             }
           });
  };
  tmp.convert();
  tmp.add(s.H3, s.sH3, s.tH3, f64_geom_a(No, Nv, Ko));
  hhh(ATRIP_TENSOR_VIJKA, &DevSystem::H3, &DevSystem::H3s);
  tmp.convert();
  tmp.add(s.V3, s.sV3, s.tV3, f64_geom_b(No, Nv, Kv));
  ppph(ATRIP_TENSOR_VABCI, &DevSystem::V3);
  tmp.convert();
  if (s.has_j) {
    tmp.add(s.H3J, s.sH3J, s.tH3J, f64_geom_a(No, Nv, Ko));
    hhh(ATRIP_TENSOR_JIJKA, &DevSystem::H3J, &DevSystem::H3Js);
    tmp.convert();
    tmp.add(s.V3J, s.sV3J, s.tV3J, f64_geom_b(No, Nv, Kv));
    ppph(ATRIP_TENSOR_JABCI, &DevSystem::V3J);
    tmp.convert();
  }
  // the small tensors whole (the reference's read_all, Atrip.cxx:176-181)
  std::vector<std::vector<double>> kept;  // until the copies are done
  auto small = [&](int t, int64_t n, double *DevSystem::*arr, const char *what) {
    std::vector<double> buf((size_t)(n * m));
    src.host(t, 0, n, buf.data());
    for (int q = 0; q < m; q++) {
      std::vector<double> part((size_t)n);
      for (int64_t e = 0; e < n; e++) part[e] = buf[e * m + q];
      kept.push_back(std::move(part));
      check(hipMemcpyAsync(dst[q]->*arr, kept.back().data(),
                           (size_t)n * sizeof(double), hipMemcpyHostToDevice, st),
            what);
    }
  };
  struct Done {  // no copy reads host memory or the stage after this returns
    hipStream_t st;
    ~Done() { (void)hipStreamSynchronize(st); }
  } done{st};
  small(ATRIP_TENSOR_TAI, Nv * No, &DevSystem::Tai, "upload Tai");
  small(ATRIP_TENSOR_EI, No, &DevSystem::ei, "upload ei");
  small(ATRIP_TENSOR_EA, Nv, &DevSystem::ea, "upload ea");
  check(hipStreamSynchronize(st), "upload");
}

// The imaginary planes of a complex system in the slots of the real ones
// (for filling them with the real-system code).
DevSystem imag_view(const DevSystem &s) {
  DevSystem v;
  v.No = s.No; v.Nv = s.Nv; v.Kv = s.Kv; v.Ko = s.Ko;
  v.has_j = s.has_j;
  v.T3 = s.T3i; v.V3 = s.V3i; v.H3 = s.H3i; v.T2N = s.T2Ni;
  v.T2TN = s.T2TNi; v.VHH = s.VHHi; v.Tai = s.Taii; v.ei = s.eii;
  v.ea = s.eai; v.V3J = s.V3Ji; v.H3J = s.H3Ji;
  v.T3s = s.T3is; v.H3s = s.H3is; v.H3Js = s.H3Jis;
  v.aprefix = s.aprefix;
  return v;
}

// Negated imaginary planes of T3 and the hole integrals.
void complex_negations(atrip_hip_ctx *ctx, DevSystem &s) {
  const int64_t nt = f64_elems(f64_geom_a(s.No, s.Nv, s.Kv)),
                nh = f64_elems(f64_geom_a(s.No, s.Nv, s.Ko));
  auto neg = [&](const double *x, double *y, int64_t n) {
    if (x && y)
      check(launch_scale(x, y, n, -1.0, ctx->stream), "negate imaginary plane");
  };
  // a swapped negated copy needs its swapped source
  auto pair = [&](const double *x, double *y, const double *xs, double *&ys,
                  int64_t n) {
    neg(x, y, n);
    if (!xs) ys = nullptr;
    neg(xs, ys, n);
  };
  pair(s.T3i, s.T3in, s.T3is, s.T3ins, nt);
  pair(s.H3i, s.H3in, s.H3is, s.H3ins, nh);
  pair(s.H3Ji, s.H3Jin, s.H3Jis, s.H3Jins, nh);
  check(hipStreamSynchronize(ctx->stream), "negations");
}

// The four real products of a complex system, two per plane of W and class
// GEMM (one after the other along K: a plane is written once): W = Wr + i Wi
// with
//   Wr = [T3r V3r + H3r N_r] + [(-T3i) V3i + H3i N_i]
//   Wi = [T3r V3i + H3r N_i] + [T3i V3r + (-H3i) N_r]
// where N = -T2 (the pre-negated hole operands) and the hole terms carry
// conj(Vhhh) = H3r - i H3i, as the reference's complex GEMM path does
// (MAYBE_CONJ, src/atrip/Equations.cxx:620-656).
void complex_passes(const DevSystem &s, DevSystem v[4]) {
  for (int q = 0; q < 4; q++) {
    v[q].No = s.No; v[q].Nv = s.Nv; v[q].Kv = s.Kv; v[q].Ko = s.Ko;
    v[q].aprefix = s.aprefix;
    v[q].has_j = s.has_j;
  }
  v[0].T3 = s.T3;   v[0].V3 = s.V3;  v[0].H3 = s.H3;   v[0].T2N = s.T2N;
  v[0].T2TN = s.T2TN;  v[0].V3J = s.V3J;  v[0].H3J = s.H3J;
  v[1].T3 = s.T3in; v[1].V3 = s.V3i; v[1].H3 = s.H3i;  v[1].T2N = s.T2Ni;
  v[1].T2TN = s.T2TNi; v[1].V3J = s.V3Ji; v[1].H3J = s.H3Ji;
  v[2].T3 = s.T3;   v[2].V3 = s.V3i; v[2].H3 = s.H3;   v[2].T2N = s.T2Ni;
  v[2].T2TN = s.T2TNi; v[2].V3J = s.V3Ji; v[2].H3J = s.H3J;
  v[3].T3 = s.T3i;  v[3].V3 = s.V3;  v[3].H3 = s.H3in; v[3].T2N = s.T2N;
  v[3].T2TN = s.T2TN;  v[3].V3J = s.V3J;  v[3].H3J = s.H3Jin;
  v[0].T3s = s.T3s;   v[0].H3s = s.H3s;   v[0].H3Js = s.H3Js;
  v[1].T3s = s.T3ins; v[1].H3s = s.H3is;  v[1].H3Js = s.H3Jis;
  v[2].T3s = s.T3s;   v[2].H3s = s.H3s;   v[2].H3Js = s.H3Js;
  v[3].T3s = s.T3is;  v[3].H3s = s.H3ins; v[3].H3Js = s.H3Jins;
}

// Host-side canonical index, identical to the device one.
struct HostIndex {
  std::vector<uint64_t> pre;
  uint64_t Nv;
  explicit HostIndex(uint64_t nv) : pre(nv + 1, 0), Nv(nv) {
    for (uint64_t a = 0; a < nv; a++) {
      const uint64_t m = nv - a;
      pre[a + 1] = pre[a] + m * (m + 1) / 2 - 1;
    }
  }
  uint64_t operator()(uint64_t a, uint64_t b, uint64_t c) const {
    return tuple_index(pre.data(), Nv, a, b, c);
  }
  // First index of tuple q.
  int64_t first_of(uint64_t q) const {
    return std::upper_bound(pre.begin(), pre.end(), q) - pre.begin() - 1;
  }
};

// Windows of a run: origins (a0, b0, c0), tuples each holds, edges.
struct Windows {
  std::vector<int32_t> origin;
  std::vector<uint64_t> count;
  int ea = 0, eb = 0, ec = 0;
  // Adds the window at an origin if it holds a tuple of [first, last): the
  // tuples of a row (a, b) are consecutive in c.
  void add(const HostIndex &h, uint64_t first, uint64_t last, uint64_t a0,
           uint64_t b0, uint64_t c0) {
    uint64_t n = 0;
    for (uint64_t a = a0; a < std::min<uint64_t>(a0 + ea, h.Nv); a++)
      for (uint64_t b = std::max(a, b0); b < std::min<uint64_t>(b0 + eb, h.Nv); b++) {
        const uint64_t c = std::max(c0, b + (a == b)),
                       e = std::min<uint64_t>(c0 + ec, h.Nv);
        if (c >= e) continue;
        const uint64_t q = std::max(first, h(a, b, c)),
                       z = std::min(last, h(a, b, e - 1) + 1);
        if (z > q) n += z - q;
      }
    if (!n) return;
    origin.insert(origin.end(), {(int32_t)a0, (int32_t)b0, (int32_t)c0});
    count.push_back(n);
  }
};

// Window plan for a system at the context's window edge: the block triples
// in lexicographic order holding a tuple, with their tuple counts.
WindowPlan &get_plan(atrip_hip_ctx *ctx, int sys, const DevSystem &s,
                     int nb_want = 0) {
  if (nb_want <= 0) nb_want = window_edge(ctx, s);
  auto it = ctx->plans.find(sys);
  if (it != ctx->plans.end() && it->second.nb == nb_want) return it->second;
  if (it != ctx->plans.end()) ctx->plans.erase(it);
  WindowPlan p;
  p.nb = nb_want;
  const HostIndex h((uint64_t)s.Nv);
  Windows w;
  w.ea = w.eb = w.ec = p.nb;
  for (int64_t a = 0; a < s.Nv; a += p.nb)
    for (int64_t b = a; b < s.Nv; b += p.nb)
      for (int64_t c = b; c < s.Nv; c += p.nb) w.add(h, 0, ~0ULL, a, b, c);
  p.origin = std::move(w.origin);
  p.wcount = std::move(w.count);
  return ctx->plans.emplace(sys, std::move(p)).first->second;
}

void ensure(void *&ptr, size_t &have, size_t need, const char *what) {
  if (have >= need && ptr) return;
  if (ptr) check(hipFree(ptr), what);
  ptr = nullptr;
  have = 0;
  check(hipMalloc(&ptr, need), what);
  have = need;
}

// Makes a filled system resident; its handle.
int add_system(atrip_hip_ctx *ctx, DevSystem &&s) {
  std::lock_guard<std::mutex> use(ctx->in_use);
  const int id = ctx->next_sys++;
  ctx->systems.emplace(id, std::move(s));
  return id;
}

struct RunResult {
  double e = 0, ect = 0;
  uint64_t tuples = 0;  // tuples computed
};

// Destroys the queued timing events (read at the end of a run, or left by
// a run that failed); each event can end one pair and start the next, so
// they are deduplicated first.
void drop_pending_events(atrip_hip_ctx *ctx) {
  std::vector<hipEvent_t> uniq;
  for (auto &pr : ctx->pending_events) {
    uniq.push_back(pr.first);
    uniq.push_back(pr.second);
  }
  std::sort(uniq.begin(), uniq.end());
  uniq.erase(std::unique(uniq.begin(), uniq.end()), uniq.end());
  for (auto ev : uniq) (void)hipEventDestroy(ev);
  ctx->pending_events.clear();
  ctx->pending_names.clear();
  ctx->pending_flop.clear();
}

// Runs every batch of windows intersecting [first, last).  When `sink` is
// given it receives the per-slot energies of each batch.
// A fixed device region a run may carve its scratch from (no allocation), and
// the bytes behind it that only the padding of class buffers may take.
struct FixedScratch {
  void *base;
  size_t bytes, pad;
};

// Which windows of the plan a run covers besides the tuple range: every
// stride-th row of windows (block pairs) from row offset, and plan windows
// [wbegin, wend) by their index in the plan.
struct WindowSel {
  uint64_t stride = 1, offset = 0;
  uint64_t wbegin = 0, wend = ~0ULL;
  int nb = 0;  // window edge of the plan; 0: the context's (window_edge)
};

template <typename Sink>
RunResult run_range(atrip_hip_ctx *ctx, int sys, int precision, int ijkabc,
                    uint64_t first, uint64_t last, Sink &&sink,
                    const WindowSel &wsel = WindowSel{},
                    const FixedScratch *fixed = nullptr) {
  std::lock_guard<std::mutex> use(ctx->in_use);
  drop_pending_events(ctx);
  DevSystem &s = get_sys(ctx, sys);
  WindowPlan &plan = get_plan(ctx, sys, s, wsel.nb);
  const uint64_t n = n_tuples(s.Nv);
  last = std::min(last, n);
  RunResult res;
  check_precision(s, precision);
  const bool g32 = precision != ATRIP_FP64;
  if (fixed) {
    // the operand copies of a mixed form are device allocations: a run
    // without allocation needs them resident already
    if (precision == ATRIP_BF16X3 && !s.tri_ready)
      throw Fail{"bf16x3 operand copies are not resident: run the system "
                 "once in bf16x3 through atrip_hip_run, or upload it with "
                 "operand_store 3"};
    if ((precision == ATRIP_SPLIT_FP32 || precision == ATRIP_FP32) &&
        !s.split_ready)
      throw Fail{"split FP32 operand copies are not resident: run the system "
                 "once in a split form through atrip_hip_run, or upload it "
                 "with operand_store 1 or 2"};
  } else if (precision == ATRIP_BF16X3) {
    ensure_tri(ctx, s);
  } else if (g32) {
    ensure_split(ctx, s);
  }
  if (first >= last) return res;
  const int nb = plan.nb;
  const bool full = first == 0 && last == n;
  // select windows and count their tuples in range
  Windows win;
  win.ea = win.eb = win.ec = nb;
  // Windows of the run's own, with edges (ea, eb, ec) of `win`, from the
  // range's first index on.
  const HostIndex hidx((uint64_t)s.Nv);
  const int64_t a0 = hidx.first_of(first), a1 = hidx.first_of(last - 1);
  auto own_windows = [&](int ea) {
    win.origin.clear();
    win.count.clear();
    win.ea = ea;
    for (int64_t a = a0; a <= a1; a += win.ea)
      for (int64_t b = a0 + (a - a0) / win.eb * win.eb; b < s.Nv; b += win.eb)
        for (int64_t c = b; c < s.Nv; c += win.ec) win.add(hidx, first, last, a, b, c);
  };
  if (full) {
    const size_t nwin = plan.wcount.size();
    int64_t pair = -1, prev_a = -1, prev_b = -1;  // (alpha, beta) row index
    for (size_t w = 0; w < nwin; w++) {
      const int32_t *o = &plan.origin[3 * w];
      if (o[0] != prev_a || o[1] != prev_b) {
        pair++;
        prev_a = o[0];
        prev_b = o[1];
      }
      if (w < wsel.wbegin || w >= wsel.wend) continue;
      if (wsel.stride > 1 && (uint64_t)pair % wsel.stride != wsel.offset % wsel.stride)
        continue;
      win.origin.insert(win.origin.end(), o, o + 3);
      win.count.push_back(plan.wcount[w]);
    }
  } else {
    // A range holds few first indices (1 % of No=40, Nv=400 about two), so it
    // takes windows of its own: the first index of the range's tuples cut
    // evenly into blocks of at most the edge.  Blocks aligned as the plan's
    // left the window columns of the other first indices empty.
    const int64_t na = a1 - a0 + 1, blocks = (na + nb - 1) / nb;
    own_windows((int)((na + blocks - 1) / blocks));
  }
  const std::vector<int32_t> &sel = win.origin;
  for (uint64_t c : win.count) res.tuples += c;
  int nsel = (int)win.count.size();
  if (!nsel) return res;
  // Device scratch of the run: class buffers G (and those of the (cT)
  // pass; two planes each for complex systems), per-slot energies, the energy
  // kernels' scratch (per-triple partials, or W cubes for complex systems
  // and the cube epilogue), batch partials and the window list.  Taken from the context's buffers (grown
  // on demand), or carved out of a fixed region without any allocation
  // (then the windows per launch shrink until the run fits, and the window
  // list and partials of a few launches at a time are held).
  int64_t per = (int64_t)win.ea * win.eb * win.ec;  // slots of a window
  const int64_t W3 = g_elems(s.No);  // one tuple's class buffer
  const bool use_j = s.has_j;
  const int nsets = s.cplx ? 2 : 1;  // W's planes
  const size_t gelem = g32 ? sizeof(float) : sizeof(double);
  const bool fused = ctx->epilogue == 0;
  struct Sizes {
    int64_t slots_max = 0;
    size_t gsz = 0, g = 0, e_slot = 0, wcube = 0, partials = 0, windows = 0;
    int nbatch = 0, group = 0;  // launches; launches of one window list
  };
  auto sizes = [&](int bw_, int64_t W3_) {
    Sizes z;
    z.slots_max = (int64_t)std::min(bw_, nsel) * per;
    z.gsz = (size_t)(3 * z.slots_max * W3_) * gelem;
    z.g = (size_t)((use_j ? 2 : 1) * nsets) * z.gsz;
    z.e_slot = (size_t)(2 * z.slots_max) * sizeof(double);
    z.wcube = (size_t)(z.slots_max * energy_scratch_per_slot(
                                         s.No, use_j, g32, s.cplx, fused)) *
              sizeof(double);
    z.nbatch = z.group = (nsel + bw_ - 1) / bw_;
    const size_t quads = (size_t)(4 * slot_partials(z.slots_max)) * sizeof(double),
                 list = (size_t)(3 * bw_) * sizeof(int32_t);
    if (fixed)
      z.group = (int)std::min<size_t>(
          z.nbatch, std::max<size_t>(1, (256 * 1024) / (quads + list)));
    z.partials = z.group * quads;
    z.windows = std::min(z.group * list, sel.size() * sizeof(int32_t));
    return z;
  };
  auto a256 = [](size_t x) { return (x + 255) / 256 * 256; };
  auto total = [&](const Sizes &z) {
    return a256(z.g) + a256(z.e_slot) + a256(z.wcube) + a256(z.partials) +
           a256(z.windows);
  };

  // (a window of a range counts by its slots)
  const int64_t least = ctx->batch > 0 ? ctx->batch : LEAST_BATCH;
  int bw = (int)std::min<int64_t>(
      4096, std::max<int64_t>(1, least * (int64_t)nb * nb * nb / per));
  const int bw_least = bw;
  if (ctx->batch == 0)
    bw = std::max(bw, auto_batch((use_j ? 2 : 1) * nsets * 3 * W3 *
                                     (int64_t)gelem, per));
  void *Gbuf = nullptr, *e_slot = nullptr, *wcube = nullptr,
       *partials = nullptr, *d_sel = nullptr;
  Sizes z;
  // per-window sums of a window-sum sink, for every selected window
  constexpr bool kWinSums = std::decay_t<Sink>::window_sums();
  const size_t wsz = kWinSums ? (size_t)(2 * nsel) * sizeof(double) : 0;
  double *wsum_dev = nullptr;
  if (fixed && kWinSums)
    throw Fail{"per-window sums are not an allocation-free run"};
  if (fixed) {
    while (bw > 1 && total(sizes(bw, W3)) > fixed->bytes) bw--;
    z = sizes(bw, W3);
    // What the region holds is counted in class buffers of GEMM order, rows
    // padded to a line.  Blocks of 8^3 take more (2.8 times at No=17, 1.7 at
    // 20), so a window that fits but for them is cut along its first index.
    // Where the edge is 1 already, their padding has `pad`.
    if (const size_t need = total(z); need > fixed->bytes) {
      const Sizes zg = sizes(1, std::min(W3, g_row_elems(s.No, g32)));
      const size_t per_slot = (zg.g + zg.wcube + zg.e_slot) / (size_t)per;
      const size_t slab = (z.g + z.wcube + z.e_slot) / (size_t)win.ea;
      const size_t limit = fixed->bytes + fixed->pad;
      int ea = total(zg) > fixed->bytes
                   ? 0
                   : (int)std::min<size_t>(win.ea, limit / slab);
      for (; ea >= 1; ea--) {
        if (ea < win.ea) own_windows(ea);
        per = (int64_t)win.ea * win.eb * win.ec;
        nsel = (int)win.count.size();
        z = sizes(1, W3);
        if (total(z) <= limit) break;
      }
      if (ea < 1) {
        // largest window edge whose single window fits (class buffers, cubes
        // and slot energies scale with edge^3)
        const size_t rest = a256(zg.partials) + a256(zg.windows) + 3 * 256;
        int fit = 0;
        for (int e = nb - 1; e >= 1 && !fit; e--)
          if ((size_t)e * e * e * per_slot + rest <= fixed->bytes) fit = e;
        throw Fail{"run needs " + std::to_string(need) +
                   " bytes of scratch for one window of edge " +
                   std::to_string(nb) + " at No=" + std::to_string(s.No) +
                   "; the allocation-free entry point holds " +
                   std::to_string(fixed->bytes) +
                   (fit ? " (window edge " + std::to_string(fit) + " fits)"
                        : " (no window edge fits this No)")};
      }
    }
    char *p = (char *)fixed->base;
    Gbuf = p;
    p += a256(z.g);
    e_slot = p;
    p += a256(z.e_slot);
    wcube = p;
    p += a256(z.wcube);
    partials = p;
    p += a256(z.partials);
    d_sel = p;  // (filled by the launches)
  } else {
    z = sizes(bw, W3);
    // the window list lives in a context buffer grown on demand (no
    // allocation and release per call); the copy is ordered on the stream
    // before the kernels that read it, and `sel` outlives it (the run
    // waits for the stream before returning)
    ensure(ctx->sel, ctx->sel_bytes, a256(z.windows) + wsz, "alloc windows");
    d_sel = ctx->sel;
    if (kWinSums) wsum_dev = (double *)((char *)d_sel + a256(z.windows));
    check(hipMemcpyAsync(d_sel, sel.data(), z.windows, hipMemcpyHostToDevice,
                         ctx->stream),
          "upload windows");
    for (;;) {
      try {
        ensure((void *&)ctx->G, ctx->G_bytes, z.g, "alloc G");
        ensure((void *&)ctx->e_slot, ctx->e_slot_bytes, z.e_slot, "alloc e_slot");
        ensure((void *&)ctx->wcube, ctx->wcube_bytes, z.wcube,
               "alloc energy scratch");
        ensure((void *&)ctx->partials, ctx->partials_bytes, z.partials,
               "alloc partials");
        break;
      } catch (const Fail &) {
        // a device with little memory left: launches of the least size, in
        // buffers of their own (those the larger one had grown kept it out),
        // and when nothing is left to take back (retry_memory) of fewer windows:
        // blocks of 8^3 can take more than four windows in GEMM order did
        if (bw == 1 || (bw <= bw_least && ctx->operand_swaps)) throw;
        (void)hipGetLastError();
        drop_run_scratch(ctx);
        bw = bw > bw_least ? bw_least : bw / 2;
        z = sizes(bw, W3);
      }
    }
    Gbuf = ctx->G;
    e_slot = ctx->e_slot;
    wcube = ctx->wcube;
    partials = ctx->partials;
  }
  const size_t gsz = z.gsz;
  const int nbatch = z.nbatch;
  int64_t nparts = 0;  // partials written
  DevSystem zpass[4];
  if (s.cplx) complex_passes(s, zpass);
  // timing events are objects the runtime creates: none without allocation
  const bool timing = ctx->timing && !fixed;
  // complex products are four real ones (the reference bench counts 4x)
  const double flop_tuple = 12.0 * (double)s.No * s.No * s.No * (s.No + s.Nv) *
                            (s.cplx ? 4.0 : 1.0);
  const char *dname = precision == ATRIP_FP64        ? "doubles"
                      : precision == ATRIP_SPLIT_FP32 ? "doubles_mixed"
                      : precision == ATRIP_BF16X3     ? "doubles_bf16x3"
                                                      : "doubles_fp32";
  hipStream_t st = ctx->stream;
  double *Gz[2], *GJz[2];
  for (int q = 0; q < 2; q++) {
    Gz[q] = (double *)((char *)Gbuf + q * gsz);
    GJz[q] = (double *)((char *)Gbuf + (2 + q) * gsz);
  }
  void *G = Gbuf;
  void *GJ = use_j ? (void *)((char *)Gbuf + gsz) : nullptr;
  std::vector<double> host_slots;
  // Neumaier over the partials in slot order
  double s0 = 0, c0 = 0, s1 = 0, c1 = 0;
  std::vector<double> part;
  auto fetch_partials = [&] {
    part.resize(4 * nparts);
    check(hipMemcpyAsync(part.data(), (double *)partials,
                         part.size() * sizeof(double), hipMemcpyDeviceToHost, st),
          "download partials");
  };
  auto add_partials = [&] {
    auto add = [](double &sum, double &comp, double x) {
      const double t = sum + x;
      comp += (std::fabs(sum) >= std::fabs(x)) ? (sum - t) + x : (x - t) + sum;
      sum = t;
    };
    for (int64_t bi = 0; bi < nparts; bi++) {
      add(s0, c0, part[4 * bi]);
      add(s0, c0, part[4 * bi + 1]);
      add(s1, c1, part[4 * bi + 2]);
      add(s1, c1, part[4 * bi + 3]);
    }
    nparts = 0;
  };
  for (int bi = 0; bi < nbatch; bi++) {
    BatchArgs b;
    const int w0 = bi * bw, listed = fixed ? bi / z.group * z.group * bw : 0;
    if (fixed && w0 == listed) {
      if (bi) {
        fetch_partials();
        check(hipStreamSynchronize(st), "run");
        add_partials();
      }
      const int n = (int)std::min<int64_t>((int64_t)z.group * bw, nsel - w0);
      check(hipMemcpyAsync(d_sel, sel.data() + 3 * (size_t)w0,
                           (size_t)(3 * n) * sizeof(int32_t),
                           hipMemcpyHostToDevice, st),
            "upload windows");
    }
    b.nw = std::min(bw, nsel - w0);
    b.windows = (const int32_t *)d_sel + 3 * (w0 - listed);
    b.aprefix = s.aprefix;
    b.ea = win.ea;
    b.eb = win.eb;
    b.ec = win.ec;
    b.first = full ? 0 : first;
    b.last = full ? ~0ULL : last;
    b.slots = (int64_t)b.nw * per;
    uint64_t cnt = 0;
    for (int w = 0; w < b.nw; w++) cnt += win.count[w0 + w];
    // the batch's timing events; destroyed here unless handed to the
    // context's pending list (a launch that throws leaves none behind)
    struct BatchEvents {
      hipEvent_t e[3] = {nullptr, nullptr, nullptr};
      bool handed = false;
      ~BatchEvents() {
        if (!handed)
          for (hipEvent_t x : e)
            if (x) (void)hipEventDestroy(x);
      }
    } ev;
    if (timing) {
      for (hipEvent_t &x : ev.e) check(hipEventCreate(&x), "event");
      check(hipEventRecord(ev.e[0], st), "event");
    }
    for (int pass = 0; pass < (use_j ? 2 : 1) && s.cplx; pass++)
      for (int q = 0; q < 2; q++)
        check(launch_doubles_f64(zpass[2 * q], &zpass[2 * q + 1], b, pass == 1,
                                 pass == 0 ? Gz[q] : GJz[q], ctx->tile, st),
              "doubles kernel (complex plane)");
    for (int pass = 0; pass < (use_j ? 2 : 1) && !s.cplx; pass++) {
      void *Gp = pass == 0 ? G : GJ;
      if (precision == ATRIP_FP64)
        check(launch_doubles_f64(s, nullptr, b, pass == 1, (double *)Gp,
                                 ctx->tile, st),
              "doubles kernel");
      else if (precision == ATRIP_BF16X3)
        check(launch_doubles_tri(s, b, pass == 1, (float *)Gp, ctx->tile, st),
              "doubles (bf16x3) kernel");
      else
        check((precision == ATRIP_SPLIT_FP32 ? launch_doubles_split
                                             : launch_doubles_fp32)(
                  s, b, pass == 1, (float *)Gp, ctx->tile, st),
              "doubles (FP32 products) kernel");
    }
    if (timing) check(hipEventRecord(ev.e[1], st), "event");
    if (s.cplx)
      check(launch_energy_z(s, b, Gz, use_j ? GJz : nullptr,
                            ijkabc ? -1.0 : 1.0, (double *)e_slot,
                            (double *)wcube, fused, st),
            "energy kernel (complex)");
    else
      check(launch_energy(s, b, G, GJ, g32, ijkabc ? -1.0 : 1.0,
                          (double *)e_slot, (double *)wcube, fused, st),
            "energy kernel");
    if (timing) {
      check(hipEventRecord(ev.e[2], st), "event");
      ctx->pending_events.push_back({ev.e[0], ev.e[1]});
      ctx->pending_names.push_back(dname);
      ctx->pending_flop.push_back(flop_tuple * cnt * (use_j ? 2 : 1));
      ctx->pending_events.push_back({ev.e[1], ev.e[2]});
      ctx->pending_names.push_back("energy");
      ctx->pending_flop.push_back(0.0);
      ev.handed = true;
    }
    check(launch_slot_sums(fused && !s.cplx ? (const double *)wcube : nullptr,
                           b.slots, energy_parts(s.No, use_j, g32),
                           (double *)e_slot, (double *)partials + 4 * nparts,
                           st),
          "slot sums kernel");
    nparts += slot_partials(b.slots);
    if constexpr (kWinSums) {
      check(launch_window_sums((const double *)e_slot, b.nw, per,
                               wsum_dev + 2 * w0, st),
            "window sums kernel");
    } else if (sink.active()) {
      host_slots.resize(2 * b.slots);
      check(hipMemcpyAsync(host_slots.data(), (double *)e_slot,
                           host_slots.size() * sizeof(double),
                           hipMemcpyDeviceToHost, st),
            "download slots");
      check(hipStreamSynchronize(st), "slots");
      sink(sel.data() + 3 * w0, b, host_slots);
    }
  }
  fetch_partials();
  std::vector<double> wsums(kWinSums ? 2 * (size_t)nsel : 0);
  if (kWinSums)
    check(hipMemcpyAsync(wsums.data(), wsum_dev, wsz, hipMemcpyDeviceToHost,
                         st),
          "download window sums");
  check(hipStreamSynchronize(st), "run");
  if constexpr (kWinSums) sink.windows(wsums);
  add_partials();
  res.e = s0 + c0;
  res.ect = s1 + c1;
  // collect event timings
  for (size_t q = 0; q < ctx->pending_events.size(); q++) {
    float ms = 0.f;
    check(hipEventElapsedTime(&ms, ctx->pending_events[q].first,
                              ctx->pending_events[q].second),
          "elapsed");
    KernelStat &k = ctx->stats[ctx->pending_names[q]];
    k.launches++;
    k.ms += ms;
    k.flop += ctx->pending_flop[q];
  }
  drop_pending_events(ctx);  // read: release them
  return res;
}

struct NoSink {
  static constexpr bool window_sums() { return false; }
  bool active() const { return false; }
  void operator()(const int32_t *, const BatchArgs &, const std::vector<double> &) {}
};

}  // namespace

int atrip_amd::window_edge(const atrip_hip_ctx *ctx, const DevSystem &s) {
  return ctx->window > 0 ? ctx->window : auto_window(s.No, s.Nv);
}

uint64_t atrip_amd::plan_windows(atrip_hip_ctx *ctx, int sys, int nb) {
  DevSystem &s = get_sys(ctx, sys);
  return get_plan(ctx, sys, s, nb).wcount.size();
}

void atrip_amd::run_plan_windows(atrip_hip_ctx *ctx, int sys, int precision,
                                 int nb, uint64_t wbegin, uint64_t wend,
                                 std::vector<double> &out) {
  out.clear();
  // per-window (sum, comp) pairs formed on the device, downloaded once
  struct WinSink {
    static constexpr bool window_sums() { return true; }
    std::vector<double> *out;
    bool active() const { return true; }
    void windows(const std::vector<double> &pairs) {
      out->insert(out->end(), pairs.begin(), pairs.end());
    }
  } sink{&out};
  WindowSel ws;
  ws.wbegin = wbegin;
  ws.wend = wend;
  ws.nb = nb;
  run_range(ctx, sys, precision, 0, 0, ~0ULL, sink, ws);
}

void atrip_amd::run_fixed(atrip_hip_ctx *ctx, int sys, int precision,
                          int ijkabc, uint64_t first, uint64_t count,
                          void *base, size_t bytes, size_t pad,
                          double *energy, double *ct_energy) {
  const uint64_t last =
      count == ~0ULL || first + count < first ? ~0ULL : first + count;
  const FixedScratch fx{base, bytes, pad};
  RunResult r = run_range(ctx, sys, precision, ijkabc, first, last, NoSink{},
                          WindowSel{}, &fx);
  *energy = ijkabc ? r.e : -r.e;
  if (ct_energy) *ct_energy = ijkabc ? r.ect : -r.ect;
}

extern "C" {

int atrip_hip_plan_model(int64_t No, int64_t Nv, int precision, int window,
                         int *nb, int *fm, int *fn) {
  if (No < 1 || Nv < 1 || window < 0 || window > 32) return 1;
  if (precision < ATRIP_FP64 || precision > ATRIP_BF16X3) return 1;
  // the same choices as window_edge and the doubles launchers make
  const int e = window > 0 ? window : auto_window(No, Nv);
  int m, n;
  if (precision == ATRIP_FP64) {
    const int t = pick_tile(-1, No, e);
    m = tile_fm(t);
    n = tile_fn(t);
  } else {
    const int t = pick_t32_tile(-1, No, e);
    m = t32_fm(t);
    n = t32_fn(t);
  }
  if (nb) *nb = e;
  if (fm) *fm = m;
  if (fn) *fn = n;
  return 0;
}

int atrip_hip_device_count(void) {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess) return 0;
  return n;
}

int atrip_hip_create(int device, atrip_hip_ctx **out) {
  if (!out) return 1;
  *out = nullptr;
  auto *ctx = new atrip_hip_ctx();
  ctx->device = device;
  int rc = guarded(ctx, [&] {
    int n = 0;
    check(hipGetDeviceCount(&n), "hipGetDeviceCount");
    if (device < 0 || device >= n)
      throw Fail{"device index " + std::to_string(device) + " out of range (" +
                 std::to_string(n) + " devices)"};
    check(hipSetDevice(device), "hipSetDevice");
    check(hipStreamCreate(&ctx->stream), "hipStreamCreate");
  });
  if (rc) {
    static thread_local std::string last;
    last = ctx->err;
    delete ctx;
    return rc;
  }
  std::lock_guard<std::mutex> all(contexts_mutex);
  contexts.push_back(ctx);
  *out = ctx;
  return 0;
}

int atrip_hip_destroy(atrip_hip_ctx *ctx) {
  if (!ctx) return 0;
  {
    std::lock_guard<std::mutex> all(contexts_mutex);
    contexts.erase(std::find(contexts.begin(), contexts.end(), ctx));
  }
  (void)hipSetDevice(ctx->device);
  if (ctx->stream) (void)hipStreamSynchronize(ctx->stream);
  for (auto &kv : ctx->systems) free_system(kv.second);
  if (ctx->G) (void)hipFree(ctx->G);
  if (ctx->e_slot) (void)hipFree(ctx->e_slot);
  if (ctx->partials) (void)hipFree(ctx->partials);
  if (ctx->sel) (void)hipFree(ctx->sel);
  if (ctx->bscratch) (void)hipFree(ctx->bscratch);
  if (ctx->wcube) (void)hipFree(ctx->wcube);
  if (ctx->stream) (void)hipStreamDestroy(ctx->stream);
  delete ctx;
  return 0;
}

const char *atrip_hip_last_error(atrip_hip_ctx *ctx) {
  return ctx ? ctx->err.c_str() : "null context";
}

int atrip_hip_upload(atrip_hip_ctx *ctx, const atrip_sys_desc *desc,
                     int *sys) {
  return guarded_memory(ctx, [&] {
    if (!desc || !sys) throw Fail{"null argument"};
    if (!desc->ei || !desc->ea || !desc->Tai || !desc->Tabij ||
        !desc->Vabij || !desc->Vijka || !desc->Vabci)
      throw Fail{"missing input tensor"};
    if ((desc->Jijka == nullptr) != (desc->Jabci == nullptr))
      throw Fail{"Jijka and Jabci must be given together"};
    check(hipSetDevice(ctx->device), "hipSetDevice");
    DevSystem s;
    try {
      alloc_system(ctx, s, desc->No, desc->Nv, desc->Jijka != nullptr);
      DescSource src(desc, 1);
      upload_tensors(ctx, s, nullptr, src);
    } catch (...) {
      free_system(s);
      throw;
    }
    *sys = add_system(ctx, std::move(s));
  });
}

int atrip_hip_upload_synthetic(atrip_hip_ctx *ctx, int64_t No, int64_t Nv,
                               uint64_t seed, int with_j, int *sys) {
  return atrip_hip_upload_synthetic_scaled(ctx, No, Nv, seed, with_j, 1.0,
                                           sys);
}

int atrip_hip_upload_synthetic_scaled(atrip_hip_ctx *ctx, int64_t No,
                                      int64_t Nv, uint64_t seed, int with_j,
                                      double scale, int *sys) {
  return guarded_memory(ctx, [&] {
    if (!sys) throw Fail{"null argument"};
    if (!std::isfinite(scale)) throw Fail{"scale must be finite"};
    check(hipSetDevice(ctx->device), "hipSetDevice");
    DevSystem s;
    try {
      alloc_system(ctx, s, No, Nv, with_j != 0);
      fill_tables(s, ctx->stream);
      check(launch_synth(s, seed, with_j != 0, ctx->stream, 0, scale),
            "synthetic fill");
      check(hipStreamSynchronize(ctx->stream), "synthetic fill");
    } catch (...) {
      free_system(s);
      throw;
    }
    *sys = add_system(ctx, std::move(s));
  });
}

int atrip_hip_upload_complex(atrip_hip_ctx *ctx, const atrip_sys_desc *desc,
                             int *sys) {
  return guarded_memory(ctx, [&] {
    if (!desc || !sys) throw Fail{"null argument"};
    if (!desc->ei || !desc->ea || !desc->Tai || !desc->Tabij ||
        !desc->Vabij || !desc->Vijka || !desc->Vabci)
      throw Fail{"missing input tensor"};
    if ((desc->Jijka == nullptr) != (desc->Jabci == nullptr))
      throw Fail{"Jijka and Jabci must be given together"};
    check(hipSetDevice(ctx->device), "hipSetDevice");
    DevSystem s;
    try {
      alloc_system(ctx, s, desc->No, desc->Nv, desc->Jijka != nullptr, true);
      // real and imaginary planes from the interleaved values in one pass
      DescSource src(desc, 2);
      DevSystem im = imag_view(s);
      upload_tensors(ctx, s, &im, src);
      complex_negations(ctx, s);
    } catch (...) {
      free_system(s);
      throw;
    }
    *sys = add_system(ctx, std::move(s));
  });
}

int atrip_hip_upload_stream(atrip_hip_ctx *ctx, int64_t No, int64_t Nv,
                            int flags, atrip_read_fn read, void *user,
                            int *sys) {
  return guarded_memory(ctx, [&] {
    if (!read || !sys) throw Fail{"null argument"};
    if (flags & ~(ATRIP_STREAM_WITH_J | ATRIP_STREAM_COMPLEX))
      throw Fail{"unknown upload flags"};
    check(hipSetDevice(ctx->device), "hipSetDevice");
    const bool with_j = flags & ATRIP_STREAM_WITH_J;
    const bool cplx = flags & ATRIP_STREAM_COMPLEX;
    DevSystem s;
    try {
      alloc_system(ctx, s, No, Nv, with_j, cplx);
      ReaderSource src(read, user, cplx ? 2 : 1,
                       std::min<int64_t>(ctx->stage_kb * 1024, PINNED_MAX));
      if (cplx) {
        DevSystem im = imag_view(s);
        upload_tensors(ctx, s, &im, src);
        complex_negations(ctx, s);
      } else {
        upload_tensors(ctx, s, nullptr, src);
      }
    } catch (...) {
      (void)hipStreamSynchronize(ctx->stream);
      free_system(s);
      throw;
    }
    *sys = add_system(ctx, std::move(s));
  });
}

int atrip_hip_upload_synthetic_complex(atrip_hip_ctx *ctx, int64_t No,
                                       int64_t Nv, uint64_t seed, int with_j,
                                       int *sys) {
  return guarded_memory(ctx, [&] {
    if (!sys) throw Fail{"null argument"};
    check(hipSetDevice(ctx->device), "hipSetDevice");
    DevSystem s;
    try {
      alloc_system(ctx, s, No, Nv, with_j != 0, true);
      fill_tables(s, ctx->stream);
      check(launch_synth(s, seed, with_j != 0, ctx->stream), "synthetic fill");
      DevSystem v = imag_view(s);
      check(launch_synth(v, seed, with_j != 0, ctx->stream, ATRIP_SYN_IMAG),
            "synthetic fill (im)");
      check(hipStreamSynchronize(ctx->stream), "synthetic fill");
      complex_negations(ctx, s);
    } catch (...) {
      free_system(s);
      throw;
    }
    *sys = add_system(ctx, std::move(s));
  });
}

int atrip_hip_release(atrip_hip_ctx *ctx, int sys) {
  return guarded(ctx, [&] {
    std::lock_guard<std::mutex> use(ctx->in_use);
    DevSystem &s = get_sys(ctx, sys);
    check(hipStreamSynchronize(ctx->stream), "sync");
    free_system(s);
    ctx->systems.erase(sys);
    ctx->plans.erase(sys);
  });
}

int atrip_hip_run(atrip_hip_ctx *ctx, int sys, int precision, int ijkabc,
                  uint64_t first, uint64_t count, double *energy,
                  double *ct_energy) {
  return guarded_memory(ctx, [&] {
    if (!energy) throw Fail{"null energy pointer"};
    check(hipSetDevice(ctx->device), "hipSetDevice");
    const uint64_t last =
        count == ~0ULL || first + count < first ? ~0ULL : first + count;
    RunResult r = run_range(ctx, sys, precision, ijkabc, first, last, NoSink{});
    // src/atrip/Atrip.cxx:1108-1111: E = -sum unless ijkabc
    *energy = ijkabc ? r.e : -r.e;
    if (ct_energy) *ct_energy = ijkabc ? r.ect : -r.ect;
  });
}

int atrip_hip_run_windows(atrip_hip_ctx *ctx, int sys, int precision,
                          int ijkabc, uint64_t stride, uint64_t offset,
                          double *energy, double *ct_energy,
                          uint64_t *tuples) {
  return guarded_memory(ctx, [&] {
    if (!energy) throw Fail{"null energy pointer"};
    if (stride == 0) throw Fail{"stride must be positive"};
    check(hipSetDevice(ctx->device), "hipSetDevice");
    WindowSel ws;
    ws.stride = stride;
    ws.offset = offset;
    RunResult r = run_range(ctx, sys, precision, ijkabc, 0, ~0ULL, NoSink{}, ws);
    *energy = ijkabc ? r.e : -r.e;
    if (ct_energy) *ct_energy = ijkabc ? r.ect : -r.ect;
    if (tuples) *tuples = r.tuples;
  });
}

int atrip_hip_tuple_energies(atrip_hip_ctx *ctx, int sys, int precision,
                             int ijkabc, uint64_t first, uint64_t count,
                             double *e, double *e_ct) {
  return guarded_memory(ctx, [&] {
    if (!e) throw Fail{"null output pointer"};
    check(hipSetDevice(ctx->device), "hipSetDevice");
    DevSystem &s = get_sys(ctx, sys);
    const uint64_t n = n_tuples(s.Nv);
    if (first > n) first = n;
    if (count > n - first) count = n - first;
    const uint64_t last = first + count;
    HostIndex hidx((uint64_t)s.Nv);
    struct Sink {
      static constexpr bool window_sums() { return false; }
      bool active() const { return true; }
      const HostIndex *h;
      uint64_t first, last, Nv;
      double *e, *ect;
      void operator()(const int32_t *win, const BatchArgs &b,
                      const std::vector<double> &slots) {
        size_t q = 0;
        for (int w = 0; w < b.nw; w++)
          for (int ta = 0; ta < b.ea; ta++)
            for (int tb = 0; tb < b.eb; tb++)
              for (int tc = 0; tc < b.ec; tc++, q++) {
                const uint64_t x = (uint64_t)win[3 * w] + ta,
                               y = (uint64_t)win[3 * w + 1] + tb,
                               z = (uint64_t)win[3 * w + 2] + tc;
                if (!tuple_ok(Nv, x, y, z)) continue;
                const uint64_t idx = (*h)(x, y, z);
                if (idx < first || idx >= last) continue;
                e[idx - first] = slots[2 * q];
                if (ect) ect[idx - first] = slots[2 * q + 1];
              }
      }
    } sink{&hidx, first, last, (uint64_t)s.Nv, e, e_ct};
    run_range(ctx, sys, precision, ijkabc, first, last, sink);
  });
}

int atrip_hip_set_option(atrip_hip_ctx *ctx, const char *key, int64_t value) {
  return guarded(ctx, [&] {
    const std::string k = key ? key : "";
    if (k == "window") {
      if (value < 0 || value > 32)
        throw Fail{"window must be in 0..32 (0: automatic)"};
      ctx->window = (int)value;
    } else if (k == "batch") {
      if (value < 0 || value > 4096)
        throw Fail{"batch must be in 0..4096 (0: automatic)"};
      ctx->batch = (int)value;
    } else if (k == "timing") {
      ctx->timing = value != 0;
    } else if (k == "tile") {
      if (value < -1 || value > 9) throw Fail{"tile must be in -1..9"};
      ctx->tile = (int)value;
    } else if (k == "operand_store") {
      if (value < 0 || value > 3)
        throw Fail{"operand_store must be 0, 1, 2 or 3"};
      ctx->operand_store = (int)value;
    } else if (k == "serve_plain_no") {
      if (value < 1 || value > (1 << 20))
        throw Fail{"serve_plain_no must be in 1..1048576"};
      ctx->serve_plain_no = (int)value;
    } else if (k == "epilogue") {
      if (value < 0 || value > 1) throw Fail{"epilogue must be 0 or 1"};
      ctx->epilogue = (int)value;
    } else if (k == "stage_kb") {
      if (value < 1 || value > ((int64_t)1 << 30))
        throw Fail{"stage_kb must be in 1..2^30"};
      ctx->stage_kb = value;
    } else if (k == "batch_scratch_mb") {
      if (value < 16 || value > (1 << 18))
        throw Fail{"batch_scratch_mb must be in 16..262144"};
      ctx->batch_scratch_mb = value;
    } else if (k == "batch_grid") {
      if (value < 0 || value > (1 << 20))
        throw Fail{"batch_grid must be in 0..1048576"};
      ctx->batch_grid = (int)value;
    } else if (k == "batch_order") {
      if (value < 0 || value > 1) throw Fail{"batch_order must be 0 or 1"};
      ctx->batch_order = (int)value;
    } else if (k == "batch_nb") {
      if (value != 0 && value != 1 && value != 2 && value != 4 && value != 8)
        throw Fail{"batch_nb must be 0, 1, 2, 4 or 8"};
      ctx->batch_nb = (int)value;
    } else if (k == "batch_tile") {
      if (value < -1 || value >= N_BTILES)
        throw Fail{"batch_tile must be in -1.." + std::to_string(N_BTILES - 1)};
      ctx->batch_tile = (int)value;
    } else {
      throw Fail{"unknown option '" + k + "'"};
    }
  });
}

int atrip_hip_get_option(atrip_hip_ctx *ctx, const char *key, int64_t *value) {
  return guarded(ctx, [&] {
    const std::string k = key ? key : "";
    if (!value) throw Fail{"null value pointer"};
    if (k == "window") *value = ctx->window;
    else if (k == "batch") *value = ctx->batch;
    else if (k == "timing") *value = ctx->timing;
    else if (k == "tile") *value = ctx->tile;
    else if (k == "operand_store") *value = ctx->operand_store;
    else if (k == "stage_kb") *value = ctx->stage_kb;
    else if (k == "epilogue") *value = ctx->epilogue;
    else if (k == "serve_plain_no") *value = ctx->serve_plain_no;
    else if (k == "batch_scratch_mb") *value = ctx->batch_scratch_mb;
    else if (k == "batch_grid") *value = ctx->batch_grid;
    else if (k == "batch_order") *value = ctx->batch_order;
    else if (k == "batch_nb") *value = ctx->batch_nb;
    else if (k == "batch_tile") *value = ctx->batch_tile;
    else throw Fail{"unknown option '" + k + "'"};
  });
}

int atrip_hip_kernel_stats(atrip_hip_ctx *ctx, const char *name,
                           uint64_t *launches, double *total_ms,
                           double *flop) {
  return guarded(ctx, [&] {
    const KernelStat k = ctx->stats[name ? name : ""];
    if (launches) *launches = k.launches;
    if (total_ms) *total_ms = k.ms;
    if (flop) *flop = k.flop;
  });
}

int atrip_hip_reset_stats(atrip_hip_ctx *ctx) {
  return guarded(ctx, [&] { ctx->stats.clear(); });
}

int atrip_hip_sys_info(atrip_hip_ctx *ctx, int sys, int64_t *No, int64_t *Nv,
                       uint64_t *n_tup, uint64_t *device_bytes) {
  return guarded(ctx, [&] {
    std::lock_guard<std::mutex> use(ctx->in_use);
    DevSystem &s = get_sys(ctx, sys);
    if (No) *No = s.No;
    if (Nv) *Nv = s.Nv;
    if (n_tup) *n_tup = n_tuples(s.Nv);
    if (device_bytes) *device_bytes = s.bytes;
  });
}

}  // extern "C"
