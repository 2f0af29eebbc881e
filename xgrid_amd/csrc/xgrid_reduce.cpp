// FP64 reductions over the cells of one boundary class of device grids:
// difference norms (convergence tests, error against a reference field) and
// the residual of a Poisson equation.  Fields may be stored in FP32 or FP64;
// every value is widened to FP64 before it is combined.
//
// One launch with a fixed partition, so the result is deterministic: each workgroup
// reduces a fixed set of chunks (wave64 shuffles, then LDS across waves) into
// one partial, and whichever workgroup ends last reduces the partials in index
// order into host memory.  Memory bounds it (512^3 FP32, two fields, the whole call: 641 us with a
// 64-bit division per cell, a second launch and a copy of the result, 208 us so, 5.2 TB/s); of a
// small call, 18 us (26 us before), the launch and the wait are nearly all.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <type_traits>

#include "xgrid_internal.h"

using namespace xgi;

namespace {

// 512 x 512: twice as many partials, or 256 or 1024 threads, are within 1 us at 256^3.
constexpr int kRedThreads = 512;
constexpr int kRedBlocks = 512;

struct Partial {
  double sum;   // sum of squares
  double max;   // largest magnitude (NaN if any value was NaN)
};

// The larger of two magnitudes, NaN if either is (no branch: loads stay in flight around it).
__device__ __forceinline__ double nanmax(double a, double b) { return ((b > a) | (b != b)) ? b : a; }

template <class T>
__device__ __forceinline__ double load(const void* p, int64_t c) {
  return (double)static_cast<const T*>(p)[c];
}

// Reduce (s, m) over the workgroup; thread 0 returns the result.
__device__ __forceinline__ Partial block_reduce(double s, double m) {
  for (int o = 32; o > 0; o >>= 1) {
    s += __shfl_xor(s, o, 64);
    m = nanmax(m, __shfl_xor(m, o, 64));
  }
  __shared__ double ws[kRedThreads / 64], wm[kRedThreads / 64];
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    ws[w] = s;
    wm[w] = m;
  }
  __syncthreads();
  Partial r{0.0, 0.0};
  if (threadIdx.x == 0) {
    for (int i = 0; i < kRedThreads / 64; ++i) {
      r.sum += ws[i];
      r.max = nanmax(r.max, wm[i]);
    }
  }
  return r;
}

// Visit the cells of the class (box, masked box or list), kUnroll chunks of 64 cells per wave
// and turn: v = load(c) of each cell's linear index c first, so that their loads are in flight
// together, then use(v, valid) (a lane without a cell repeats the last one, not valid).
//   wide box    a chunk is 64 columns of one row: the wave divides once per turn and steps on
//   narrow box  (rows of at most 32 cells) a chunk is 64 >> lg rows of 1 << lg lanes; a
//               one-cell-wide wall of 512^2 cells would otherwise take a turn per 4 cells
//   list        a chunk is 64 entries
// The 64-bit division per cell that this replaces kept the vector units as busy as the loads.
constexpr int kUnroll = 4;
__device__ __forceinline__ uint64_t udiv(uint64_t a, uint32_t b) { return a >> 32 ? a / b : (uint32_t)a / b; }
template <class L, class U>
__device__ __forceinline__ void for_class(const xg_dom& dom, int32_t s1, int32_t s2, int64_t chunks, L&& load, U&& use) {
  const uint32_t lane = threadIdx.x & 63;
  const int64_t wave = blockIdx.x * (kRedThreads / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t step = (int64_t)gridDim.x * (kRedThreads / 64) * kUnroll;
  const uint32_t e0 = (uint32_t)(dom.hi[0] - dom.lo[0]), e1 = (uint32_t)(dom.hi[1] - dom.lo[1]);
  const uint32_t e2 = (uint32_t)(dom.hi[2] - dom.lo[2]);
  const int64_t origin = ((int64_t)dom.lo[0] * s1 + dom.lo[1]) * s2 + dom.lo[2];
  for (int64_t q = wave * kUnroll; q < chunks; q += step) {
    int64_t c[kUnroll];
    bool ok[kUnroll];
    if (dom.kind == XG_DOM_LIST) {
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        const int64_t k = (q + u) * 64 + lane;
        ok[u] = k < dom.count;
        c[u] = dom.list[ok[u] ? k : dom.count - 1];
      }
    } else {
      if (e2 > 32) {
        const uint32_t per_row = (e2 + 63) / 64;
        const uint64_t row = udiv((uint64_t)q, per_row);
        uint32_t ch = (uint32_t)(q - row * per_row), i0 = (uint32_t)udiv(row, e1), i1 = (uint32_t)(row - (uint64_t)i0 * e1);
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
          const uint32_t col = ch * 64 + lane;
          ok[u] = (q + u < chunks) & (col < e2);
          c[u] = origin + ((int64_t)i0 * s1 + i1) * s2 + (col < e2 ? col : e2 - 1);
          if (q + u + 1 < chunks && ++ch == per_row) {
            ch = 0;
            if (++i1 == e1) i1 = 0, ++i0;
          }
        }
      } else {
        const uint32_t lg = e2 > 1 ? 32 - __builtin_clz(e2 - 1) : 0;
        const uint32_t col = lane & ((1u << lg) - 1);
        const int64_t rows = (int64_t)e0 * e1;
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
          const int64_t r = ((q + u) << (6 - lg)) + (lane >> lg);
          ok[u] = (r < rows) & (col < e2);
          const int64_t row = r < rows ? r : rows - 1, i0 = (int64_t)udiv((uint64_t)row, e1);
          c[u] = origin + (i0 * s1 + (row - i0 * e1)) * s2 + (col < e2 ? col : e2 - 1);
        }
      }
      if (dom.kind == XG_DOM_MASKED) {
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) ok[u] = (dom.mask[c[u]] == dom.klass) & ok[u];
      }
    }
    decltype(load(c[0])) v[kUnroll];
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) v[u] = load(c[u]);
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) use(v[u], ok[u]);
  }
}

// This workgroup's partial; the last workgroup to end reduces all of them in index order.
// Partials and counts travel as atomics, which act where every XCD sees them: an exchange
// has been performed there once its old value is back, so the count that announces a
// partial waits for that.  (A device-wide fence instead writes an XCD's whole L2 back: with one
// per workgroup a 256^3 FP32 norm took 67 us instead of 51.)  Counts are taken in two steps,
// one line of memory per eighth of the workgroups and one for the eighths, and wrap, so they
// are 0 again for the next launch.
constexpr int kDoneLines = 9, kDoneLine = 32;   // lines of 128 bytes
__device__ __forceinline__ void publish(double* to, double v) {
  const uint64_t old = __hip_atomic_exchange((uint64_t*)to, __double_as_longlong(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  asm volatile("s_waitcnt vmcnt(0)" ::"v"(old) : "memory");
}
__device__ __forceinline__ bool is_last(uint32_t* count, uint32_t n) {
  const uint32_t before = __hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (before != n - 1) return false;
  __hip_atomic_store(count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return true;
}
__device__ __forceinline__ double published(const double* p) {
  return __longlong_as_double(__hip_atomic_load((const uint64_t*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}
__device__ __forceinline__ void finish_block(double s, double m, Partial* part, uint32_t* done, Partial* out) {
  const Partial r = block_reduce(s, m);
  __shared__ bool last;
  if (threadIdx.x == 0) {
    publish(&part[blockIdx.x].sum, r.sum);
    publish(&part[blockIdx.x].max, r.max);
    const uint32_t n = gridDim.x, x = blockIdx.x % 8;
    last = is_last(done + x * kDoneLine, (n - x + 7) / 8) && is_last(done + 8 * kDoneLine, n < 8 ? n : 8);
  }
  __syncthreads();
  if (!last) return;
  double ts = 0.0, tm = 0.0;
  for (uint32_t i = threadIdx.x; i < gridDim.x; i += kRedThreads) {
    ts += published(&part[i].sum);
    tm = nanmax(tm, published(&part[i].max));
  }
  const Partial t = block_reduce(ts, tm);
  if (threadIdx.x == 0) *out = t;
}

// a, b: element types (float / double); b may be null.
template <class TA, class TB, bool HAS_B>
__global__ void __launch_bounds__(kRedThreads) diff_norm(const void* a, const void* b, xg_dom dom, int32_t s1,
                                                         int32_t s2, int64_t chunks, Partial* part, uint32_t* done,
                                                         Partial* out) {
  double s = 0.0, m = 0.0;
  for_class(dom, s1, s2, chunks,
            [&](int64_t c) {
              double d = load<TA>(a, c);
              if constexpr (HAS_B) d -= load<TB>(b, c);
              return d;
            },
            [&](double x, bool valid) {
              const double d = valid ? x : 0.0;
              s += d * d;
              m = nanmax(m, d < 0 ? -d : d);
            });
  finish_block(s, m, part, done, out);
}

// r = sum_a coef[a] * (p[+e_a] - 2 p + p[-e_a]) - scale * rhs over class cells
// (every class cell is at least one cell inside the grid: checked on the host).
template <class TP, class TR, int DIMS>
__global__ void __launch_bounds__(kRedThreads) poisson_norm(const void* p, const void* rhs, xg_dom dom, int32_t s1,
                                                            int32_t s2, double c0, double c1, double c2, double scale,
                                                            int64_t chunks, Partial* part, uint32_t* done,
                                                            Partial* out) {
  const int64_t st[3] = {(int64_t)s1 * s2, s2, 1};
  const double cf[3] = {c0, c1, c2};
  double s = 0.0, m = 0.0;
  for_class(dom, s1, s2, chunks,
            [&](int64_t c) {
              const double pc = load<TP>(p, c);
              double lap = 0.0;
#pragma unroll
              for (int a = 0; a < DIMS; ++a) {
                const int ax = 3 - DIMS + a;   // grid axis a is stored as axis ax of the padded 3-D shape
                lap += cf[a] * ((load<TP>(p, c + st[ax]) - 2.0 * pc) + load<TP>(p, c - st[ax]));
              }
              return lap - scale * load<TR>(rhs, c);
            },
            [&](double x, bool valid) {
              const double r = valid ? x : 0.0;
              s += r * r;
              m = nanmax(m, r < 0 ? -r : r);
            });
  finish_block(s, m, part, done, out);
}

Partial* g_part = nullptr;   // kRedBlocks partials, kept for the process

// Scratch of the allocation-free entry point (xg_grid_norm_diff_noalloc): the
// same kRedBlocks partials, in device memory that
// every GPU the library runs on holds until the process ends.  In host code
// `scratch` names a host-side stand-in, not a device address: set-up looks up
// each device's copy once (reduce_setup, from xg_init) and only that address
// is passed to kernels.
static __device__ __align__(256) Partial scratch[kRedBlocks];
// Workgroups done, one set of counts per scratch (finish_block).
static __device__ __align__(128) uint32_t done_count[2][kDoneLines * kDoneLine];
constexpr int kMaxDevices = 64;
Partial* g_scratch[kMaxDevices] = {};
uint32_t* g_done[kMaxDevices] = {};
// Results, one per scratch: host memory that kernels write, read after a wait for the stream
// (a copy of 16 bytes out of device memory, and its launch, took 15 us more).
Partial* g_result = nullptr;

int ensure_partials() {
  if (g_part) return XG_OK;
  void* p = nullptr;
  XG_HIP(hipMalloc(&p, sizeof(Partial) * kRedBlocks));
  g_part = (Partial*)p;
  return XG_OK;
}

// Cells of class `klass` of G as a 3-D padded domain (axes shifted so the last
// grid axis is the contiguous one); returns the number of 64-lane chunks for_class cuts them into.
int64_t class_domain(const xg_grid* G, int32_t klass, xg_dom& dom, int32_t* shape3) {
  const ClassPlan& p = G->plan(klass);
  std::memset(&dom, 0, sizeof dom);
  dom.kind = p.kind;
  dom.klass = klass;
  dom.count = p.count;
  dom.list = p.d_list;
  dom.mask = G->d_mask;
  const int D = G->dims;
  for (int a = 0; a < 3; ++a) {
    const int g = a - (3 - D);      // grid axis of padded axis a
    shape3[a] = g >= 0 ? G->shape[g] : 1;
    dom.lo[a] = g >= 0 ? p.lo[g] : 0;
    dom.hi[a] = g >= 0 ? p.hi[g] : 1;
  }
  const int64_t rows = (int64_t)(dom.hi[0] - dom.lo[0]) * (dom.hi[1] - dom.lo[1]);
  const int64_t e2 = dom.hi[2] - dom.lo[2];
  if (p.kind == XG_DOM_EMPTY || p.count == 0) return 0;
  if (p.kind == XG_DOM_LIST) return ceil_div(p.count, 64);
  if (e2 > 32) return rows * ceil_div(e2, 64);
  int lg = 0;
  while ((int64_t)1 << lg < e2) ++lg;
  return ceil_div(rows, (int64_t)64 >> lg);
}

// Where one reduction's partials, count and result go: scratch 0 or 1.  Held from the launch until
// the result is read: calls of several threads take turns.
std::mutex g_space[2];
struct RedSpace {
  Partial* part;
  uint32_t* done;
  Partial* out;
  std::unique_lock<std::mutex> held;
};

int red_space(int which, RedSpace& r) {
  if (g_dev.id < 0 || g_dev.id >= kMaxDevices || !g_done[g_dev.id] || !g_result)
    return fail(XG_ERR_STATE, "the device's scratch address was not looked up (xg_init)");
  r.held = std::unique_lock<std::mutex>(g_space[which]);
  if (!which)
    if (int rc = ensure_partials()) return rc;
  r.part = which ? g_scratch[g_dev.id] : g_part;
  r.done = g_done[g_dev.id] + which * kDoneLines * kDoneLine;
  r.out = g_result + which;
  return XG_OK;
}

int red_blocks(int64_t chunks) {
  return (int)std::min<int64_t>(kRedBlocks, ceil_div(chunks, kUnroll * (kRedThreads / 64)));
}

int finish(int64_t chunks, double* l2, double* linf, const Partial* out) {
  Partial h{0.0, 0.0};
  if (chunks > 0) {
    XG_HIP(hipGetLastError());
    XG_HIP(hipStreamSynchronize(g_dev.stream));
    h = *out;
  }
  if (l2) *l2 = std::sqrt(h.sum);
  if (linf) *linf = h.max;
  return XG_OK;
}

bool float_type(int32_t t) { return t == XG_T_F32 || t == XG_T_F64; }

// L2 / Linf of a - b over class klass of a.  Every partial the last workgroup reads is
// written by the same call first, so nothing needs clearing.
int norm_diff(xg_grid* a, int32_t level_a, int32_t type_a, xg_grid* b, int32_t level_b, int32_t type_b,
              int32_t klass, double* l2, double* linf, int64_t* cells, const RedSpace& sp) {
  if (!a || level_a < 0 || level_a >= (int32_t)a->levels.size() || !float_type(type_a))
    return fail(XG_ERR_ARG, "invalid first grid, level or element type");
  if (b && (level_b < 0 || level_b >= (int32_t)b->levels.size() || !float_type(type_b)))
    return fail(XG_ERR_ARG, "invalid second grid, level or element type");
  if (b && (b->dims != a->dims || std::memcmp(b->shape, a->shape, sizeof a->shape) != 0))
    return fail(XG_ERR_ARG, "grids of different shapes");
  if ((int64_t)a->elem != (type_a == XG_T_F32 ? 4 : 8) || (b && (int64_t)b->elem != (type_b == XG_T_F32 ? 4 : 8)))
    return fail(XG_ERR_ARG, "element type does not match the grid's element size");
  xg_dom dom;
  int32_t sh[3];
  const int64_t chunks = class_domain(a, klass, dom, sh);
  if (cells) *cells = a->plan(klass).count;
  if (chunks > 0) {
    const void* pa = a->levels[(size_t)level_a];
    const void* pb = b ? b->levels[(size_t)level_b] : nullptr;
    const bool fa = type_a == XG_T_F32, fb = type_b == XG_T_F32;
    auto* k = !b ? (fa ? diff_norm<float, float, false> : diff_norm<double, double, false>)
              : fa ? (fb ? diff_norm<float, float, true> : diff_norm<float, double, true>)
                   : (fb ? diff_norm<double, float, true> : diff_norm<double, double, true>);
    hipLaunchKernelGGL(k, dim3(red_blocks(chunks)), dim3(kRedThreads), 0, g_dev.stream, pa, pb, dom, sh[1], sh[2], chunks,
                       sp.part, sp.done, sp.out);
  }
  return finish(chunks, l2, linf, sp.out);
}

}  // namespace

namespace xgi {

int reduce_setup(int device) {
  if (device < 0 || device >= kMaxDevices) return fail(XG_ERR_ARG, "device index beyond the scratch table");
  if (g_scratch[device]) return XG_OK;
  void* p = nullptr;
  XG_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(done_count)));
  g_done[device] = (uint32_t*)p;
  if (!g_result) XG_HIP(hipHostMalloc((void**)&g_result, 2 * sizeof(Partial), hipHostMallocPortable));
  XG_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
  g_scratch[device] = (Partial*)p;
  return XG_OK;
}

}  // namespace xgi

extern "C" {

int xg_grid_norm_diff(xg_grid* a, int32_t level_a, int32_t type_a, xg_grid* b, int32_t level_b, int32_t type_b,
                      int32_t klass, double* l2, double* linf, int64_t* cells) {
  if (int rc = check_ready()) return rc;
  RedSpace sp;
  if (int rc = red_space(0, sp)) return rc;
  return norm_diff(a, level_a, type_a, b, level_b, type_b, klass, l2, linf, cells, sp);
}

int xg_grid_norm_diff_noalloc(xg_grid* a, int32_t level_a, int32_t type_a, xg_grid* b, int32_t level_b,
                              int32_t type_b, int32_t klass, double* l2, double* linf, int64_t* cells) {
  if (int rc = check_ready()) return rc;
  // The partials fit whatever the class size: at most kRedBlocks workgroups.
  RedSpace sp;
  if (int rc = red_space(1, sp)) return rc;
  return norm_diff(a, level_a, type_a, b, level_b, type_b, klass, l2, linf, cells, sp);
}

int xg_grid_poisson_residual(xg_grid* p, int32_t level_p, int32_t type_p, xg_grid* rhs, int32_t level_rhs,
                             int32_t type_rhs, int32_t klass, const double* coef, double rhs_scale, double* l2,
                             double* linf) {
  if (int rc = check_ready()) return rc;
  if (!p || !rhs || !coef || level_p < 0 || level_p >= (int32_t)p->levels.size() || level_rhs < 0 ||
      level_rhs >= (int32_t)rhs->levels.size() || !float_type(type_p) || !float_type(type_rhs))
    return fail(XG_ERR_ARG, "invalid grid, level, element type or coefficients");
  if (rhs->dims != p->dims || std::memcmp(rhs->shape, p->shape, sizeof p->shape) != 0)
    return fail(XG_ERR_ARG, "grids of different shapes");
  if ((int64_t)p->elem != (type_p == XG_T_F32 ? 4 : 8) || (int64_t)rhs->elem != (type_rhs == XG_T_F32 ? 4 : 8))
    return fail(XG_ERR_ARG, "element type does not match the grid's element size");
  const ClassPlan& cp = p->plan(klass);
  if (cp.kind != XG_DOM_EMPTY && cp.count > 0)
    for (int a = 0; a < p->dims; ++a)
      if (cp.lo[a] < 1 || cp.hi[a] > p->shape[a] - 1)
        return fail(XG_ERR_ARG, "the class reaches the edge of the grid: the residual's stencil would leave it");
  RedSpace sp;
  if (int rc = red_space(0, sp)) return rc;
  xg_dom dom;
  int32_t sh[3];
  const int64_t chunks = class_domain(p, klass, dom, sh);
  if (chunks > 0) {
    double c[3] = {0.0, 0.0, 0.0};
    for (int a = 0; a < p->dims; ++a) c[a] = coef[a];
    const bool fp = type_p == XG_T_F32, fr = type_rhs == XG_T_F32;
    auto pick = [&](auto dims) {
      constexpr int D = decltype(dims)::value;
      return fp ? (fr ? poisson_norm<float, float, D> : poisson_norm<float, double, D>)
                : (fr ? poisson_norm<double, float, D> : poisson_norm<double, double, D>);
    };
    auto* k = p->dims == 1 ? pick(std::integral_constant<int, 1>())
              : p->dims == 2 ? pick(std::integral_constant<int, 2>()) : pick(std::integral_constant<int, 3>());
    hipLaunchKernelGGL(k, dim3(red_blocks(chunks)), dim3(kRedThreads), 0, g_dev.stream, p->levels[(size_t)level_p],
                       rhs->levels[(size_t)level_rhs], dom, sh[1], sh[2], c[0], c[1], c[2], rhs_scale, chunks, sp.part,
                       sp.done, sp.out);
  }
  return finish(chunks, l2, linf, sp.out);
}

}  // extern "C"
