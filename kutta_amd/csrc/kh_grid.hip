// The coarse part of the V-cycle in one launch of several workgroups (no
// reference counterpart; bitwise the per-level launches of kh_linalg.hip).
//
// What bounds it: below about 20,000 rows a level's launch costs 4-7 us
// whatever it computes (a kernel boundary and three dependent memory round
// trips), and a V(5,5) cycle makes about 12 of them per level and 32 on the
// coarsest. One workgroup (the coarse tail) pays no launches but computes on
// one CU. Here the rows of every level are split over `parts` workgroups that
// stay on one XCD and keep their operators in LDS for the whole cycle. A sweep
// then takes 2.3 to 2.5 us (1.3 the rows' serial sums, 0.6 the barrier, 0.4 the
// window); a pressure solve (AMG-PCG, V(5,5)) of 10,368 cells takes 2.6 ms and
// without it 4.6, of 78,246 4.9 and 5.8, of 998,250 17.3 and 18.3 (the rule
// that picks the first level has the whole table). 512 or 256 threads instead
// of 1024 measured the same on small levels, slower on large.
//
// Exchange: a sweep's new values go out as write-through stores and come in,
// after a barrier over the workgroups, as one coalesced window of the iterate
// per workgroup, from that XCD's L2. (Values tagged with their step and polled
// by their readers, without a barrier, measured slower: the polls of 8 to 32
// workgroups slow the stores they wait for.)
//
// Which workgroups take part: the launch has 8 x parts workgroups, dispatched
// round-robin over the XCDs; those that find themselves on the control
// block's home XCD take a rank, the others leave at once. Nothing depends on
// that placement but speed: the exchanged data is read and written with
// agent-scope accesses, and when not exactly `parts` workgroups meet within
// the time limit (another stream's kernel holds the CUs), one workgroup does
// the whole cycle by itself from global memory (solo_cycle). No workgroup
// waits for one that may not be running: the barrier is used only after all
// have met.
#include "kh_device_math.hpp"
#include "kh_grid_gather.hpp"

namespace kh {
namespace {

constexpr int kGridThreads = 1024;
constexpr int kCoarseMax = 24;  // largest coarsest level solved by amg_coarse_solve (linalg/amg.cpp:287)
constexpr int kMaxLevels = 16;

__device__ __forceinline__ unsigned xcc_id() {
  unsigned v;
  asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(v));
  return v & 15u;
}
// Global memory through a pointer of its own address space, where the pointer
// comes out of a table and would be taken for a generic one.
#define GLOBAL __attribute__((address_space(1)))
// Exchanged data: agent-scope relaxed accesses are served by the L2 (and
// written through), past the CU's own vector cache.
__device__ __forceinline__ float exchange_load(const float* p) {
  return __uint_as_float(__hip_atomic_load((const GLOBAL unsigned*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}
__device__ __forceinline__ void exchange_store(float* p, float v) {
  __hip_atomic_store((GLOBAL unsigned*)p, __float_as_uint(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned ctl_load(const unsigned* p) {
  return __hip_atomic_load((const GLOBAL unsigned*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Every earlier store of this wavefront has reached the coherence point.
__device__ __forceinline__ void stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Control block (KH_GRID_CTL_WORDS words, in cache lines of their own), as
// kh_grid_gather.hpp uses it; the limit is in ticks of the 100 MHz clock.
struct GridCtl {
  unsigned *arrived, *settled, *bar, *home, *left;
  long limit;
  long long start = 0;
  __device__ GridCtl(unsigned* w, long limit_ticks)
      : arrived(w), settled(w + 32), bar(w + 64), home(w + KH_GRID_CTL_HOME), left(w + 128), limit(limit_ticks) {}
  __device__ static unsigned add(unsigned* p, unsigned v) {
    return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __device__ unsigned arrive(unsigned v) { return add(arrived, v); }
  __device__ unsigned arrivals() { return ctl_load(arrived); }
  __device__ unsigned settle(unsigned to) {
    unsigned expected = 0;
    __hip_atomic_compare_exchange_strong(settled, &expected, to, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
    stores_done();  // also where the result is not used
    return expected;
  }
  __device__ unsigned state() { return ctl_load(settled); }
  __device__ unsigned leave() { return add(left, 1); }
  __device__ void wait() { start = wall_clock64(); }
  __device__ bool expired() { return wall_clock64() - start > limit; }
  __device__ void clear() {
    for (unsigned* p : {bar, left, settled, arrived})
      __hip_atomic_store(p, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  // Through a global pointer: behind a flat atomic the cycle's loops wait for
  // more than they need, 0.1 us a sweep.
  __device__ void count(int what) const {
    GLOBAL int* report = (GLOBAL int*)*reinterpret_cast<int**>(arrived + KH_GRID_CTL_REPORT);
    if (report != nullptr) __hip_atomic_fetch_add(report + what, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
};

// Barrier over the members: all of them are running (grid_enter), and each
// passes the same barriers, so the wait ends. It is bounded all the same: after
// `polls` polls of some 0.3 us each a member gives up, which opens this and the
// launch's later barriers to all and is reported, since the iterate is wrong.
// What this needs is kept in LDS: the cycle is short of scalar registers.
constexpr unsigned kGivenUp = 1u << 31, kBarrierPolls = 1u << 21;
struct GridWait {
  GridPlace place;
  unsigned polls, given_up;
};
__device__ __forceinline__ GridWait& grid_wait() {
  __shared__ GridWait w;
  return w;
}
__device__ __forceinline__ void grid_sync(const GridCtl& c, int parts, unsigned& passed) {
  stores_done();
  __syncthreads();
  passed += unsigned(parts);
  if (threadIdx.x == 0) {
    GLOBAL unsigned* bar = (GLOBAL unsigned*)c.bar;
    __hip_atomic_fetch_add(bar, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    unsigned polls = 0, seen;
    while ((seen = ctl_load(c.bar)) < passed && polls < grid_wait().polls) ++polls;
    if (seen < passed) {
      __hip_atomic_fetch_or(bar, kGivenUp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      grid_wait().given_up = 1;
    }
  }
  __syncthreads();
}

struct CycleArgs {
  const kh_grid_level* levels;
  const kh_grid_part* table;
  unsigned* ctl;
  int count, grid, pre, post, coarse_sweeps, parts, lds_words, limit_us;
  const float* rhs;
  float* out;
  const int* status;
};

// One workgroup, from global memory: the fallback when the others do not meet.
// Each sweep is the per-level kernels' row update (k_amg_smooth,
// k_fused_smooth_from_zero, k_fused_prolong_smooth, amg_coarse_solve).
__device__ void solo_sweep(const kh_grid_level& L, const float* in, const float* b, const float* coarse,
                           float* out, bool residual) {
  for (int i = threadIdx.x; i < L.rows; i += kGridThreads) {
    const auto gather = [&](int j) {
      const float v = exchange_load(in + j);
      if (coarse == nullptr) return v;
      const int g = L.aggregate[j];
      return g >= 0 ? v + exchange_load(coarse + g) : v;
    };
    const float r = row_residual_chunked<kChunk>(exchange_load(b + i), L.row_ptr[i], L.row_ptr[i + 1], L.col,
                                                 L.val, gather);
    exchange_store(out + i, residual ? r : gather(i) + (2.0f / 3.0f) * L.inverse[i] * r);
  }
  stores_done();
  __syncthreads();
}
__device__ void solo_zero(const kh_grid_level& L, const float* b, float* out) {
  for (int i = threadIdx.x; i < L.rows; i += kGridThreads) {
    const float bi = exchange_load(b + i), w = (2.0f / 3.0f) * L.inverse[i];
    exchange_store(out + i, bi - bi != 0.0f
                                ? 0.0f + w * row_residual_chunked<kChunk>(bi, L.row_ptr[i], L.row_ptr[i + 1], L.col,
                                                                          L.val, [](int) { return 0.0f; })
                                : 0.0f + w * (bi + 0.0f));
  }
  stores_done();
  __syncthreads();
}
__device__ void solo_cycle(const CycleArgs& A) {
  for (int k = 0; k < A.count; ++k) {
    const kh_grid_level L = A.levels[k];
    const bool coarsest = k + 1 == A.count;
    const float* b = k == 0 ? A.rhs : L.b;
    float* x = k == 0 ? A.out : L.x;
    const int pre = coarsest ? A.coarse_sweeps : A.pre, total = coarsest ? pre : pre + A.post;
    const auto target = [&](int t) { return (total - t) % 2 == 0 ? x : L.w; };
    if (coarsest && L.rows <= kCoarseMax) {
      for (int i = threadIdx.x; i < L.rows; i += kGridThreads) exchange_store(target(0) + i, 0.0f);
      stores_done();
      __syncthreads();
      for (int t = 1; t <= pre; ++t) solo_sweep(L, target(t - 1), b, nullptr, target(t), false);
      break;
    }
    solo_zero(L, b, target(1));
    for (int t = 2; t <= pre; ++t) solo_sweep(L, target(t - 1), b, nullptr, target(t), false);
    if (coarsest) break;
    float* spare = target(pre + 1);
    solo_sweep(L, target(pre), b, nullptr, spare, true);
    const kh_grid_level C = A.levels[k + 1];
    for (int g = threadIdx.x; g < C.rows; g += kGridThreads) {
      Kahan s;
      for (int m = L.member_offsets[g]; m < L.member_offsets[g + 1]; ++m) s.add(exchange_load(spare + L.members[m]));
      exchange_store(C.b + g, s.s);
    }
    stores_done();
    __syncthreads();
  }
  for (int k = A.count - 2; k >= 0; --k) {
    const kh_grid_level L = A.levels[k];
    const float* b = k == 0 ? A.rhs : L.b;
    float* x = k == 0 ? A.out : L.x;
    const int total = A.pre + A.post;
    const auto target = [&](int t) { return (total - t) % 2 == 0 ? x : L.w; };
    for (int t = A.pre + 1; t <= total; ++t)
      solo_sweep(L, target(t - 1), b, t == A.pre + 1 ? A.levels[k + 1].x : nullptr, target(t), false);
  }
}

// LDS data through pointers of its own address space (a generic pointer would
// make every access a flat one).
#define LDS __attribute__((address_space(3)))
typedef float vec4 __attribute__((ext_vector_type(4)));
typedef int quad_t __attribute__((ext_vector_type(4)));
typedef uint16_t short4_t __attribute__((ext_vector_type(4)));
extern __shared__ __align__(16) uint32_t grid_pool[];
template <class T>
__device__ __forceinline__ LDS T* lds_at(int word) {
  return (LDS T*)((LDS uint32_t*)grid_pool + word);
}

// The tables do not change during a launch: scalar loads.
#define CONSTANT __attribute__((address_space(4)))
typedef const CONSTANT kh_grid_part* PartTable;
typedef const CONSTANT kh_grid_level* LevelTable;

// One member's rows of one level, in LDS: values and window-local columns in
// padded rows, and per row its first slot, its length in chunks of kStep, the
// (2/3) l1 inverse and the right-hand side.
constexpr int kStep = 4;
constexpr uint16_t kPadCol = 0xffff;
struct GridRows {
  LDS vec4* val;
  LDS short4_t* col;
  LDS float* weight;
  LDS float* rhs;
  LDS uint16_t* place;  // in chunks
  LDS uint16_t* chunks;
  // Where a sweep forms them first: terms t = -(a x) and product errors,
  // `quads` chunks each.
  LDS vec4* term;
  LDS vec4* error;
  int first, rows, window, window_rows, quads;
  bool terms;
};
__device__ __forceinline__ GridRows grid_rows(PartTable part) {
  const CONSTANT kh_grid_part& P = *part;
  GridRows g;
  int at = P.lds;
  g.val = lds_at<vec4>(at);
  at += P.slots;
  g.col = lds_at<short4_t>(at);
  at += P.slots / 2;
  g.weight = lds_at<float>(at);
  g.rhs = g.weight + P.rows;
  g.place = (LDS uint16_t*)(g.rhs + P.rows);
  g.chunks = g.place + P.rows;
  g.quads = P.slots / kStep;
  g.term = lds_at<vec4>(P.terms);
  g.error = g.term + g.quads;
  g.first = P.first;
  g.rows = P.rows;
  g.window = P.window;
  g.window_rows = P.window_rows;
  g.terms = P.mode != 0;
  return g;
}
__device__ __forceinline__ void grid_stage(LevelTable level, PartTable part) {
  const GridRows g = grid_rows(part);
  const CONSTANT kh_grid_level& L = *level;
  const CONSTANT kh_grid_part& P = *part;
  const GLOBAL quad_t* slot = (const GLOBAL quad_t*)(L.slot + P.slot0);
  const GLOBAL short4_t* local = (const GLOBAL short4_t*)(L.local_col + P.slot0);
  const GLOBAL float* val = (const GLOBAL float*)L.val;
  for (int q = threadIdx.x; q < g.quads; q += kGridThreads) {
    const quad_t src = slot[q];
    const short4_t c = local[q];
    g.val[q] = vec4{src.x >= 0 ? val[src.x] : 1.0f, src.y >= 0 ? val[src.y] : 1.0f, src.z >= 0 ? val[src.z] : 1.0f,
                    src.w >= 0 ? val[src.w] : 1.0f};
    g.col[q] = c;
  }
  for (int r = threadIdx.x; r < g.rows; r += kGridThreads) {
    const int i = g.first + r;
    const GLOBAL int* row_ptr = (const GLOBAL int*)L.row_ptr;
    g.place[r] = uint16_t(((const GLOBAL uint16_t*)L.place)[i] / kStep);
    g.chunks[r] = uint16_t((row_ptr[i + 1] - row_ptr[i] + kStep - 1) / kStep);
    g.weight[r] = (2.0f / 3.0f) * ((const GLOBAL float*)L.inverse)[i];
  }
}

// Four entries' terms and product errors. Padding entries (value 1) carry the
// term -0 and no error, which leave a row's running sum and error as they are:
// s + (-0) = s for every s, its own error is +0, and e (which starts at +0)
// never holds -0. Rows that hold an infinity or a NaN end as NaN either way.
__device__ __forceinline__ void four_terms(vec4 a, short4_t c, const LDS float* xw, vec4& term, vec4& error) {
  float x[kStep], prod[kStep];
  bool pad[kStep], plain = true;
#pragma unroll
  for (int u = 0; u < kStep; ++u) {
    pad[u] = c[u] == kPadCol;
    x[u] = xw[pad[u] ? 0 : int(c[u])];
  }
#pragma unroll
  for (int u = 0; u < kStep; ++u) {
    x[u] = pad[u] ? 1.0f : x[u];
    prod[u] = a[u] * x[u];
    term[u] = pad[u] ? -0.0f : -prod[u];
    // Where product_error is one FMA.
    const float m = fabsf(prod[u]);
    plain = plain && m >= 0x1p-100f && m <= 0x1p100f && fabsf(a[u]) <= 1.0e30f && fabsf(x[u]) <= 1.0e30f;
    error[u] = __builtin_fmaf(a[u], x[u], -prod[u]);
  }
  if (!plain) {
#pragma unroll
    for (int u = 0; u < kStep; ++u) error[u] = product_error(a[u], x[u], prod[u]);
  }
}
__device__ __forceinline__ float correction(float s, float t, float n) {
  return fabsf(s) >= fabsf(t) ? (s - n) + t : (t - n) + s;
}
// Four steps of RowResidual::add_split.
__device__ __forceinline__ void add_four(float& s, float& e, vec4 t, vec4 x) {
  const float n0 = s + t.x, n1 = n0 + t.y, n2 = n1 + t.z, n3 = n2 + t.w;
  const float c0 = correction(s, t.x, n0), c1 = correction(n0, t.y, n1), c2 = correction(n1, t.z, n2),
              c3 = correction(n2, t.w, n3);
  e += c0;
  e -= x.x;
  e += c1;
  e -= x.y;
  e += c2;
  e -= x.z;
  e += c3;
  e -= x.w;
  s = n3;
}
// The workgroup's residuals of its rows over the window xw (RowResidual,
// entries in order): emit(r, residual, mine) is called by every lane of a
// wavefront that has a row (r clamped to the last; `mine` false beyond it).
// A row is a serial chain of nine operations per entry in one lane; with the
// products formed first by all lanes (`terms`) the lane only adds; that chain is
// what a sweep then takes (forming the corrections by all lanes too, in two more
// passes, measured no faster).
template <class Emit>
__device__ __forceinline__ void grid_residuals(const GridRows& g, const LDS float* xw, Emit emit) {
  if (g.terms) {
    for (int q = threadIdx.x; q < g.quads; q += kGridThreads) {
      vec4 t, x;
      four_terms(g.val[q], g.col[q], xw, t, x);
      g.term[q] = t;
      g.error[q] = x;
    }
    __syncthreads();
  }
  const int lane = threadIdx.x & 63;
  for (int r0 = int(threadIdx.x) - lane; r0 < g.rows; r0 += kGridThreads) {
    const int r = min(r0 + lane, g.rows - 1);
    const int begin = g.place[r], last = begin + g.chunks[r] - 1;
    float s = g.rhs[r], e = 0.0f;
    if (!g.terms) {
      for (int q = begin; q <= last; ++q) {
        vec4 t, x;
        four_terms(g.val[q], g.col[q], xw, t, x);
        add_four(s, e, t, x);
      }
    } else {
      int q = begin;
      for (; q + 1 <= last; q += 2) {
        const vec4 t0 = g.term[q], t1 = g.term[q + 1], x0 = g.error[q], x1 = g.error[q + 1];
        add_four(s, e, t0, x0);
        add_four(s, e, t1, x1);
      }
      if (q <= last) add_four(s, e, g.term[q], g.error[q]);
    }
    emit(r, s + e, r0 + lane < g.rows);
  }
}
// The first sweep's value of row r, from the zero iterate.
__device__ __forceinline__ float zero_row(const GridRows& g, int r) {
  const float b = g.rhs[r];
  if (b - b == 0.0f) return 0.0f + g.weight[r] * (b + 0.0f);
  RowResidual acc(b);
  const LDS float* val = (const LDS float*)g.val;
  const LDS uint16_t* col = (const LDS uint16_t*)g.col;
  for (int j = kStep * int(g.place[r]), end = j + kStep * int(g.chunks[r]); j < end; ++j)
    if (col[j] != kPadCol) acc.add(val[j], 0.0f);
  return 0.0f + g.weight[r] * acc.value();
}
// The window of an exchanged iterate, coalesced, with the coarse iterate
// (null: none) added: x + P c.
__device__ __forceinline__ void load_window(const GridRows& g, const float* in, const int* aggregate,
                                            const float* coarse, LDS float* xw) {
  constexpr int kAhead = 4;
  for (int j0 = threadIdx.x; j0 < g.window_rows; j0 += kAhead * kGridThreads) {
    float v[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const int j = min(j0 + u * kGridThreads, g.window_rows - 1);
      v[u] = exchange_load(in + g.window + j);
      if (coarse != nullptr) {
        const int a = ((const GLOBAL int*)aggregate)[g.window + j];
        if (a >= 0) v[u] = v[u] + exchange_load(coarse + a);
      }
    }
#pragma unroll
    for (int u = 0; u < kAhead; ++u) xw[min(j0 + u * kGridThreads, g.window_rows - 1)] = v[u];
  }
}

// The members' cycle. One loop makes every sweep of every level, so that each
// piece of code is there once: a member runs it over and over from one
// instruction cache. Levels [grid, count) are the first member's alone, with
// their iterates in LDS (two per level); the others go on to wait for their
// result.
__device__ __forceinline__ void member_cycle(const CycleArgs& A, const GridCtl& ctl, int rank) {
  constexpr int kBottom = KH_GRID_BOTTOM_ROWS;
  const PartTable parts = (PartTable)A.table + rank * A.count;
  const LevelTable levels = (LevelTable)A.levels;
  LDS float* const window = lds_at<float>(0);
  const int iterates = A.grid < A.count ? parts[A.grid].iterates : 0;
  unsigned passed = 0;
  for (int k = 0; k < A.count; ++k)
    if (k < A.grid || rank == 0) grid_stage(levels + k, parts + k);
  {
    const GridRows g = grid_rows(parts);
    for (int r = threadIdx.x; r < g.rows; r += kGridThreads) g.rhs[r] = ((const GLOBAL float*)A.rhs)[g.first + r];
  }
  __syncthreads();
  int k = 0, t = 0;  // the level, and its sweeps so far
  bool up = false;   // past the coarsest level
  while (true) {     // one visit of level k, down or up
    const bool local = k >= A.grid, coarsest = k + 1 == A.count;
    const int pre = coarsest ? A.coarse_sweeps : A.pre, total = coarsest ? pre : pre + A.post;
    const CONSTANT kh_grid_level& L = levels[k];
    const GridRows g = grid_rows(parts + k);
    // Sweep t's iterate, so that the last is x.
    float* const x = k == 0 ? A.out : L.x;
    float* const w = L.w;
    const auto target = [&](int s) { return ((total - s) & 1) == 0 ? x : w; };
    LDS float* const own = lds_at<float>(iterates + 2 * (k - A.grid) * kBottom);  // a local level's
    const auto local_target = [&](int s) { return own + ((total - s) & 1) * kBottom; };
    for (const int end = up || coarsest ? total : pre + 1; t < end; ++t) {
      const bool prolong = up && t == pre, residual = !up && t == pre;
      if (!up && t == 0) {
        // amg_coarse_solve starts from stored zeros, the others from none.
        const bool stored = coarsest && local && g.rows <= kCoarseMax;
        for (int r = threadIdx.x; r < g.rows; r += kGridThreads) {
          if (stored) local_target(0)[r] = 0.0f;
          else if (local) local_target(1)[r] = zero_row(g, r);
          else exchange_store(target(1) + g.first + r, zero_row(g, r));
        }
        if (!local) grid_sync(ctl, A.parts, passed);
        else __syncthreads();
        if (!stored) continue;
      }
      LDS float* xw = window;
      if (local) {
        xw = local_target(t);
        if (prolong) {
          const LDS float* c = own + 2 * kBottom;  // the next level's x
          for (int r = threadIdx.x; r < g.rows; r += kGridThreads) {
            const int a = ((const GLOBAL int*)L.aggregate)[r];
            if (a >= 0) xw[r] = xw[r] + c[a];
          }
          __syncthreads();
        }
      } else {
        load_window(g, target(t), L.aggregate, prolong ? levels[k + 1].x : nullptr, xw);
        __syncthreads();
      }
      float* const out = target(t + 1);
      LDS float* const local_out = local_target(t + 1);
      grid_residuals(g, xw, [&](int r, float rr, bool mine) {
        const float v = residual ? rr : xw[g.first - g.window + r] + g.weight[r] * rr;
        if (!mine) return;
        if (local) local_out[r] = v;
        else exchange_store(out + g.first + r, v);
      });
      if (local) __syncthreads();
      else if (k > 0 || t + 1 < total || residual) grid_sync(ctl, A.parts, passed);
    }
    if (up || coarsest) {
      if (k == 0) return;
      if (k == A.grid) {  // the first member's result goes to all
        for (int r = threadIdx.x; r < g.rows; r += kGridThreads) exchange_store(x + r, own[r]);
        grid_sync(ctl, A.parts, passed);
      }
      --k;
      t = A.pre;
      up = true;
      continue;
    }
    // The next level's right-hand side, by the owners of its rows: its
    // members' residuals in member order (k_amg_restrict).
    ++k;
    t = 0;
    if (k < A.grid || rank == 0) {
      const GridRows c = grid_rows(parts + k);
      const float* from = target(pre + 1);
      const LDS float* here = local_target(pre + 1);
      const GLOBAL int* offsets = (const GLOBAL int*)L.member_offsets;
      const GLOBAL int* members = (const GLOBAL int*)L.members;
      for (int r = threadIdx.x; r < c.rows; r += kGridThreads) {
        Kahan sum;
        for (int m = offsets[c.first + r], last = offsets[c.first + r + 1]; m < last; ++m)
          sum.add(local ? here[members[m]] : exchange_load(from + members[m]));
        c.rhs[r] = sum.s;
      }
      __syncthreads();
    } else {
      grid_sync(ctl, A.parts, passed);  // the first member's result
      --k;
      t = A.pre;
      up = true;
    }
  }
}

__global__ void __launch_bounds__(kGridThreads) k_grid_cycle(const CycleArgs A) {
  if (A.status[0] != 0) return;
  GridCtl ctl(A.ctl, long(A.limit_us) * 100);
  if (threadIdx.x == 0) {
    const unsigned polls = ctl_load(A.ctl + KH_GRID_CTL_POLLS);
    grid_wait() = {grid_enter(ctl, gridDim.x, A.parts, xcc_id() == ctl_load(ctl.home)), polls, 0};
  }
  __syncthreads();
  const GridPlace place = grid_wait().place;
  const GridRole role = GridRole(__builtin_amdgcn_readfirstlane(int(place.role)));
  if (role == GridRole::Member) member_cycle(A, ctl, __builtin_amdgcn_readfirstlane(place.rank));
  else if (role == GridRole::Solo) solo_cycle(A);
  __syncthreads();
  if (threadIdx.x == 0) {
    if (role == GridRole::Solo) ctl.count(KH_GRID_REPORT_ALONE);
    if (role == GridRole::Member && place.rank == 0) ctl.count(KH_GRID_REPORT_TOGETHER);
    if (grid_wait().given_up) ctl.count(KH_GRID_REPORT_GIVEN_UP);
    grid_leave(ctl, gridDim.x);
  }
}

// Clears a control block and records the XCD of this workgroup as its home.
__global__ void k_grid_init(unsigned* ctl) {
  for (int i = threadIdx.x; i < KH_GRID_CTL_WORDS; i += blockDim.x) ctl[i] = 0;
  __syncthreads();
  if (threadIdx.x == 0) {
    ctl[KH_GRID_CTL_HOME] = xcc_id();
    ctl[KH_GRID_CTL_POLLS] = kBarrierPolls;
  }
}
// Counts the workgroups of a launch that are on the home XCD.
__global__ void k_grid_spread(unsigned* ctl) {
  if (threadIdx.x == 0 && xcc_id() == ctl[KH_GRID_CTL_HOME]) GridCtl::add(ctl + KH_GRID_CTL_SPREAD, 1);
}

void allow_lds(kh_device* d) {
  if (d->grid_ready) return;
  check(hipFuncSetAttribute(reinterpret_cast<const void*>(k_grid_cycle), hipFuncAttributeMaxDynamicSharedMemorySize,
                            KH_GRID_POOL_WORDS * 4),
        "grid_cycle LDS size");
  d->grid_ready = true;
}
void l_grid_init(kh_device* d, int, const kh_arg* a) {
  allow_lds(d);  // not first under a capture
  k_grid_init<<<dim3(1), dim3(64), 0, d->stream>>>(static_cast<unsigned*>(buf(a, 0)));
  k_grid_spread<<<dim3(8 * KH_GRID_MAX_PARTS), dim3(64), 0, d->stream>>>(static_cast<unsigned*>(buf(a, 0)));
}
// levels, table, ctl, count, grid, pre, post, coarse_sweeps, parts, lds_words,
// limit_us, rhs, out, status
void l_grid_cycle(kh_device* d, int n, const kh_arg* a) {
  CycleArgs c;
  c.levels = static_cast<const kh_grid_level*>(buf(a, 0));
  c.table = static_cast<const kh_grid_part*>(buf(a, 1));
  c.ctl = static_cast<unsigned*>(buf(a, 2));
  c.count = i32(a, 3);
  c.grid = i32(a, 4);
  c.pre = i32(a, 5);
  c.post = i32(a, 6);
  c.coarse_sweeps = i32(a, 7);
  c.parts = i32(a, 8);
  c.lds_words = i32(a, 9);
  c.limit_us = i32(a, 10);
  c.rhs = static_cast<const float*>(buf(a, 11));
  c.out = static_cast<float*>(buf(a, 12));
  c.status = static_cast<const int*>(buf(a, 13));
  if (c.count < 1 || c.count > kMaxLevels || c.grid < 1 || c.grid > c.count)
    throw std::runtime_error("grid_cycle: bad level counts");
  if (c.pre < 1 || c.post < 1 || c.coarse_sweeps < 1)
    throw std::runtime_error("grid_cycle: sweep counts must be positive");
  if (c.parts < 1 || c.parts > KH_GRID_MAX_PARTS || c.lds_words < 1 || c.lds_words > KH_GRID_POOL_WORDS ||
      c.limit_us < 0)
    throw std::runtime_error("grid_cycle: bad launch shape");
  if (n < 1) return;
  allow_lds(d);
  k_grid_cycle<<<dim3(unsigned(8 * c.parts)), dim3(kGridThreads), std::size_t(c.lds_words) * 4, d->stream>>>(c);
}

}  // namespace

const std::vector<KernelEntry>& grid_kernels() {
  static const std::vector<KernelEntry> table = {
      {KH_GRID_INIT, "grid_init", "b", l_grid_init},
      {KH_GRID_CYCLE, "grid_cycle", "bbbiiiiiiiibbb", l_grid_cycle},
  };
  return table;
}

}  // namespace kh
