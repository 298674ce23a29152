// A host model of a few workgroups, for builds of device headers with a plain C++ compiler: every
// thread of the launch is a fiber, and a scheduler interleaves the waves at random.
//
// * A thread runs until it reaches a barrier, an operation of its wave (ballot, DPP, readlane), or
//   an access of device memory by an atomic, and the scheduler then takes another wave.  Which wave
//   comes next is drawn with weights that are drawn again now and then, so that some waves fall far
//   behind others between two barriers.
// * An operation of a wave waits for all of its 64 lanes: one that only some lanes reach, or a barrier
//   that only some waves reach, ends the run with an error.
// * Atomics of device memory without a result, and stores, land later, in any order among different
//   addresses, at the latest when their wave waits for them (wait_memory); an access of the same
//   address by the same wave finds them landed.
// * wall_clock64() counts scheduling steps.
//
// Only what the scheduler, the register-resident visits and their loop use is here.
#pragma once

#include <hip/hip_runtime_api.h>
#include <setjmp.h>
#include <ucontext.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <memory>
#include <random>
#include <type_traits>
#include <utility>
#include <vector>

#undef __device__
#undef __host__
#undef __global__
#undef __forceinline__
#undef __noinline__
#define __device__
#define __host__
#define __global__
#define __forceinline__ inline
#define __noinline__ __attribute__((noinline))
#define __launch_bounds__(...)

// ------------------------------------------------------------------------------------------
// scalar helpers
// ------------------------------------------------------------------------------------------
using std::max;
using std::min;

template <class To, class From>
inline To simt_cast(From v) {
  static_assert(sizeof(To) == sizeof(From), "");
  To t;
  std::memcpy(&t, &v, sizeof t);
  return t;
}
inline unsigned __float_as_uint(float f) { return simt_cast<unsigned>(f); }
inline float __uint_as_float(unsigned u) { return simt_cast<float>(u); }
inline int __popc(unsigned v) { return __builtin_popcount(v); }
inline int __popcll(unsigned long long v) { return __builtin_popcountll(v); }
inline int __ffs(unsigned v) { return __builtin_ffs((int)v); }
inline int __ffsll(unsigned long long v) { return __builtin_ffsll((long long)v); }
#define __builtin_amdgcn_sqrtf(x) std::sqrt((float)(x))
#define __builtin_amdgcn_rcpf(x) (1.f / (float)(x))
inline int simt_frexp_exp(float x) {
  int e = 0;
  if (x != 0.f && std::isfinite(x)) (void)std::frexp(x, &e);
  return e;
}
#define __builtin_amdgcn_frexp_expf(x) simt_frexp_exp(x)

// ------------------------------------------------------------------------------------------
// fibers, waves, workgroups
// ------------------------------------------------------------------------------------------
namespace simt {

constexpr int kLanes = 64;
struct Dim { unsigned x = 0, y = 0, z = 0; };
enum State { kReady, kWaveOp, kWait, kBarrier, kEnded };

struct Wave;
struct Thread {
  ucontext_t ctx;  // its first entry; later switches are jumps
  jmp_buf at;
  bool entered = false;
  std::unique_ptr<char[]> stack;
  State state = kReady;
  Dim tid, bid;
  Wave* wave = nullptr;
  int lane = 0;
  uint64_t value = 0;  // what it gave to the wave operation it waits for
  int kind = 0;
};
struct Op {
  void* address;
  std::function<void()> land;
};
struct Wave {
  std::vector<Thread*> lanes;
  int group = 0;
  uint64_t seen[2][kLanes] = {};  // what the lanes gave, of alternate operations
  uint32_t ops = 0;
  std::vector<Op> pending;
  double weight = 1.0;
};
struct Group {
  std::vector<Wave*> waves;
};

inline Thread* g_me = nullptr;
inline jmp_buf g_main;
inline unsigned long long g_clock = 0;
inline std::mt19937_64 g_rng;
inline Dim g_grid, g_block;
inline std::function<void()> g_body;
inline bool g_yield_atomics = true;
inline const char* g_error = nullptr;

inline Thread& me() { return *g_me; }
inline void to_scheduler() {
  if (_setjmp(g_me->at) == 0) _longjmp(g_main, 1);
}
__attribute__((noinline)) inline void resume(Thread* t) {
  g_me = t;
  if (_setjmp(g_main) != 0) return;
  if (t->entered) _longjmp(t->at, 1);
  t->entered = true;
  setcontext(&t->ctx);
}
inline void yield() { to_scheduler(); }
inline void entry() {
  g_body();
  g_me->state = kEnded;
  to_scheduler();
}

// All lanes of the wave meet; the values that they gave.
inline const uint64_t* meet(int kind, uint64_t value) {
  Thread& t = me();
  t.value = value;
  t.kind = kind;
  t.state = kWaveOp;
  to_scheduler();
  return t.wave->seen[(t.wave->ops - 1) & 1];
}
// Until the wave's memory operations have landed: its other lanes come first to where they wait too.
inline void wait() {
  me().state = kWait;
  to_scheduler();
}
inline void barrier() {
  me().state = kBarrier;
  to_scheduler();
}

inline void land(Wave& w, size_t i) {
  Op op = std::move(w.pending[i]);
  w.pending.erase(w.pending.begin() + (long)i);
  op.land();
}
inline void land_all(Wave& w) {
  while (!w.pending.empty()) land(w, g_rng() % w.pending.size());
}
inline void land_address(Wave& w, const void* p) {
  for (size_t i = 0; i < w.pending.size();)
    if (w.pending[i].address == p) land(w, i);
    else ++i;
}
// Words of 8 bytes and their halves count as one address.
inline void* word_of(const volatile void* p) {
  return reinterpret_cast<void*>(reinterpret_cast<uintptr_t>(p) & ~(uintptr_t)7);
}

// An atomic whose result may be taken (it happens now) or not (it lands later).
template <class T, class F>
struct Result {
  T* p;
  F f;
  bool taken = false;
  Result(T* p_, F f_) : p(p_), f(f_) {}
  Result(const Result&) = delete;
  operator T() {
    taken = true;
    land_address(*me().wave, word_of(p));
    const T old = *p;
    *p = f(old);
    return old;
  }
  ~Result() {
    if (taken) return;
    T* q = p;
    F g = f;
    me().wave->pending.push_back({word_of(q), [q, g] { *q = g(*q); }});
  }
};
template <class T>
inline T load(const T* p) {
  if (g_yield_atomics) yield();
  land_address(*me().wave, word_of(p));
  return *p;
}
template <class T, class V>
inline void store(T* p, V v) {
  if (g_yield_atomics) yield();
  const T t = (T)v;
  // in order with the wave's earlier accesses of the address
  land_address(*me().wave, word_of(p));
  me().wave->pending.push_back({word_of(p), [p, t] { *p = t; }});
}
template <class T, class F>
inline Result<T, F> atomic(T* p, F f) {
  if (g_yield_atomics) yield();
  land_address(*me().wave, word_of(p));
  return Result<T, F>(p, f);
}

// Runs `groups` workgroups of `threads` (a multiple of 64), at most `resident` at a time: a further one
// starts when one has ended.  Returns null, or what went wrong.
inline const char* run(unsigned groups, unsigned threads, uint64_t seed, unsigned resident,
                       const std::function<void()>& body, unsigned long long max_steps = 1ull << 33) {
  g_rng.seed(seed);
  g_clock = 1;
  g_error = nullptr;
  g_grid = {groups, 1, 1};
  g_block = {threads, 1, 1};
  g_body = body;
  constexpr size_t kStack = 64 << 10;
  std::vector<std::unique_ptr<Thread>> ts;
  std::vector<std::unique_ptr<Wave>> ws;
  std::vector<Group> gs(groups);
  for (unsigned g = 0; g < groups; ++g)
    for (unsigned i = 0; i < threads; ++i) {
      if (i % kLanes == 0) {
        ws.emplace_back(new Wave());
        ws.back()->group = (int)g;
        gs[g].waves.push_back(ws.back().get());
      }
      ts.emplace_back(new Thread());
      Thread& t = *ts.back();
      t.tid.x = i;
      t.bid.x = g;
      t.wave = ws.back().get();
      t.lane = (int)(i % kLanes);
      t.stack.reset(new char[kStack]);
      getcontext(&t.ctx);
      t.ctx.uc_stack.ss_sp = t.stack.get();
      t.ctx.uc_stack.ss_size = kStack;
      t.ctx.uc_link = nullptr;
      makecontext(&t.ctx, entry, 0);
      ws.back()->lanes.push_back(&t);
    }
  auto uniform = [] { return (double)(g_rng() >> 11) * 0x1p-53; };
  size_t left = ws.size();
  std::vector<Wave*> order;  // the waves that run
  unsigned started = 0;
  auto start = [&] {
    for (Wave* w : gs[started].waves) order.push_back(w);
    ++started;
  };
  while (started < std::min(groups, resident)) start();
  while (left > 0) {
    if (++g_clock > max_steps) return "too many steps";
    if (g_clock % 256 == 2)
      for (auto& w : ws) w->weight = std::exp(8.0 * uniform() * uniform());
    // the next wave: the better of a few drawn by weight
    Wave* w = nullptr;
    double best = -1.0;
    bool stuck = true;
    const size_t at = g_rng() % order.size();
    for (size_t k = 0; k < order.size(); ++k) {
      Wave* c = order[(at + k) % order.size()];
      bool ready = false;
      for (Thread* t : c->lanes) ready = ready || t->state == kReady;
      if (!ready) continue;
      stuck = false;
      const double x = uniform() * c->weight;
      if (x > best) best = x, w = c;
    }
    if (stuck) return g_error ? g_error : "every thread waits";
    if (!w->pending.empty() && uniform() < 0.2) land(*w, g_rng() % w->pending.size());
    for (Thread* t : w->lanes)
      if (t->state == kReady) resume(t);
    // the wave's operation, when all of its lanes have come to one
    size_t at_op = 0, at_barrier = 0, at_wait = 0, ended = 0, ready = 0;
    for (Thread* t : w->lanes) {
      ready += t->state == kReady;
      at_wait += t->state == kWait;
      at_op += t->state == kWaveOp;
      at_barrier += t->state == kBarrier;
      ended += t->state == kEnded;
    }
    const size_t n = w->lanes.size();
    if (ready == 0 && at_wait > 0) {
      land_all(*w);
      for (Thread* t : w->lanes)
        if (t->state == kWait) t->state = kReady;
    } else if (at_op == n) {
      for (Thread* t : w->lanes) {
        if (t->kind != w->lanes[0]->kind) return "lanes of a wave at different operations";
        w->seen[w->ops & 1][t->lane] = t->value;
        t->state = kReady;
      }
      ++w->ops;
    } else if (ready == 0 && at_op > 0) {
      return "an operation of a wave that some lanes do not reach";
    }
    if (ended == n) {
      land_all(*w);
      --left;
      for (size_t i = 0; i < order.size(); ++i)
        if (order[i] == w) {
          order.erase(order.begin() + (long)i);
          break;
        }
      bool gone = true;
      for (Wave* v : gs[(size_t)w->group].waves)
        for (Thread* t : v->lanes) gone = gone && t->state == kEnded;
      if (gone && started < groups) start();
    }
    // the workgroup's barrier
    bool all = true, any_ended = false;
    for (Wave* v : gs[(size_t)w->group].waves)
      for (Thread* t : v->lanes) {
        all = all && t->state == kBarrier;
        any_ended = any_ended || t->state == kEnded;
      }
    if (all)
      for (Wave* v : gs[(size_t)w->group].waves)
        for (Thread* t : v->lanes) t->state = kReady;
    if (any_ended && at_barrier == n) g_error = "a barrier that some waves do not reach";
  }
  return nullptr;
}

}  // namespace simt

#define threadIdx (simt::me().tid)
#define blockIdx (simt::me().bid)
#define gridDim (simt::g_grid)
#define blockDim (simt::g_block)

inline unsigned __lane_id() { return (unsigned)simt::me().lane; }
inline unsigned long long wall_clock64() { return simt::g_clock; }
inline void __syncthreads() { simt::barrier(); }

// ------------------------------------------------------------------------------------------
// operations of a wave
// ------------------------------------------------------------------------------------------
inline unsigned long long __ballot(bool p) {
  const uint64_t* v = simt::meet(1, p ? 1 : 0);
  unsigned long long m = 0;
  for (int i = 0; i < simt::kLanes; ++i) m |= (unsigned long long)(v[i] & 1) << i;
  return m;
}
template <class T>
inline T simt_readlane(T x, int l) {
  return (T)simt::meet(2, (uint64_t)x)[l];
}
#define __builtin_amdgcn_readlane(x, l) simt_readlane((x), (l))
#define __builtin_amdgcn_readfirstlane(x) simt_readlane((x), 0)
#define __builtin_amdgcn_wave_barrier() ((void)simt::meet(3, 0))
inline unsigned long long __shfl_down(unsigned long long x, int off, int) {
  const uint64_t* v = simt::meet(4, x);
  const int l = simt::me().lane + off;
  return l < simt::kLanes ? v[l] : x;
}
// row_shr:n (0x110 + n), row_bcast:15 (0x142), row_bcast:31 (0x143); lanes without a source keep old
inline int simt_dpp(int old, int x, int ctrl, int row_mask) {
  const uint64_t* v = simt::meet(ctrl, (uint32_t)x);
  const int l = simt::me().lane, row = l >> 4;
  if (!((row_mask >> row) & 1)) return old;
  int from = -1;
  if (ctrl > 0x110 && ctrl < 0x120) from = (l & 15) >= ctrl - 0x110 ? l - (ctrl - 0x110) : -1;
  else if (ctrl == 0x142) from = row ? 16 * row - 1 : -1;
  else if (ctrl == 0x143) from = row >= 2 ? 31 : -1;
  else std::abort();
  return from < 0 ? old : (int)(uint32_t)v[from];
}
#define __builtin_amdgcn_update_dpp(old, x, ctrl, row_mask, bank_mask, bound) \
  simt_dpp((old), (x), (ctrl), (row_mask))
inline unsigned simt_mbcnt(uint32_t mask, unsigned base, int lo) {
  const int l = simt::me().lane, n = std::min(std::max(l - lo, 0), 32);
  const uint32_t below = n == 32 ? ~0u : (1u << n) - 1u;
  return base + (unsigned)__builtin_popcount(mask & below);
}
#define __builtin_amdgcn_mbcnt_lo(m, b) simt_mbcnt((m), (b), 0)
#define __builtin_amdgcn_mbcnt_hi(m, b) simt_mbcnt((m), (b), 32)
#define __builtin_amdgcn_s_sleep(n) simt::yield()
#define __builtin_amdgcn_s_waitcnt(n) simt::wait()

// ------------------------------------------------------------------------------------------
// atomics: of device memory (with a scope), and of the LDS
// ------------------------------------------------------------------------------------------
#define __HIP_MEMORY_SCOPE_AGENT 0
#define __HIP_MEMORY_SCOPE_SYSTEM 0
template <class T, class V>
inline auto simt_fetch_min(T* p, V v) {
  const T t = (T)v;
  return simt::atomic(p, [t](T old) { return t < old ? t : old; });
}
template <class T, class V>
inline auto simt_fetch_add(T* p, V v) {
  const T t = (T)v;
  return simt::atomic(p, [t](T old) { return (T)(old + t); });
}
template <class T, class V>
inline bool simt_cas(T* p, T* expected, V v) {
  simt::yield();
  simt::land_address(*simt::me().wave, simt::word_of(p));
  if (*p != *expected) {
    *expected = *p;
    return false;
  }
  *p = (T)v;
  return true;
}
#define __hip_atomic_load(p, order, scope) simt::load(p)
#define __hip_atomic_store(p, v, order, scope) simt::store((p), (v))
#define __hip_atomic_fetch_min(p, v, order, scope) simt_fetch_min((p), (v))
#define __hip_atomic_fetch_add(p, v, order, scope) simt_fetch_add((p), (v))
#define __hip_atomic_compare_exchange_strong(p, e, v, o1, o2, scope) simt_cas((p), (e), (v))

template <class T, class V>
inline T atomicMin(T* p, V v) {
  const T old = *p;
  if ((T)v < old) *p = (T)v;
  return old;
}
template <class T, class V>
inline T atomicAdd(T* p, V v) {
  const T old = *p;
  *p = (T)(old + (T)v);
  return old;
}
template <class T, class V>
inline T atomicOr(T* p, V v) {
  const T old = *p;
  *p = (T)(old | (T)v);
  return old;
}
template <class T, class V>
inline T atomicExch(T* p, V v) {
  const T old = *p;
  *p = (T)v;
  return old;
}
