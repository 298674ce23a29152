// block_sched.h -- which block a persistent workgroup visits next (device code).
//
// Every block of a launch has a state word.  A visit that lowers a time in a dependent's halo sets
// the dependent's dirty bit; a workgroup that finds a dirty block claims it (dirty -> visiting) and
// visits it.  Blocks have an owner, workgroup b mod G, whose words lie together: an idle workgroup
// polls its own few words, and, when they stay clean, looks through other owners' words for blocks
// that wait (their owner is busy, or is not resident).  Nothing is queued, so a hand-off costs one
// atomic without a result on a word of its own.  A single ring with one tail word costs every push
// an atomic on that word, and one word takes about 85 device-scope atomics per microsecond over
// the whole chip (12 ns each; words of their own: 3,000 per microsecond): the 64^3 solve ran at
// that rate, whatever its visits cost.
//
// The end of the solve: `ctl` counts the busy workgroups (low half) and the times one became busy
// (high half).  A workgroup raises it with its first claim and lowers it, after every mark of its
// visits has landed, when it finds no more work.  The one that lowers it to zero reads all words;
// if every one is clean and ctl has not changed meanwhile, no visit ran while it read, so there is
// no work left, and it sets `done`.  If a word is dirty, the workgroup that claims it repeats this.
#pragma once

#include <hip/hip_runtime.h>

#include "fim_kernels.h"
#include "lane_ops.h"

namespace eik {

// A block's word: the key in the low half (the smallest time its suppliers have lowered since its
// last visit began, as float bits, or kClean), and in the high half whether it is under visit.
constexpr uint32_t kClean = 0xffffffffu;
constexpr size_t kSchedCtlBytes = 512;  // ctl, and done in a line of its own

struct Sched {
  unsigned long long* word;  // per slot
  unsigned long long* ctl;   // (times busy) << 32 | busy workgroups
  uint32_t* done;            // 1: the solve has ended; then, in one word of 64 bits with it, the workgroups
                             // that gave up, and in the next word the stretches taken (write_times)
  uint32_t owners;           // G: workgroups of the launch
  uint32_t per_owner;        // words per owner
  uint32_t stride;           // slots from one owner's words to the next's
  uint32_t windows;          // of 64 slots
  uint32_t step;             // windows from one look to the next: a walk over all of them
  int32_t nblocks;
  unsigned long long wait_limit;  // wall-clock ticks a workgroup may find no work
};

// The layout of the words of a launch of `owners` workgroups over nblocks blocks; where every
// owner has one, each lies in a cache line of its own.  At most sched_max_words slots.
inline void sched_shape(Sched& s, int64_t nblocks, int64_t owners) {
  s.owners = (uint32_t)owners;
  s.per_owner = (uint32_t)((nblocks + owners - 1) / owners);
  s.stride = s.per_owner == 1 ? 16 : s.per_owner;
  s.windows = (s.owners * s.stride + 63) / 64;
  s.step = s.windows % 37 ? 37 % s.windows : 1;
  s.nblocks = (int32_t)nblocks;
}
inline size_t sched_max_words(size_t nblocks, size_t max_owners) {
  return nblocks + 16 * max_owners;
}

__device__ __forceinline__ uint32_t sched_slot(const Sched& s, int32_t b) {
  const uint32_t i = (uint32_t)b / s.owners;
  return ((uint32_t)b - i * s.owners) * s.stride + i;
}

__device__ __forceinline__ int32_t sched_block(const Sched& s, uint32_t slot) {
  const uint32_t w = slot / s.stride;
  return (int32_t)((slot - w * s.stride) * s.owners + w);
}

__device__ __forceinline__ unsigned long long load_word(const unsigned long long* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint32_t* key_of(const Sched& s, uint32_t slot) {
  return reinterpret_cast<uint32_t*>(&s.word[slot]);
}
__device__ __forceinline__ uint32_t* lock_of(const Sched& s, uint32_t slot) {
  return reinterpret_cast<uint32_t*>(&s.word[slot]) + 1;
}

// Marks a block dirty with a key; no result is waited for.
__device__ __forceinline__ void sched_mark(const Sched& s, uint32_t slot, uint32_t key) {
  (void)__hip_atomic_fetch_min(key_of(s, slot), key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// What one wave of a workgroup keeps between its searches.
struct Finder {
  bool busy = false;  // counted in ctl
  uint32_t me;        // the workgroup's owner index; s.owners or more: it owns no blocks
  uint32_t probe;     // next slot to look at among all
  int others = 0;     // dirty blocks seen beside the one claimed
  uint32_t idle = 0;  // looks so far that may have gone without a window of all words
  uint64_t waits = 0; // those of the last look that were dirty (one block per owner)
};

constexpr int32_t kNoWork = -1, kNothing = -2, kGaveUp = -3;

// Smallest value over the lanes of a wave (uniform).
__device__ __forceinline__ uint32_t wave_umin(uint32_t v) {
  auto m = [](int a, int b) { return (int)((uint32_t)a < (uint32_t)b ? (uint32_t)a : (uint32_t)b); };
  int x = (int)v;
  x = m(x, __builtin_amdgcn_update_dpp(-1, x, 0x111, 0xf, 0xf, false));  // row_shr:1
  x = m(x, __builtin_amdgcn_update_dpp(-1, x, 0x112, 0xf, 0xf, false));  // row_shr:2
  x = m(x, __builtin_amdgcn_update_dpp(-1, x, 0x114, 0xf, 0xf, false));  // row_shr:4
  x = m(x, __builtin_amdgcn_update_dpp(-1, x, 0x118, 0xf, 0xf, false));  // row_shr:8
  x = m(x, __builtin_amdgcn_update_dpp(-1, x, 0x142, 0xa, 0xf, false));  // row_bcast:15
  x = m(x, __builtin_amdgcn_update_dpp(-1, x, 0x143, 0xc, 0xf, false));  // row_bcast:31
  return (uint32_t)__builtin_amdgcn_readlane(x, 63);
}

// Whether every word is clean and unlocked (one wave).
__device__ __forceinline__ bool sched_all_clean(const Sched& s) {
  const uint32_t n = s.owners * s.stride;
  for (uint32_t i0 = 0; i0 < n; i0 += 16 * 64) {
    unsigned long long v[16];
    bool bad = false;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const uint32_t i = i0 + 64 * j + __lane_id();
      v[j] = i < n ? load_word(&s.word[i]) : (unsigned long long)kClean;
    }
#pragma unroll
    for (int j = 0; j < 16; ++j) bad |= v[j] != (unsigned long long)kClean;
    if (__ballot(bad)) return false;
  }
  return true;
}

// Claims a slot seen unlocked with this key, for a visit: nothing is taken if the word has changed.  (An
// exchange would take a mark that came in under another workgroup's visit and put it back: for that
// moment, before the count of the one that took it has landed, every word could look clean.)  The
// workgroup is counted busy in the same round trip.
__device__ __forceinline__ bool sched_claim(const Sched& s, Finder& f, uint32_t slot, uint32_t key) {
  uint32_t got = 0;
  if (__lane_id() == 0) {
    if (!f.busy)
      (void)__hip_atomic_fetch_add(s.ctl, (1ull << 32) + 1ull, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
    unsigned long long seen = key;
    got = __hip_atomic_compare_exchange_strong(&s.word[slot], &seen, (1ull << 32) | kClean,
                                               __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT);
  }
  f.busy = true;
  // the count has landed before the visit marks anything
  wait_memory();
  return __builtin_amdgcn_readfirstlane(got) != 0u;
}

// One look: a block for this workgroup, claimed; kNoWork at the end of the solve; kNothing if there is
// none now.  Called by one whole wave.
// THIN: an idle workgroup looks at others' words at every 32nd look only, and sleeps between looks.  For the
// general kernels of multi-solve launches, of whose small workgroups up to 16 fit a CU: with a few blocks
// per owner, hundreds of idle ones read all words all the time, and every visit waited for that traffic
// (24 level-6 icospheres at 500 vertices per block, 1,944 blocks, records from memory: 5.36 ms looking at a
// window every time, 2.89 every 8th, 2.38 every 32nd with the sleep; 4 at 64, 2,560 blocks: 3.85 / 2.00 / 1.25).
// The register-resident kernels, with fewer and larger workgroups, look every time (12 level-6 icospheres at
// 64 vertices per block 0.81 ms, every 32nd 0.89).
template <bool THIN = false>
__device__ __forceinline__ int32_t sched_look(const Sched& s, Finder& f) {
  const uint32_t lane = __lane_id();
  const uint32_t own = f.me * s.stride;
  const uint32_t total = s.owners * s.stride;
  const uint32_t dn = __hip_atomic_load(s.done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  uint32_t key = kClean, at = 0;
  for (uint32_t base = lane; base < s.per_owner && f.me < s.owners; base += 64) {
    const unsigned long long v = load_word(&s.word[own + base]);
    if ((v >> 32) == 0ull && (uint32_t)v < key) key = (uint32_t)v, at = own + base;
  }
  // With several blocks per owner, a window of all words too: the smallest key of the two looks
  // is near the smallest of the launch, and an idle workgroup finds what a busy owner leaves.
  // With one block per owner its owner visits it, resident; now and then a window is looked at
  // for blocks that stay dirty because their owner is not running (yet).
  if (s.per_owner > 1 ? !THIN || f.busy || (++f.idle & 31u) == 0u : (++f.idle & 63u) == 0u) {
    const uint32_t i = f.probe + lane;
    const unsigned long long v = i < total ? load_word(&s.word[i]) : (unsigned long long)kClean;
    bool take = (v >> 32) == 0ull;
    bool next = true;
    if (s.per_owner == 1) {
      const uint64_t waits = __ballot(v < (unsigned long long)kClean);
      take = take && ((f.waits >> lane) & 1ull);
      next = (f.waits & waits) == 0ull && f.waits != 0ull;
      f.waits = f.waits ? 0ull : waits;
      next = next || f.waits == 0ull;
    }
    if (take && (uint32_t)v < key) key = (uint32_t)v, at = i;
    if (next) {
      f.probe += 64 * s.step;
      while (f.probe >= 64 * s.windows) f.probe -= 64 * s.windows;
    }
  }
  const uint32_t best = wave_umin(key);
  // (done is not set while a workgroup is busy; one that is never leaves without lowering ctl)
  if (best == kClean) return !f.busy && __builtin_amdgcn_readfirstlane(dn) ? kNoWork : kNothing;
  const int l = __ffsll((unsigned long long)__ballot(key == best)) - 1;
  f.others = __popcll(__ballot(key != kClean)) - 1;
  const uint32_t slot = (uint32_t)__builtin_amdgcn_readlane((int)at, l);
  return sched_claim(s, f, slot, best) ? sched_block(s, slot) : kNothing;
}

// The next block for this workgroup, claimed; kNoWork at the end of the solve; kGaveUp when the
// wait outlasted s.wait_limit.  Called by one whole wave, when every mark and release of the
// workgroup's visits has landed.
template <bool THIN = false>
__device__ __forceinline__ int32_t sched_find(const Sched& s, Finder& f) {
  unsigned long long since = 0;
  for (;;) {
    const int32_t b = sched_look<THIN>(s, f);
    if (b != kNothing) return b;
    if (f.busy) {
      unsigned long long old = 0;
      if (__lane_id() == 0)
        old = __hip_atomic_fetch_add(s.ctl, ~0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      f.busy = false;
      const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)old);
      if (lo == 1u && sched_all_clean(s) && __lane_id() == 0 &&
          __hip_atomic_load(s.ctl, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == old - 1ull)
        __hip_atomic_store(s.done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      since = wall_clock64();
      continue;
    }
    if (since == 0) since = wall_clock64();
    else if (wall_clock64() - since > s.wait_limit) return kGaveUp;
    __builtin_amdgcn_s_sleep(THIN ? 8 : 1);
  }
}

// One workgroup starts busy, so that a solve without work (no valid source) ends too.  Called by
// one whole wave before its first search.  me: the workgroup's owner index.
__device__ __forceinline__ void sched_enter(const Sched& s, Finder& f, uint32_t me) {
  f.me = me;
  f.probe = 64 * (f.me % 61 % s.windows);
  if (f.me != 0) return;
  if (__lane_id() == 0)
    (void)__hip_atomic_fetch_add(s.ctl, (1ull << 32) + 1ull, __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT);
  f.busy = true;
}

// The smallest key of this owner's blocks that no workgroup visits (one whole wave).
__device__ __forceinline__ uint32_t sched_waiting(const Sched& s, uint32_t me) {
  uint32_t key = kClean;
  for (uint32_t i = __lane_id(); i < s.per_owner && me < s.owners; i += 64) {
    const unsigned long long v = load_word(&s.word[me * s.stride + i]);
    if ((v >> 32) == 0ull && (uint32_t)v < key) key = (uint32_t)v;
  }
  return wave_umin(key);
}

// Before a further visit of a claimed block: marks up to here are answered by it, its loads follow
// once this store has completed (one thread).
__device__ __forceinline__ void sched_again(const Sched& s, uint32_t slot) {
  __hip_atomic_store(key_of(s, slot), kClean, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Gives a claimed block back after its marks have landed; key: kClean, or what it waits with.  Returns
// when the release has landed, so that the end of the solve can be found.
__device__ __forceinline__ void sched_leave(const Sched& s, uint32_t slot, uint32_t key) {
  if (key != kClean) {
    sched_mark(s, slot, key);
    wait_memory();
  }
  __hip_atomic_store(lock_of(s, slot), 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  wait_memory();
}

}  // namespace eik
