// sched_model.cpp -- the scheduler of the persistent workgroups (csrc/block_sched.h, as it is) on a host
// model of the device (simt/hip/hip_runtime.h), with visits that are a few relaxations: many schedules
// of many idle workgroups, where work comes late and from afar.
//
// A launch solves shortest paths over a random graph of blocks.  Workgroups are one wave each, find blocks,
// relax them, mark dependents, visit a block again or give it back, in the order of visit_loop.h.
// Checked: every launch ends, no word is dirty or locked then, and every value is the shortest path.
//
// usage: sched_model <launches> <seed>
#include <hip/hip_runtime.h>

#include "block_sched.h"

using namespace eik;

namespace {

struct Graph {
  int nb = 0;
  std::vector<std::vector<std::pair<int, uint32_t>>> sup;  // of a block: supplier and weight
  std::vector<std::vector<int>> dep;
};

std::mt19937_64 rng;
int rnd(int n) { return (int)(rng() % (uint64_t)n); }

Graph make_graph() {
  Graph g;
  g.nb = 1 + rnd(rnd(3) ? 40 : 300);
  g.sup.resize((size_t)g.nb);
  g.dep.resize((size_t)g.nb);
  const int chords = rnd(3);
  for (int b = 0; b < g.nb; ++b)
    for (int k = 0; k <= chords; ++k) {
      const int c = k == 0 ? (b + 1) % g.nb : rnd(g.nb);
      if (c == b || g.sup[(size_t)b].size() >= 30 || g.sup[(size_t)c].size() >= 30) continue;
      const uint32_t w = 1 + (uint32_t)rnd(100);
      g.sup[(size_t)b].push_back({c, w});
      g.sup[(size_t)c].push_back({b, w});
      g.dep[(size_t)c].push_back(b);
      g.dep[(size_t)b].push_back(c);
    }
  return g;
}

constexpr uint32_t kFar = 0x7fffffffu;

std::vector<uint32_t> shortest(const Graph& g, const std::vector<int>& seeds) {
  std::vector<uint32_t> v((size_t)g.nb, kFar);
  for (int s : seeds) v[(size_t)s] = 0;
  for (bool changed = true; changed;) {
    changed = false;
    for (int b = 0; b < g.nb; ++b)
      for (auto& e : g.sup[(size_t)b])
        if (v[(size_t)e.first] != kFar && v[(size_t)e.first] + e.second < v[(size_t)b])
          v[(size_t)b] = v[(size_t)e.first] + e.second, changed = true;
  }
  return v;
}

struct Launch {
  Graph g;
  Sched s;
  std::vector<unsigned long long> words;
  alignas(256) unsigned char ctl[kSchedCtlBytes];
  std::vector<uint32_t> value;
  std::vector<uint32_t> mine;  // a block's value as its elements know it (only its visitor's)
  uint64_t again_in;           // a visit is cut off, on average, one time in this many (0: never)
};

// One workgroup (one wave).
template <bool THIN>
int work(Launch& l) {
  const Sched& s = l.s;
  Finder f;
  sched_enter(s, f, blockIdx.x);
  std::mt19937 own(blockIdx.x * 977u + 13u);  // the same in every lane
  int32_t b = kNothing;
  for (;;) {
    if (b == kNothing) b = sched_find<THIN>(s, f);
    if (b < 0) return b;
    const uint32_t slot = sched_slot(s, b);
    const auto& sup = l.g.sup[(size_t)b];
    const auto& dep = l.g.dep[(size_t)b];
    const unsigned lane = __lane_id();
    for (;;) {
      // the suppliers' values, then the block's own
      uint32_t v = kFar;
      if (lane < sup.size()) {
        const uint32_t t = __hip_atomic_load(&l.value[(size_t)sup[lane].first], __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT);
        if (t != kFar) v = t + sup[lane].second;
      }
      const uint32_t best = wave_umin(v);
      const uint32_t old = __builtin_amdgcn_readfirstlane(
          __hip_atomic_load(&l.value[(size_t)b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
      const bool fell = best < old;
      const bool first = __ballot(l.mine[(size_t)b] != old) != 0ull;  // (a source: its value is news too)
      const uint32_t now = fell ? best : old;
      if (lane == 0) l.mine[(size_t)b] = now;
      const bool more = l.again_in && own() % l.again_in == 0;
      if (fell && lane == 0)
        (void)__hip_atomic_fetch_min(&l.value[(size_t)b], best, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (more && lane == 0) sched_again(s, slot);
      wait_memory();
      const bool again = more && own() % 2;
      if ((fell || first) && lane < dep.size()) sched_mark(s, sched_slot(s, dep[lane]), now);
      if (again) continue;
      wait_memory();
      if (lane == 0) sched_leave(s, slot, more ? now : kClean);
      __builtin_amdgcn_wave_barrier();
      break;
    }
    b = own() % 2 && s.per_owner > 1 ? sched_look<THIN>(s, f) : kNothing;
  }
}

}  // namespace

int main(int argc, char** argv) {
  if (argc != 3) return 2;
  const int launches = std::atoi(argv[1]);
  rng.seed(std::strtoull(argv[2], nullptr, 10));
  int failures = 0;
  for (int i = 0; i < launches; ++i) {
    Launch l;
    l.g = make_graph();
    const int nb = l.g.nb, groups = 1 + rnd(rnd(2) ? 6 : 24);
    sched_shape(l.s, nb, groups);
    l.words.assign((size_t)l.s.owners * l.s.stride, (unsigned long long)kClean);
    std::memset(l.ctl, 0, sizeof l.ctl);
    l.s.word = l.words.data();
    l.s.ctl = reinterpret_cast<unsigned long long*>(l.ctl);
    l.s.done = reinterpret_cast<uint32_t*>(l.ctl + kSchedCtlBytes / 2);
    l.s.wait_limit = ~0ull;
    l.value.assign((size_t)nb, kFar);
    l.mine.assign((size_t)nb, kFar);
    static const uint64_t cuts[] = {0, 2, 3, 5};
    l.again_in = cuts[rnd(4)];
    std::vector<int> seeds;
    for (int k = rnd(4); k > 0; --k) seeds.push_back(rnd(nb));  // none: the launch ends too
    for (int s : seeds) {
      l.value[(size_t)s] = 0;
      l.words[sched_slot(l.s, s)] = 0ull;
    }
    const char* err = simt::run((unsigned)groups, 64, rng(), 1 + (unsigned)rnd(groups), [&] { (void)(i % 2 ? work<true>(l) : work<false>(l)); });
    int dirty = 0, wrong = 0;
    for (unsigned long long w : l.words) dirty += w != (unsigned long long)kClean;
    const std::vector<uint32_t> ref = shortest(l.g, seeds);
    for (int b = 0; b < nb; ++b) wrong += l.value[(size_t)b] != ref[(size_t)b];
    if (err || dirty || wrong) {
      ++failures;
      std::printf("launch %d: %d blocks, %d workgroups: %s, %d words not clean, %d values wrong\n", i, nb, groups,
                  err ? err : "ended", dirty, wrong);
      if (err) break;
    }
  }
  std::printf("%d launches, failures %d\n", launches, failures);
  return failures ? 1 : 0;
}
