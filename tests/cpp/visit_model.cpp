// visit_model.cpp -- whole solves by the loop of the persistent workgroups (csrc/visit_loop.h with
// block_sched.h and resident.h, as they are) on a host model of the device (simt/hip/hip_runtime.h):
// waves interleaved at random, atomics that land late, simulated clock.
//
// Every solve must end by itself with all block words clean, and its times must be a fixed point: no
// corner solve of any element gives less than its target's time (the solver and its arithmetic are
// those of the visits).  The output must be the times in caller order, complete, whether or not
// workgroups gave up waiting before the end.
//
// usage: visit_model <triN|tetN|cap4> <mesh size> <vertices per block> <workgroups> <inner sweeps> <runs>
//                    <seed> <wait limit, steps; 0: none> [eps [workgroups that run at a time]]
// cap4: tets, 4 elements per thread, a work-item queue that holds a twentieth of a block's pairs.
// With eps > 0 a visit ends when a sweep lowers nothing by more than that, and what its last sweep
// lowered counts as evaluated; a fall of a halo vertex is evaluated, however small: only the corner
// solves from halo vertices alone are looked at then.
#include <hip/hip_runtime.h>

#include "visit_loop.h"

namespace eik {
void set_error(const std::string&) {}
int fail(int code, const std::string& msg) {
  std::fprintf(stderr, "%s\n", msg.c_str());
  return code;
}
void device_release(Mesh&) {}
int check_end(const unsigned char*, hipStream_t, unsigned long long) { return 0; }
}  // namespace eik

using namespace eik;

namespace {

struct Items {
  std::vector<int2> range;
  std::vector<uint32_t> id;
  std::vector<float4> len;
  std::vector<uint16_t> rec;
};

// As k_tri_items: the updatable corners of a block's records, in record order.
Items tri_items(const Layout& L) {
  Items t;
  for (const BlockDesc& d : L.blocks) {
    const int start = (int)t.id.size();
    for (int e = 0; e < d.nelem; ++e) {
      const TriRec& r = L.tris[(size_t)(d.estart + e)];
      static const int other[3][2] = {{1, 2}, {0, 2}, {0, 1}};
      // lengths {01, 12, 20}: of the two edges at the target, then of the one opposite
      static const int len[3][3] = {{0, 2, 1}, {0, 1, 2}, {2, 1, 0}};
      for (int k = 0; k < 3; ++k) {
        if (!(r.mask >> k & 1) || r.v[k] >= d.nown) continue;
        t.id.push_back(r.v[other[k][0]] | (uint32_t)r.v[other[k][1]] << kItemSlotBits |
                       (uint32_t)r.v[k] << (2 * kItemSlotBits));
        t.len.push_back(make_float4(r.L[len[k][0]], r.L[len[k][1]], r.L[len[k][2]], r.H[k]));
        t.rec.push_back((uint16_t)e);
      }
    }
    t.range.push_back(make_int2(start, (int)t.id.size() - start));
  }
  return t;
}

struct Solve {
  const Mesh& m;
  Items items;
  std::vector<float> T, seen, out;
  std::vector<unsigned long long> words;
  alignas(256) unsigned char ctl[kSchedCtlBytes] = {};
  LoopArgs a = {};
  explicit Solve(const Mesh& mesh) : m(mesh) {
    if (m.dim == 2) items = tri_items(m.layout);
  }
};

struct ModelBlocks {
  static constexpr bool kSingle = true;
  Solve& s;
  BlockData operator()(int32_t b) const {
    const Layout& L = s.m.layout;
    BlockData d = {};
    d.blocks = L.blocks.data();
    d.elems = s.m.dim == 3 ? (const void*)L.tets.data() : (const void*)L.tris.data();
    d.halo = L.halo.data();
    d.T = s.T.data();
    d.seen = s.seen.data();
    d.vmask = L.vmask.data();
    d.dep_start = L.dep_start.data();
    d.dep = L.dep.data();
    d.rmult = nullptr;
    d.unit = L.height_unit;
    d.items = {s.items.range.data(), s.items.id.data(), s.items.len.data(), s.items.rec.data()};
    d.b = b;
    d.base = 0;
    return d;
  }
};

// Corner solves that give less than their target's time (owned corners of every record).
int improvable(const Solve& s, bool halo_only) {
  const Mesh& m = s.m;
  const Layout& L = m.layout;
  int bad = 0;
  for (const BlockDesc& d : L.blocks)
    for (int e = 0; e < d.nelem; ++e) {
      float t[4] = {0, 0, 0, 0};
      const int K = m.dim + 1;
      const uint16_t* v = m.dim == 3 ? L.tets[(size_t)(d.estart + e)].v : L.tris[(size_t)(d.estart + e)].v;
      for (int k = 0; k < K; ++k)
        t[k] = s.T[(size_t)(v[k] < d.nown ? d.vstart + v[k] : L.halo[(size_t)(d.hstart + v[k] - d.nown)])];
      for (int k = 0; k < K; ++k) {
        if (v[k] >= d.nown) continue;
        bool owned = false;
        for (int j = 0; j < K; ++j) owned = owned || (j != k && v[j] < d.nown);
        if (halo_only && owned) continue;
        float least = EIK_INF, cand, h;
        for (int j = 0; j < K; ++j)
          if (j != k) least = std::min(least, t[j]);
        if (m.dim == 3) {
          const TetRec& r = L.tets[(size_t)(d.estart + e)];
          h = r.H[k];
          cand = tet_rotation(k, t[0], t[1], t[2], t[3], r.L[0], r.L[1], r.L[2], r.L[3], r.L[4], r.L[5],
                              EIK_LARGENUM_3D);
        } else {
          const TriRec& r = L.tris[(size_t)(d.estart + e)];
          if (!(r.mask >> k & 1)) continue;
          h = r.H[k];
          cand = tri_rotation(k, t[0], t[1], t[2], r.L[0], r.L[1], r.L[2], EIK_LARGENUM_2D);
        }
        bad += t[k] > least + h && std::max(cand, 0.f) < t[k];
      }
    }
  return bad;
}

struct Group {
  std::vector<uint4> lds;
  LoopShared sh;
  int end = 0;
};

template <int DIM, int N, int BT, bool CAP = false>
int run_solves(Mesh& m, int groups, int inner, int runs, uint64_t seed, unsigned long long limit, float eps,
               int resident) {
  const Layout& L = m.layout;
  const int need = DIM == 3 ? L.max_elem : L.max_items;
  if (need > N * BT || L.max_own > BT || L.max_local > kItemSlots || L.vmask.empty()) {
    std::printf("blocks of %d do not fit\n", need);
    return 2;
  }
  std::mt19937_64 rng(seed);
  Solve s(m);
  const float large = DIM == 3 ? EIK_LARGENUM_3D : EIK_LARGENUM_2D;
  int failures = 0, gave_up = 0, unfinished = 0, shortened = 0;
  long long visits = 0;
  for (int run = 0; run < runs; ++run) {
    s.T.assign((size_t)m.nv, large);
    s.seen.assign((size_t)m.nv + L.halo.size(), EIK_INF);
    s.out.assign((size_t)m.nv, -1.f);
    std::memset(s.ctl, 0, sizeof s.ctl);
    Sched& sc = s.a.s;
    sched_shape(sc, L.nblocks, groups);
    s.words.assign((size_t)sc.owners * sc.stride, (unsigned long long)kClean);
    sc.word = s.words.data();
    sc.ctl = reinterpret_cast<unsigned long long*>(s.ctl);
    sc.done = reinterpret_cast<decltype(sc.done)>(s.ctl + kSchedCtlBytes / 2);
    sc.wait_limit = limit ? limit : ~0ull;
    s.a.eps = eps;
    s.a.max_inner = inner;
    s.a.max_visits = 1 << 30;
    s.a.max_local = L.max_local;
    s.a.max_elem = L.max_elem;
    s.a.max_queue = DIM != 3 ? 0 : CAP ? L.max_items / 20 : L.max_items;
    const int nsrc = 1 + (int)(rng() % 3);
    for (int k = 0; k < nsrc; ++k) {
      const int32_t v = L.iperm[rng() % (uint64_t)m.nv], b = L.owner[(size_t)v];
      s.T[(size_t)v] = 0.f;
      auto mark = [&](int32_t c) { s.words[sched_slot(sc, c)] = 0ull; };
      mark(b);
      for (int32_t j = L.dep_start[(size_t)b]; j < L.dep_start[(size_t)b + 1]; ++j) mark(L.dep[(size_t)j]);
    }
    std::vector<Group> gs((size_t)groups);
    const size_t lds = loop_lds_bytes(DIM, L.max_local, L.max_elem, s.a.max_queue);
    for (Group& g : gs) {
      g.lds.resize(lds / sizeof(uint4) + 64);
      std::memset(&g.sh, 0, sizeof g.sh);
    }
    const ModelBlocks blocks{s};
    const char* err = simt::run((unsigned)groups, BT, seed * 1000003u + (uint64_t)run, (unsigned)resident, [&] {
      Group& g = gs[blockIdx.x];
      const int end = resident_loop<DIM, N, BT, CAP>(s.a, blocks, blockIdx.x, g.lds.data(), g.sh);
      write_times(s.a.s, end, s.T.data(), L.iperm.data(), m.nv, s.out.data(), &g.sh.block);
      g.end = end;
    });
    if (err) {
      std::printf("run %d: %s\n", run, err);
      return 1;
    }
    bool ended = false;
    const int before = gave_up;
    for (Group& g : gs) {
      ended = ended || g.end == kNoWork;
      gave_up += g.end == kGaveUp;
      visits += (long long)g.sh.acc[0];
    }
    const int given = gave_up - before;
    int unwritten = 0;
    for (int64_t v = 0; v < m.nv; ++v) unwritten += s.out[(size_t)v] != s.T[(size_t)L.iperm[(size_t)v]];
    if (unwritten) {
      ++failures;
      std::printf("run %d: %d of %lld times not written\n", run, unwritten, (long long)m.nv);
    }
    if (!ended) {
      ++unfinished;
      continue;
    }
    shortened += given > 0;
    int dirty = 0;
    for (unsigned long long w : s.words) dirty += w != (unsigned long long)kClean;
    const int bad = improvable(s, eps > 0.f);
    if (dirty || bad) {
      ++failures;
      std::printf("run %d: ended with %d words not clean, %d solves that lower a time\n", run, dirty, bad);
    }
  }
  std::printf("%d runs of %d blocks, %lld visits, gave up %d, ended short %d, unfinished %d, failures %d\n",
              runs, L.nblocks, visits, gave_up, shortened, unfinished, failures);
  return failures ? 1 : 0;
}

}  // namespace

int main(int argc, char** argv) {
  if (argc < 9 || argc > 11) return 2;
  const std::string kind = argv[1];
  const int size = std::atoi(argv[2]), vpb = std::atoi(argv[3]), groups = std::atoi(argv[4]);
  const int inner = std::atoi(argv[5]), runs = std::atoi(argv[6]);
  const uint64_t seed = std::strtoull(argv[7], nullptr, 10);
  const unsigned long long limit = std::strtoull(argv[8], nullptr, 10);
  const float eps = argc > 9 ? (float)std::atof(argv[9]) : 0.f;
  const int resident = argc > 10 ? std::atoi(argv[10]) : groups;
  Mesh m;
  if (kind.size() != 4) return 2;
  const bool cap = kind == "cap4", tets = cap || kind.substr(0, 3) == "tet";
  if (tets ? gen_kuhn_cube(size, 0.2f, seed, m) : gen_icosphere(size, m)) return 2;
  // uneven speeds, so that times arrive out of order
  std::mt19937_64 rng(seed);
  m.metric_kind = 1;
  m.metric.resize((size_t)m.ne);
  for (float& f : m.metric) f = std::exp(1.5f * (float)((double)(rng() >> 11) * 0x1p-53 - 0.5));
  if (!tets) tri_virtual_faces(m);
  if (partition_by_size(m, vpb) || build_layout(m)) return 2;
  const int n = std::atoi(kind.c_str() + 3);
  if (cap) return run_solves<3, 4, 256, true>(m, groups, inner, runs, seed, limit, eps, resident);
  if (tets) return n == 2 ? run_solves<3, 2, 512>(m, groups, inner, runs, seed, limit, eps, resident)
                          : run_solves<3, 4, 256>(m, groups, inner, runs, seed, limit, eps, resident);
  return n == 1   ? run_solves<2, 1, 256>(m, groups, inner, runs, seed, limit, eps, resident)
         : n == 2 ? run_solves<2, 2, 512>(m, groups, inner, runs, seed, limit, eps, resident)
                  : run_solves<2, 4, 512>(m, groups, inner, runs, seed, limit, eps, resident);
}
