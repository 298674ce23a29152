// visit_loop.h -- the loop of a persistent workgroup over register-resident blocks (device code),
// shared by single solves (solver.hip) and multi-solve launches (batch.hip).
#pragma once

#include <type_traits>

#include "block_sched.h"
#include "device.h"
#include "resident.h"

namespace eik {

// Elements per thread of the tet shapes: with 256 and 512 threads as many as 128 VGPRs hold beside the
// solver, so that a block takes the smaller workgroup (the smallest blocks have a shape of 4).
template <int BT>
constexpr int kTetN = BT == 1024 ? 4 : 6;

// What a visit reads of a block's mesh and solve.
struct BlockData {
  const BlockDesc* blocks;
  const void* elems;
  const int32_t* halo;
  float* T;
  float* seen;
  const uint64_t* vmask;
  const int32_t* dep_start;
  const int32_t* dep;
  const float* rmult;  // a factor per record on the squared lengths, or null
  float unit;          // tets: of the heights (Layout::height_unit)
  TriItems items;      // triangles
  int32_t b;           // the block within its mesh
  int32_t base;        // launch-wide index of its mesh's first block
};

struct LoopArgs {
  Sched s;
  float eps;
  int32_t max_inner;
  int64_t max_visits;  // runaway guard: visits of one workgroup after which it marks nothing
  int32_t max_local;   // LDS strides: local vertices and elements of the largest block
  int32_t max_elem;
  int32_t max_queue;   // pairs the work-item queue holds (tets)
};

// The workgroup's static LDS.
struct LoopShared {
  unsigned long long acc[kNumCounters];  // its tally
  int64_t max_visits;  // LoopArgs (read here with what it is compared with)
  int flag[3];       // a sweep's "a time fell", in a ring over the sweeps
  int full;          // the last visit with a sweep that selected more pairs than the queue holds
  int qn[2];         // work-item counters of alternate sweeps (tets)
  unsigned mark[2];  // dependents whose halo holds a vertex lowered in this visit
  int block;
  unsigned waiting;  // smallest key of the owner's waiting blocks when last looked
  unsigned key;      // smallest time the visit lowered
  int crowd;         // dirty blocks seen waiting when this one was claimed
};

// Words of an LDS array of local vertices; what follows three of them is 16-byte aligned.
__host__ __device__ inline int32_t lds_stride(int32_t max_local) { return (max_local + 3) & ~3; }

// Dynamic LDS of the loop, bytes, with a work-item queue of max_queue pairs (tets).
inline size_t loop_lds_bytes(int dim, int32_t max_local, int32_t max_elem, int32_t max_queue) {
  size_t n = sizeof(float) * 3 * (size_t)lds_stride(max_local);
  if (dim == 3) n += 2 * sizeof(uint4) * (size_t)max_elem + sizeof(uint16_t) * (size_t)max_queue;
  return n;
}

// Pairs the work-item queue holds: all a block has, unless that costs the CU a workgroup and as many
// as it has elements do not (a sweep selects about a tenth of the pairs; what a full queue turns
// away is selected again by the next sweep).  For the workgroups of 512 threads: 64 cubes at 192 vertices
// per block 8.1 -> 5.2 ms with two of them instead of one.
inline int32_t loop_queue(int dim, int bt, int32_t max_local, int32_t max_elem, int32_t max_items) {
  if (dim != 3) return 0;
  if (bt != 512) return max_items;
  // what each of the CU's workgroups has beside the static LDS
  const size_t most = 163840 / (1024 / bt) - ((sizeof(LoopShared) + 15) & ~(size_t)15);
  const size_t none = loop_lds_bytes(dim, max_local, max_elem, 0);
  if (none + sizeof(uint16_t) * (size_t)max_items <= most) return max_items;
  if (none + sizeof(uint16_t) * (size_t)max_elem > most) return max_items;
  return (int32_t)((most - none) / sizeof(uint16_t));
}

// Blocks seen waiting when a tet block is claimed from which on its visit runs up to max_inner sweeps:
// while work waits, a block is loaded for more than one sweep (96^3 cube with 16 sources, 1 sweep
// always / 1 / 8 / 16 waiting blocks: 1.66 / 1.52 / 1.52 / 1.57 ms); while workgroups wait for work,
// one sweep, whose times reach the dependents sooner.
constexpr int kCrowd = 8;

// One whole wave: the next block (look: or kNothing), with the time spent in the workgroup's tally.  THIN: see
// sched_look.
template <bool THIN>
__device__ __forceinline__ int32_t find_next(const Sched& s, Finder& f, unsigned long long* acc,
                                             bool look = false) {
  const unsigned long long w0 = wall_clock64();
  const int32_t b = look ? sched_look<THIN>(s, f) : sched_find<THIN>(s, f);
  if (__lane_id() == 0) {
    acc[6] += wall_clock64() - w0;
    if (b == kGaveUp) acc[kCntAbandoned] += 1;
  }
  return b;
}

// Writes a solve's times in caller order, when a workgroup has found no further block (end).  At the end of
// the solve (every visit has ended and every published time has landed) each workgroup writes a stripe of
// them.  Where workgroups have given up, their stripes would be missing: the ones that find the end, or
// the last to give up (then the times are not final), write stretches that they take from a counter until
// none is left.  A workgroup that gives up counts itself in the word that says that the solve has ended:
// either it finds the end there, or whoever finds the end later finds the count.  (Counted and looked at
// here, not where blocks are found: there it cost every look registers, level-8 icosphere 1.64 -> 1.71 ms.)
constexpr int64_t kOutStretch = 8192;
__device__ __forceinline__ void write_times(const Sched& s, int end, const float* T, const int32_t* iperm,
                                            int64_t nv, float* out, int* shared) {
  if (!out) return;
  enum { kStripe, kStretches, kNothingToWrite };
  __syncthreads();  // (the shared word has been read)
  if (threadIdx.x == 0) {
    unsigned long long* word = reinterpret_cast<unsigned long long*>(s.done);
    if (end == kNoWork) {
      *shared = load_word(word) >> 32 ? kStretches : kStripe;
    } else {
      const unsigned long long old =
          __hip_atomic_fetch_add(word, 1ull << 32, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      *shared = (uint32_t)old || (uint32_t)(old >> 32) + 1u == s.owners ? kStretches : kNothingToWrite;
    }
  }
  __syncthreads();
  const int what = __builtin_amdgcn_readfirstlane(*shared);
  if (what == kStripe) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nv; i += stride)
      out[i] = load_T<true>(T + iperm[i]);
  }
  while (what == kStretches) {
    __syncthreads();
    if (threadIdx.x == 0)
      *shared = (int)(uint32_t)__hip_atomic_fetch_add(s.done + 2, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    const int64_t from = (int64_t)*shared * kOutStretch;
    if (from >= nv) break;
    const int64_t to = from + kOutStretch < nv ? from + kOutStretch : nv;
    for (int64_t i = from + threadIdx.x; i < to; i += blockDim.x) out[i] = load_T<true>(T + iperm[i]);
  }
}

// The loop of one workgroup over the blocks of a launch, until the solve has ended or it gives up:
// blocks whose element data fits the workgroup's registers
// (resident.h): N items or elements per thread.  Blocks are found and handed on as block_sched.h
// says; a workgroup that visits a block again, at once or when it is dirty again and nothing smaller
// waits, keeps its registers and LDS, and only times are read again.  A visit of a tet block is one
// sweep while few blocks wait (kCrowd); a block that has not converged is visited again at once
// unless a block of the same owner waits with a smaller time.
// What bounds it: the chain of a visit (64^3 cube: 2.7 us a sweep, of which 2.3 us without other
// workgroups on the CU, 0.4 us until its times have landed, 1.0 us of marks and halo loads, 3.1 us to load a
// block into the registers and LDS every third visit), and on large tet meshes the instructions too:
// the 96^3 solve keeps the vector units issuing for half of its time.  Held to 128 VGPRs, so that four
// workgroups fit a CU: with 45 of them spilled the 96^3 solve took 2.1 ms, without 1.7.
// Visit kernels, against the staged records of visit_block and one queue ring: 64^3 cube 1.045 ->
// 0.63 ms, 96^3 with 16 sources 3.67 -> 1.41, 33^3 tensor 0.448 -> 0.267, 16^3 0.285 -> 0.135; level-8
// icosphere 3.29 -> 1.51, level-7 anisotropic 1.02 -> 0.48, level 5 0.328 -> 0.118, 32^2 square 0.158 ->
// 0.057.
// blocks(g) gives the data of launch-wide block g; me is the workgroup's owner index.  Returns kNoWork
// or kGaveUp.  The workgroup's tally is added to sh.acc, which the caller has cleared (behind a
// barrier) and flushes.
template <int DIM, int N, int BT, bool CAP, class Blocks>
__device__ __forceinline__ int resident_loop(const LoopArgs& a, const Blocks& blocks, uint32_t me,
                                             uint4* lds4, LoopShared& sh) {
  const int tid = threadIdx.x;
  // the times first: their offsets in the LDS are constants of the instructions that read them
  const int ls = lds_stride(a.max_local);
  float* sT = reinterpret_cast<float*>(lds4);
  float* sP = sT + ls;
  int* sHidx = reinterpret_cast<int*>(sP + ls);
  uint4* sA = reinterpret_cast<uint4*>(sHidx + ls);
  uint4* sB = sA + (DIM == 3 ? a.max_elem : 0);
  uint16_t* sQ = reinterpret_cast<uint16_t*>(sB + (DIM == 3 ? a.max_elem : 0));
  const float eps = a.eps, large = DIM == 3 ? EIK_LARGENUM_3D : EIK_LARGENUM_2D;
  // (the barrier before the first visit orders these)
  if (tid < 3) sh.flag[tid] = 0;
  if (tid < 2) sh.qn[tid] = 0;
  if (tid < 2) sh.mark[tid] = 0;
  if (tid == 0) {
    sh.key = kClean;
    sh.max_visits = a.max_visits;
  }
  if (tid == 0) sh.full = 0;
  // the second wave looks for work, while the first hands on what the last visit did
  const bool finder = tid >= 64 && tid < 128;
  Finder f;
  if (finder) sched_enter(a.s, f, me);
  int ring = 0;  // sweeps run so far, modulo 3
  int qc = 0;
  uint32_t solves = 0;
  int visit = 1;
  __syncthreads();
  if (finder) {
    const int32_t nb = find_next<false>(a.s, f, sh.acc);
    if (tid == 64) {
      sh.block = nb;
      sh.crowd = f.others;
    }
  }
  __syncthreads();
  int b = __builtin_amdgcn_readfirstlane(sh.block);
  while (b >= 0) {
    unsigned long long t0 = wall_clock64();
    const int cur = b;
    // the resident block: one owned vertex per thread, its items or elements in registers
    const uint32_t slot = sched_slot(a.s, b);
    const BlockData m = blocks(b);
    const BlockDesc d = m.blocks[m.b];
    float* T = m.T;
    float* seen = m.seen + d.vstart + d.hstart;
    const int32_t s0 = m.dep_start[m.b];
    const int ndep = m.dep_start[m.b + 1] - s0;
    const float* rmult = m.rmult ? m.rmult + d.estart : nullptr;
    float own = 0.f;  // the owned vertex's time as last published
    uint64_t vm = 0;
    uint32_t dep_slot = 0;
    std::conditional_t<DIM == 2, TriRegs<N>, TetRegs<N>> r;
    const int t = this_thread();
    if (t < d.nown) {
      own = load_T<true>(T + d.vstart + t);
      sP[t] = seen[t];
      vm = m.vmask[d.vstart + t];
      sT[t] = own;
    }
    for (int i = t; i < d.nhalo; i += BT) {
      const int32_t h = m.halo[d.hstart + i];
      sHidx[i] = h;
      sP[d.nown + i] = seen[d.nown + i];
      sT[d.nown + i] = load_T<true>(T + h);
    }
    if (t < ndep) dep_slot = sched_slot(a.s, m.base + m.dep[s0 + t]);
    if constexpr (DIM == 2)
      tri_load<N, BT>(r, m.items, m.items.range[m.b], rmult);
    else
      tet_load<N, BT>(r, m.elems, d, sA, sB, m.unit, rmult);
    wait_memory();  // the copies to LDS too
    __syncthreads();
    if constexpr (DIM == 2) tri_seen<N>(r, sP);
    else tet_seen<N>(r, sP);
    unsigned long long t1 = wall_clock64();
    bool rerun = false;
    unsigned waiting = kClean;  // smallest key of the owner's other blocks when last looked
    // visits of this block: the next one at once, or when the block is dirty again and nothing
    // smaller waits
    for (;;) {
      const int inner = DIM == 2 || sh.crowd >= kCrowd ? a.max_inner : 1;
      uint64_t marks = 0;  // dependents holding this thread's vertex, if it fell
      uint32_t key = kClean;
      // The owned time left in `seen` by a visit whose last sweep lowered times: at least every value that the
      // block's elements were last evaluated with.  For tets the time before the last sweep.  For triangles
      // the one published before that: no barrier parts the publishing from the next sweep, which lowers
      // times in place, so the time published after the last sweep but one may be one of the last sweep's
      // already, which items evaluated before it fell have not seen.
      float own_last = own, own_seen = own;
      int sweep = 0;
      bool conv = false;
      while (sweep < inner) {
        bool ch = false;
        int nq = 1;
        if constexpr (DIM == 2) {
          ch = tri_sweep<N>(r, sT, large, eps, solves);
        } else {
          tet_select<N, BT, CAP>(r, d.nelem, sT, sQ, a.max_queue, &sh.qn[qc], &sh.flag[ring],
                            &sh.full, visit);
          __syncthreads();
          nq = sh.qn[qc];
          if (CAP) nq = min(nq, a.max_queue);
          if (tid == 0) sh.qn[qc ^ 1] = 0;
          qc ^= 1;
          if (nq) ch = tet_solve<N, BT>(r, sA, sB, sQ, nq, sT, large, eps, solves);
        }
        if (ch) sh.flag[ring] = 1;
        // (no pair selected: no time fell, and no thread waits for another's solve)
        if (nq) __syncthreads();
        const int any = nq ? sh.flag[ring] : 0;
        ring = ring == 2 ? 0 : ring + 1;
        if (tid == 0) sh.flag[ring == 2 ? 0 : ring + 1] = 0;
        ++sweep;
        // publish the owned times that fell
        own_seen = DIM == 2 ? own_last : own;
        own_last = own;
        if (tid < d.nown) {
          const float v = sT[tid];
          if (v < own) {
            own = v;
            (void)__hip_atomic_fetch_min(reinterpret_cast<unsigned*>(T + d.vstart + tid),
                                         __float_as_uint(v), __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
            marks |= vm;
            key = __float_as_uint(v);
          }
        }
        if (!any) {
          conv = true;
          break;
        }
      }
      const unsigned long long t2 = wall_clock64();
      // visits beyond the bound mark nothing more (runaway guard)
      const bool cap_ok = (int64_t)sh.acc[0] < sh.max_visits;
      const bool more = !conv && cap_ok;
      // marks made from here on are seen by the halo loads of the next visit or after it
      if (more && tid == 0) sched_again(a.s, slot);
      // reduced over the wave first, and by one lane: the compiler turns an LDS atomic with a uniform
      // address into a scalar loop over the lanes (a third of a triangle sweep)
      if (__ballot(key != kClean)) {
        const uint32_t lo = wave_or((uint32_t)marks), hi = wave_or((uint32_t)(marks >> 32));
        key = wave_umin(key);
        if (__lane_id() == 63) {
          lds_min(&sh.key, key);
          lds_or(&sh.mark[0], lo);
          lds_or(&sh.mark[1], hi);
        }
      }
      // What the owner's other blocks wait with, for the next visit's decision.  In single solves of
      // triangles, most of whose visits are followed by another, it is loaded in the same wait as the
      // publishing: 301^2 square with 16 sources 0.334 -> 0.322 ms, level-8 icosphere 1.56 -> 1.51 (in
      // launches of several solves, with more visits that converge, 1.88 -> 1.93).  It sees the owner's
      // first 64 blocks: with more of them a visit may be followed by another though a smaller one waits,
      // which is right too (level-9 icosphere, 80 blocks per owner, 5.05 ms; looking at all 5.27).
      constexpr bool kEarlyLook = DIM == 2 && Blocks::kSingle;
      unsigned long long word = ~0ull;
      if (kEarlyLook && tid < 64 && (uint32_t)tid < a.s.per_owner && a.s.per_owner > 1)
        word = load_word(&a.s.word[me * a.s.stride + tid]);
      // the published times have reached the device's coherence point before the dependents are
      // marked
      wait_memory();
      __syncthreads();
      const unsigned long long tq = wall_clock64();
      const uint32_t vkey = sh.key;
      const bool full = DIM == 3 && CAP && sh.full == visit;
      ++visit;
      const uint32_t lkey = full ? 0u : vkey;  // what the block waits with: its smallest new time
      // visited again at once, unless another of the owner's blocks waits with a smaller time
      const bool again = more && !(waiting < lkey);
      if (tid < 64) {
        const uint64_t mask = (uint64_t)sh.mark[0] | ((uint64_t)sh.mark[1] << 32);
        if (cap_ok && tid < ndep && ((mask >> tid) & 1ull)) sched_mark(a.s, dep_slot, vkey);
        __builtin_amdgcn_wave_barrier();  // (the mask has been read by every lane)
        if (tid < 2) sh.mark[tid] = 0;
        if (tid == 0) {
          VisitResult vr;
          vr.sweeps = sweep;
          vr.t_load = t1 - t0;
          vr.t_sweep = t2 - t1;
          vr.t_wb = tq - t2;
          tally_visit(sh.acc, d, vr, 0, kAlgoElemBytes<DIM>, tq - t0, rerun, rerun);
        }
        if (again) {
          // (with one block per owner there is no other, and no wait for its word: 33^3 cube 0.281 ->
          // 0.267 ms, level-5 icosphere 0.130 -> 0.118)
          const uint32_t w = kEarlyLook ? wave_umin((word >> 32) == 0ull ? (uint32_t)word : kClean)
                             : a.s.per_owner > 1 ? sched_waiting(a.s, me) : kClean;
          if (tid == 0) sh.waiting = w;
          if (tid == 0) sh.acc[10] += wall_clock64() - tq;
        } else {
          wait_memory();  // the marks have landed before this block can count as clean
          if (tid == 0) {
            sched_leave(a.s, slot, more ? lkey : kClean);
            sh.waiting = kClean;
            sh.acc[10] += wall_clock64() - tq;
          }
        }
      } else if (!again) {
        if (finder) {
          const int32_t nb = a.s.per_owner > 1 ? find_next<false>(a.s, f, sh.acc, true) : kNothing;
          if (tid == 64) {
            sh.block = nb;
            sh.crowd = f.others;
          }
        }
      } else {
        // the halo times of the next visit (by the waves that mark nothing)
        for (int i = tid - 64; i < d.nhalo; i += BT - 64)
          sT[d.nown + i] = load_T<true>(T + sHidx[i]);
      }
      if (!again) {
        // what this visit evaluated the block's elements with: every time, but for the owned
        // vertices that fell in the last sweep of a visit cut off by the sweep cap (triangles: or of one
        // that ended with falls within eps).  A later visit that misses these (they are plain stores)
        // evaluates more than it has to.  After a full queue, nothing counts as evaluated.
        if (tid < d.nown) seen[tid] = full ? EIK_INF : conv && (DIM == 3 || eps == 0.f) ? own : own_seen;
        for (int i = tid; i < d.nhalo; i += BT) seen[d.nown + i] = full ? EIK_INF : sT[d.nown + i];
      }
      __syncthreads();
      waiting = sh.waiting;
      if (tid == 0) sh.key = kClean;
      t0 = t1 = wall_clock64();
      rerun = again;
      if (again) continue;
      b = __builtin_amdgcn_readfirstlane(sh.block);
      if (b == kNothing) {
        __syncthreads();
        if (finder) {
          const int32_t nb = find_next<false>(a.s, f, sh.acc);
          if (tid == 64) {
            sh.block = nb;
            sh.crowd = f.others;
          }
        }
        __syncthreads();
        b = __builtin_amdgcn_readfirstlane(sh.block);
      }
      if (b != cur) break;
      // the same block, still resident: only times may have fallen (the owned ones if another
      // workgroup visited the block meanwhile)
      if (tid < d.nown) {
        own = load_T<true>(T + d.vstart + tid);
        sT[tid] = own;
      }
      for (int i = tid; i < d.nhalo; i += BT) sT[d.nown + i] = load_T<true>(T + sHidx[i]);
      __syncthreads();
      t1 = wall_clock64();
    }
  }
  unsigned long long all = solves;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) all += __shfl_down(all, off, 64);
  if (__lane_id() == 0 && all) atomicAdd(&sh.acc[3], all);
  __syncthreads();
  return b;
}

}  // namespace eik
