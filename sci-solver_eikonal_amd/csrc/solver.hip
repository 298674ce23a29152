// solver.hip -- device state, kernels and the solve entry points of the C ABI.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <mutex>
#include <string>
#include <type_traits>
#include <vector>

#include "device.h"
#include "visit_loop.h"

namespace eik {

// Results of up to this many vertices are copied out through pinned memory in the solve's one wait;
// larger ones straight to the caller's memory after it.
constexpr int64_t kSmallOut = 65536;
// Up to this many seeds are read from pinned host memory by the kernel that needs them, without a copy.
constexpr int64_t kDirectSeeds = 1024;

static int dev_free(DeviceState* d) {
  if (!d) return EIK_OK;
  for (float* p : d->hist) (void)hipFree(p);
  void* ptrs[] = {d->esel, d->elen, d->rec_elem, d->vmask, d->vh_start, d->vh_pos, d->seen, d->blocks, d->elems,  d->halo,  d->iperm,
                  d->dep_start, d->dep, d->owner, d->T,      d->out,      d->stamp[0],
                  d->stamp[1], d->list[0], d->list[1], d->count, d->counters, d->sync_acc, d->seeds,
                  d->seedvals, d->words, d->sctl,
                  d->item_range, d->item_id, d->item_len, d->item_rec};
  for (void* p : ptrs)
    if (p) (void)hipFree(p);
  if (d->h_seed) (void)hipHostFree(d->h_seed);
  if (d->h_cnt) (void)hipHostFree(d->h_cnt);
  if (d->ev0) (void)hipEventDestroy(d->ev0);
  if (d->ev1) (void)hipEventDestroy(d->ev1);
  if (d->evA) (void)hipEventDestroy(d->evA);
  if (d->evB) (void)hipEventDestroy(d->evB);
  if (d->stream) (void)hipStreamDestroy(d->stream);
  delete d;
  return EIK_OK;
}

void device_release(Mesh& m) {
  dev_free(m.dev);
  m.dev = nullptr;
}

int ensure_stream(Mesh& m) {
  if (!m.dev) m.dev = new DeviceState();
  DeviceState* d = m.dev;
  if (!d->stream) {
    int ndev = 0;
    HIP_TRY(hipGetDeviceCount(&ndev));
    if (ndev <= 0) return fail(EIK_ERR_HIP, "no HIP device");
    HIP_TRY(hipGetDevice(&d->device));
    HIP_TRY(hipStreamCreateWithFlags(&d->stream, hipStreamNonBlocking));
    HIP_TRY(hipEventCreate(&d->ev0));
    HIP_TRY(hipEventCreate(&d->ev1));
    HIP_TRY(hipEventCreate(&d->evA));
    HIP_TRY(hipEventCreate(&d->evB));
  }
  return EIK_OK;
}

// ------------------------------------------------------------------------------------------
// Kernels
// ------------------------------------------------------------------------------------------
__global__ void k_fill_segs(FillSegs f) {
  if (f.begin && blockIdx.x == 0 && threadIdx.x == 0) *f.begin = wall_clock64();
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  const int64_t i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  for (int k = 0; k < f.count; ++k) {
    int32_t* p = f.p[k];
    const int32_t v = f.v[k];
    for (int64_t i = i0; i < f.n[k]; i += stride) p[i] = v;
  }
  for (int k = 0; k < 2; ++k)
    for (int64_t i = i0; i < f.nwords[k]; i += stride) f.words[k][i] = kClean;
}

void launch_fill(const FillSegs& f, hipStream_t s) {
  int64_t most = std::max<int64_t>(1, std::max(f.nwords[0], f.nwords[1]));
  for (int k = 0; k < f.count; ++k) most = std::max(most, f.n[k]);
  hipLaunchKernelGGL(k_fill_segs, dim3((unsigned)std::min<int64_t>(grid1d(most, 256), 2048)),
                     dim3(256), 0, s, f);
}

// The active blocks of an iteration of the synchronous scheduler: their number and list, and per
// block the last iteration it was put on a list of this parity.
struct Active {
  int32_t* stamp;
  int32_t* list;
  int32_t* count;
};

// One whole wave: lane j of the first m puts block c on the list of iteration it, unless it is there.
__device__ __forceinline__ void activate(const Active& next, int32_t it, bool mine, int32_t c) {
  const bool add = mine && atomicExch(&next.stamp[c], it) != it;
  const uint64_t bal = __ballot(add);
  if (!bal) return;
  int base = 0;
  if (__lane_id() == 0) base = atomicAdd(next.count, __popcll(bal));
  base = __builtin_amdgcn_readfirstlane(base);
  if (add) next.list[base + __popcll(bal & lane_mask_lt())] = c;
}

// A source's time as the words order times: -0 counts as 0 (its own bits are the largest word).
static __device__ __forceinline__ unsigned seed_key(const float* vals, int64_t i) {
  return __float_as_uint(vals ? vals[i] + 0.f : 0.f);
}

// seeds: caller ids -> new ids; T = value; the owner block of each seed and its dependents are active
// in iteration 1 (one workgroup per seed).
__global__ void k_sync_seed(const int32_t* seeds, const float* vals, int64_t n, const int32_t* iperm,
                            const int32_t* owner, const int32_t* dep_start, const int32_t* dep,
                            float* T, Active next) {
  for (int64_t i = blockIdx.x; i < n; i += gridDim.x) {
    const int32_t v = iperm[seeds[i]];
    if (threadIdx.x == 0)
      atomicMin(reinterpret_cast<unsigned*>(&T[v]), seed_key(vals, i));
    const int32_t b = owner[v], s0 = dep_start[b], nd = dep_start[b + 1] - s0;
    for (int j0 = 0; j0 <= nd; j0 += 64) {
      const int j = j0 + (int)threadIdx.x;
      activate(next, 1, j <= nd, j < nd ? dep[s0 + j] : b);
    }
  }
}

struct SyncArgs {
  VisitArgs v;
  size_t rec_lds_bytes;
  Active now, next;
  int32_t* count_after;      // cleared here: the visits of the next iteration fill it
  int32_t* last;             // the last iteration that visited a block
  unsigned long long* told;  // pinned host memory: last << 32 | it, once iteration it has begun
  const int32_t* dep;
  int32_t nb;
  int32_t it;
  float* snap;               // the times after this iteration (the per-iteration history), or null
  unsigned long long* acc;   // kSyncSlots slot lines of counters
  int32_t elem_bytes;        // algorithmic bytes per element (visit_algo_bytes)
  TriItems items;            // register-resident visits: triangles, and the LDS (LoopArgs)
  int32_t max_local, max_elem, max_queue;
  float height_unit;
};
constexpr int kSnapBlocks = 16;  // blocks whose times a workgroup copies to the history

// Adds one visit's counters to the workgroup's slot line (kSyncSlots lines, summed by
// k_sum_slots after the solve).
__device__ void block_counters(unsigned long long* acc, const BlockDesc& d, int sweeps,
                               uint64_t solves, int elem_bytes, unsigned long long busy_ticks,
                               const VisitResult& r, unsigned long long* sRed) {
  uint64_t s = solves;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
  if (__lane_id() == 0) atomicAdd(sRed, (unsigned long long)s);
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long* c = acc + (blockIdx.x % kSyncSlots) * kSyncSlotWords;
    atomicAdd(&c[0], 1ull);
    atomicAdd(&c[1], (unsigned long long)d.nown);
    atomicAdd(&c[2], (unsigned long long)sweeps);
    atomicAdd(&c[3], *sRed);
    atomicAdd(&c[4], visit_algo_bytes(elem_bytes, d));
    atomicAdd(&c[kCntAlgoLoaded], visit_algo_bytes(elem_bytes, d));
    atomicAdd(&c[5], busy_ticks);
    atomicAdd(&c[7], r.t_load);
    atomicAdd(&c[8], r.t_sweep);
    atomicAdd(&c[9], r.t_wb);
  }
}

// counters[k] += the sum of word k over the kSyncSlots slot lines
__global__ void k_sum_slots(const unsigned long long* acc, unsigned long long* counters) {
  const int k = threadIdx.x;
  if (k >= kNumCounters) return;
  unsigned long long s = 0;
  for (int i = 0; i < kSyncSlots; ++i) s += acc[i * kSyncSlotWords + k];
  counters[k] += s;
}

// One outer iteration: workgroup i visits the i-th active block and puts the blocks whose halo holds a
// vertex it lowered, and itself if it did not converge, on the list of the next iteration.  Replaces
// the reference's host loop over blockCon and m_BlockNeighbor (meshFIM3dEikonal.cu:445-488, 518-527;
// meshFIM2d_eikonal.cu:730-799).  The host enqueues several iterations without waiting, so the grid
// covers every block and the workgroups beyond this iteration's active count leave at once (an
// iteration after convergence is empty).  For the history, a visit writes its block's times, and
// the workgroups from nb on copy those of the blocks that are not active, which no one changes now:
// one launch per iteration (48^3 cube with history, 43 iterations, in all: 1.35 -> 1.06 ms; a launch
// that looked through every block's suppliers took 5 us of each, the host's waits 0.2 ms).
//
// The block this workgroup visits, or -1 (the history copy done).
__device__ __forceinline__ int sync_begin(const SyncArgs& a) {
  const int n = *a.now.count;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    *a.count_after = 0;
    const int32_t last = n > 0 ? a.it : *a.last;
    *a.last = last;
    __hip_atomic_store(a.told, (unsigned long long)last << 32 | (unsigned)a.it, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_SYSTEM);
  }
  if ((int)blockIdx.x < a.nb) return (int)blockIdx.x < n ? a.now.list[blockIdx.x] : -1;
  if (n <= 0) return -1;
  const int c0 = ((int)blockIdx.x - a.nb) * kSnapBlocks;
  for (int c = c0 + (int)(threadIdx.x >> 6); c < min(c0 + kSnapBlocks, a.nb); c += (int)(blockDim.x >> 6)) {
    if (a.now.stamp[c] == a.it) continue;
    const BlockDesc d = a.v.blocks[c];
    for (int i = (int)__lane_id(); i < d.nown; i += 64) a.snap[d.vstart + i] = a.v.T[d.vstart + i];
  }
  return -1;
}

// After a visit: the next iteration's blocks (first wave), the history.
__device__ __forceinline__ void sync_end(const SyncArgs& a, int b, const BlockDesc& d, bool bnd_changed,
                                         bool converged, const float* sT) {
  if (threadIdx.x < 64) {
    const int32_t s0 = a.v.dep_start[b];
    const int nd = bnd_changed ? a.v.dep_start[b + 1] - s0 : 0;
    const int m = nd + (converged ? 0 : 1);
    for (int j0 = 0; j0 < m; j0 += 64) {
      const int j = j0 + (int)threadIdx.x;
      activate(a.next, a.it + 1, j < m, j < nd ? a.dep[s0 + j] : b);
    }
  }
  if (a.snap)
    for (int i = (int)threadIdx.x; i < d.nown; i += (int)blockDim.x) a.snap[d.vstart + i] = sT[i];
}

template <int DIM>
__global__ __launch_bounds__(kBlockThreads) void k_visit_sync(SyncArgs a) {
  extern __shared__ uint4 lds4[];
  __shared__ int sFlag[4];
  __shared__ int sQn[2];  // work-item counters of alternate chunks
  __shared__ unsigned long long sRed;
  const int b = sync_begin(a);
  if (b < 0) return;
  const BlockDesc d = a.v.blocks[b];
  VisitLds l = carve_lds<DIM>(lds4, a.rec_lds_bytes, a.v.queue_cap, d);
  if (threadIdx.x == 0) sRed = 0;
  uint64_t solves = 0;
  const unsigned long long t0 = wall_clock64();
  VisitResult r = visit_block<DIM, false>(a.v, b, l.rec, l.T, l.old, l.chg, l.hidx, l.vm, l.q, l.mark,
                                          sFlag, sQn, &solves);
  sync_end(a, b, d, r.bnd_changed, r.converged, l.T);
  block_counters(a.acc, d, r.sweeps, solves, a.elem_bytes, wall_clock64() - t0, r, &sRed);
}

// The same visit with the block's element data in registers (resident.h), where the blocks fit: its
// sweeps are the ones of the persistent kernel (visit_loop.h).  Kernel ms against k_visit_sync: 48^3
// cube with history 0.91 -> 0.82, 64^3 1.60 -> 1.51, 96^3 with 16 sources 3.87 -> 3.65, level-7
// anisotropic icosphere 1.42 -> 1.22, level 5 0.45 -> 0.30, 32^2 square 0.21 -> 0.14.
template <int DIM, int N, int BT, bool CAP = false>
__global__ __launch_bounds__(BT) __attribute__((amdgpu_waves_per_eu(4))) void k_visit_sync_resident(SyncArgs a) {
  extern __shared__ uint4 lds4[];
  __shared__ int sFlag[3], sQn[2], sBnd, sFull;
  __shared__ unsigned long long sRed;
  const int b = sync_begin(a);
  if (b < 0) return;
  const BlockDesc d = a.v.blocks[b];
  const int tid = threadIdx.x;
  const int ls = lds_stride(a.max_local);
  float* sT = reinterpret_cast<float*>(lds4);
  float* sP = sT + ls;
  uint4* sA = reinterpret_cast<uint4*>(sP + 2 * ls);
  uint4* sB = sA + (DIM == 3 ? a.max_elem : 0);
  uint16_t* sQ = reinterpret_cast<uint16_t*>(sB + (DIM == 3 ? a.max_elem : 0));
  const float eps = a.v.eps, large = a.v.large;
  float* T = a.v.T;
  float* seen = a.v.seen + d.vstart + d.hstart;
  if (tid < 3) sFlag[tid] = 0;
  if (tid < 2) sQn[tid] = 0;
  if (tid == 0) {
    sRed = 0;
    sBnd = sFull = 0;
  }
  const unsigned long long t0 = wall_clock64();
  float own = 0.f;
  if (tid < d.nown) {
    own = T[d.vstart + tid];
    sP[tid] = seen[tid];
    sT[tid] = own;
  }
  for (int i = tid; i < d.nhalo; i += BT) {
    sP[d.nown + i] = seen[d.nown + i];
    sT[d.nown + i] = T[a.v.halo[d.hstart + i]];
  }
  std::conditional_t<DIM == 2, TriRegs<N>, TetRegs<N>> r;
  if constexpr (DIM == 2) tri_load<N, BT>(r, a.items, a.items.range[b], nullptr);
  else tet_load<N, BT>(r, a.v.elems, d, sA, sB, a.height_unit, nullptr);
  wait_memory();  // the copies to LDS too
  __syncthreads();
  if constexpr (DIM == 2) tri_seen<N>(r, sP);
  else tet_seen<N>(r, sP);
  const unsigned long long t1 = wall_clock64();
  uint32_t solves = 0;
  float last = own;  // the owned time before the last sweep
  bool conv = false;
  int sweep = 0;
  while (sweep < a.v.max_inner && !conv) {
    const int f = sweep % 3;
    bool ch = false;
    int nq = 1;
    if constexpr (DIM == 2) {
      ch = tri_sweep<N>(r, sT, large, eps, solves);
    } else {
      tet_select<N, BT, CAP>(r, d.nelem, sT, sQ, a.max_queue, &sQn[sweep & 1], &sFlag[f], &sFull,
                             sweep + 1);
      __syncthreads();
      nq = sQn[sweep & 1];
      if (CAP) nq = min(nq, a.max_queue);
      if (tid == 0) sQn[(sweep & 1) ^ 1] = 0;
      if (nq) ch = tet_solve<N, BT>(r, sA, sB, sQ, nq, sT, large, eps, solves);
    }
    if (ch) sFlag[f] = 1;
    wait_memory();
    __syncthreads();
    conv = !sFlag[f];
    if (tid == 0) sFlag[(f + 2) % 3] = 0;
    ++sweep;
    if (!conv && sweep < a.v.max_inner) {
      if (tid < d.nown) last = sT[tid];
      if constexpr (DIM == 2) __syncthreads();  // (read before the next sweep lowers it)
    }
  }
  const unsigned long long t2 = wall_clock64();
  // What this visit evaluated the block's elements with: every time, but for the owned vertices that
  // fell in the last sweep of a visit cut off by the sweep cap; after a full queue, nothing.
  const bool full = DIM == 3 && CAP && !conv && sFull == sweep;
  if (tid < d.nown) {
    const float v = sT[tid];
    seen[tid] = full ? EIK_INF : conv ? v : last;
    if (v < own) {
      T[d.vstart + tid] = v;
      if (tid >= d.nbnd0) sBnd = 1;
    }
  }
  for (int i = tid; i < d.nhalo; i += BT) seen[d.nown + i] = full ? EIK_INF : sT[d.nown + i];
  __syncthreads();
  sync_end(a, b, d, sBnd != 0, conv, sT);
  VisitResult vr;
  vr.t_load = t1 - t0;
  vr.t_sweep = t2 - t1;
  vr.t_wb = wall_clock64() - t2;
  block_counters(a.acc, d, sweep, solves, a.elem_bytes, wall_clock64() - t0, vr, &sRed);
}

static dim3 seed_grid(int64_t nseeds) {
  return dim3((unsigned)std::min<int64_t>(nseeds, 1 << 16));
}

struct SolveArgs {
  VisitArgs v;
  Sched s;
  TriItems items;      // triangles
  const int32_t* dep_start;
  const int32_t* dep;
  const int32_t* iperm;
  float* out;          // the times in caller order, written at the end of the launch (or null)
  unsigned long long* told;  // pinned host memory: the last one copies the counters here (or null)
  int64_t nv;
  unsigned long long* counters;
  int64_t max_visits;  // runaway guard: visits of one workgroup after which it marks nothing
  int32_t elem_bytes;  // algorithmic bytes per element (visit_algo_bytes)
  int32_t max_local;   // LDS strides: local vertices and elements of the largest block
  int32_t max_elem;
  int32_t max_queue;
  float height_unit;     // tets (BlockData)
  size_t rec_lds_bytes;  // k_visit_general: staged records
};

// The end of a workgroup: its tally, and, if it is the last one, the sums to the host, with the ticks at
// which the solve and its visits began and this one.
__device__ __forceinline__ void finish(const SolveArgs& a, const unsigned long long* acc) {
  if (threadIdx.x < kNumCounters && acc[threadIdx.x])
    atomicAdd(&a.counters[threadIdx.x], acc[threadIdx.x]);
  if (!a.told || threadIdx.x >= 64) return;
  wait_memory();
  unsigned before = 0;
  // (workgroups that have finished: a control word of its own line)
  if (threadIdx.x == 0) before = atomicAdd(reinterpret_cast<unsigned*>(a.s.ctl) + kSchedCtlBytes / 16, 1u);
  if (__builtin_amdgcn_readfirstlane(before) + 1u != gridDim.x) return;
  if (threadIdx.x <= kNumCounters)
    __hip_atomic_store(&a.told[threadIdx.x], load_word(&a.counters[threadIdx.x]), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_SYSTEM);
  if (threadIdx.x == 0) a.told[kNumCounters + 2] = wall_clock64();
}

// The start of the visit launch (the fill before it left its own behind the counters).
__device__ __forceinline__ void begin(const SolveArgs& a) {
  if (a.told && blockIdx.x == 0 && threadIdx.x == 0) a.told[kNumCounters + 1] = wall_clock64();
}

struct SingleBlocks {
  static constexpr bool kSingle = true;
  const SolveArgs& a;
  __device__ __forceinline__ BlockData operator()(int32_t b) const {
    return {a.v.blocks, a.v.elems, a.v.halo, a.v.T,   a.v.seen, a.v.vmask,
            a.dep_start, a.dep,    nullptr,  a.height_unit, a.items, b, 0};
  }
};

template <int DIM, int N, int BT, bool CAP = false>
__global__ __launch_bounds__(BT) __attribute__((amdgpu_waves_per_eu(4))) void k_visit_resident(SolveArgs a) {
  extern __shared__ uint4 lds4[];
  __shared__ LoopShared sh;
  if (threadIdx.x < kNumCounters) sh.acc[threadIdx.x] = 0;
  begin(a);
  const LoopArgs la = {a.s, a.v.eps, a.v.max_inner, a.max_visits, a.max_local, a.max_elem, a.max_queue};
  const int end = resident_loop<DIM, N, BT, CAP>(la, SingleBlocks{a}, blockIdx.x, lds4, sh);
  write_times(a.s, end, a.v.T, a.iperm, a.nv, a.out, &sh.block);
  finish(a, sh.acc);
}

// Seeds of a solve of the scheduler above: the sources' times, and the owner block of each source
// and that block's dependents marked (one workgroup per source, one lane per block to mark).
__global__ void k_sched_seed(Sched s, const int32_t* seeds, const float* vals, int64_t n,
                             const int32_t* iperm, const int32_t* owner, const int32_t* dep_start,
                             const int32_t* dep, float* T, int64_t nv) {
  for (int64_t i = blockIdx.x; i < n; i += gridDim.x) {
    if (seeds[i] < 0 || seeds[i] >= nv) continue;
    const int32_t v = iperm[seeds[i]];
    const int32_t b = owner[v];
    if (threadIdx.x == 0)
      atomicMin(reinterpret_cast<unsigned*>(&T[v]), seed_key(vals, i));
    const int32_t s0 = dep_start[b], nd = dep_start[b + 1] - s0;
    for (int j = threadIdx.x; j <= nd; j += blockDim.x)
      sched_mark(s, sched_slot(s, j == 0 ? b : dep[s0 + j - 1]), seed_key(vals, i));
  }
}

// The persistent kernel over blocks of any size: the records staged in LDS or read from memory,
// the selected pairs through the LDS queue (visit_block).  Scheduling as in k_visit_resident.
template <int DIM>
__global__ __launch_bounds__(kBlockThreads) __attribute__((amdgpu_waves_per_eu(3))) void k_visit_general(SolveArgs a) {
  extern __shared__ uint4 lds4[];
  __shared__ int sFlag[4];
  __shared__ int sQn[2];  // work-item counters of alternate chunks
  __shared__ int sBlock;
  __shared__ unsigned sKey;  // smallest time the visit lowered
  __shared__ int sCrowd;     // dirty blocks seen waiting when this one was claimed
  __shared__ unsigned long long sRed;
  __shared__ unsigned long long sAcc[kNumCounters];
  const int tid = threadIdx.x;
  begin(a);
  if (tid < kNumCounters) sAcc[tid] = 0;
  Finder f;
  if (tid < 64) sched_enter(a.s, f, blockIdx.x);
  for (;;) {
    if (tid < 64) {
      const int32_t nb = find_next<false>(a.s, f, sAcc);
      if (tid == 0) {
        sBlock = nb;
        sCrowd = f.others;
      }
    }
    __syncthreads();
    const int b = __builtin_amdgcn_readfirstlane(sBlock);
    if (b < 0) break;
    const BlockDesc d = a.v.blocks[b];
    const VisitLds l = carve_lds<DIM>(lds4, a.rec_lds_bytes, a.v.queue_cap, d);
    const uint32_t slot = sched_slot(a.s, b);
    const int32_t s0 = a.dep_start[b];
    const int ndep = a.dep_start[b + 1] - s0;
    bool rerun = false;  // the previous visit of this workgroup was of block b, and this one's
                         // times are in LDS already (rerun_load)
    // few blocks wait: one sweep of a tet block per visit (see kCrowd; 1 / 3 / 8 times as many here, records
    // from memory: 64^3 cube 1.04 / 1.04 / 1.05 ms, at 192 vertices per block 1.32 / 1.29 / 1.32, 96^3 with 16
    // sources 2.95 / 3.01 / 3.30)
    const int inner = DIM == 3 && sCrowd < 3 * kCrowd ? 1 : 0;
    for (;;) {
      if (tid == 0) {
        sRed = 0;
        sKey = kClean;
      }
      const unsigned long long t0 = wall_clock64();
      uint64_t solves = 0;
      const VisitResult r =
          visit_block<DIM, true>(a.v, b, l.rec, l.T, l.old, l.chg, l.hidx, l.vm, l.q, l.mark, sFlag,
                                 sQn, &solves, rerun, inner, rerun);
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) solves += __shfl_down(solves, off, 64);
      if (__lane_id() == 0) atomicAdd(&sRed, (unsigned long long)solves);
      uint32_t key = kClean;
      for (int i = tid; i < d.nown; i += kBlockThreads)
        if (l.T[i] < l.old[i]) key = min(key, __float_as_uint(l.T[i]));
      key = wave_umin(key);
      if (__lane_id() == 0 && key != kClean) atomicMin(&sKey, key);
      // visits beyond the bound mark nothing more (runaway guard)
      const bool again = !r.converged && (int64_t)sAcc[0] < a.max_visits;
      // (marks made meanwhile stay: clearing them here would cost every visit a round trip, and the
      // block a further visit at the end where there were any)
      __syncthreads();
      const unsigned long long tq = wall_clock64();
      if (tid < 64) {
        // the visit's times have reached the device's coherence point (visit_block)
        const uint64_t mask = a.v.vmask ? ((uint64_t)(uint32_t)l.mark[0] |
                                           ((uint64_t)(uint32_t)l.mark[1] << 32))
                                        : 0ull;
        if (r.bnd_changed && (int64_t)sAcc[0] < a.max_visits)
          for (int j = tid; j < ndep; j += 64)
            if (a.v.vmask ? ((mask >> j) & 1ull) != 0ull : l.mark[j] != 0)
              sched_mark(a.s, sched_slot(a.s, a.dep[s0 + j]), sKey);
        if (again) {
          // the next visit starts with clear marks (they have all been read above)
          if (a.v.vmask) {
            if (tid < 2) l.mark[tid] = 0;
          } else {
            for (int j = tid; j < ndep; j += 64) l.mark[j] = 0;
          }
        } else {
          wait_memory();  // the marks have landed before this block can count as clean
          if (tid == 0) sched_leave(a.s, slot, kClean);
        }
        if (tid == 0) {
          tally_visit(sAcc, d, r, sRed, a.elem_bytes, tq - t0, rerun, rerun && a.v.rec_lds);
          sAcc[10] += wall_clock64() - tq;
        }
      } else if (again) {
        rerun_load<true, kBlockThreads>(a.v, d, r.sweeps, l.T, l.old, l.chg, l.hidx, sFlag, 64);
      }
      __syncthreads();
      if (!again) break;
      rerun = true;
    }
  }
  write_times(a.s, __builtin_amdgcn_readfirstlane(sBlock), a.v.T, a.iperm, a.nv, a.out, &sBlock);
  finish(a, sAcc);
}

// The items of every triangle block (TriItems) from its records: one workgroup per block, items in
// record order.  mask: the record's updatable corners; corners not owned have no item.
__global__ __launch_bounds__(256) void k_tri_items(const BlockDesc* blocks, const uint4* recs,
                                                   const int2* range, uint32_t* id, float4* len,
                                                   uint16_t* rec) {
  __shared__ int sWave[4];
  const BlockDesc d = blocks[blockIdx.x];
  int at = range[blockIdx.x].x;
  for (int e0 = 0; e0 < d.nelem; e0 += 256) {
    const int e = e0 + (int)threadIdx.x;
    const Elem x = load_elem<2>(recs, d.estart + (e < d.nelem ? e : 0));
    unsigned m = e < d.nelem ? x.mask & 7u : 0u;
    if (x.v0 >= d.nown) m &= ~1u;
    if (x.v1 >= d.nown) m &= ~2u;
    if (x.v2 >= d.nown) m &= ~4u;
    const int n = __popc(m), end = wave_scan(n);
    if (__lane_id() == 63) sWave[threadIdx.x >> 6] = end;
    __syncthreads();
    int q = at + end - n, total = 0;
    for (int w = 0; w < 4; ++w) {
      if (w < (int)(threadIdx.x >> 6)) q += sWave[w];
      total += sWave[w];
    }
    // the corner order and lengths of tri_rotation
    if (m & 1u) {
      id[q] = x.v1 | (x.v2 << kItemSlotBits) | ((uint32_t)x.v0 << (2 * kItemSlotBits));
      rec[q] = (uint16_t)e;
      len[q++] = make_float4(x.L0, x.L2, x.L1, x.H0);
    }
    if (m & 2u) {
      id[q] = x.v0 | (x.v2 << kItemSlotBits) | ((uint32_t)x.v1 << (2 * kItemSlotBits));
      rec[q] = (uint16_t)e;
      len[q++] = make_float4(x.L0, x.L1, x.L2, x.H1);
    }
    if (m & 4u) {
      id[q] = x.v0 | (x.v1 << kItemSlotBits) | ((uint32_t)x.v2 << (2 * kItemSlotBits));
      rec[q] = (uint16_t)e;
      len[q++] = make_float4(x.L2, x.L1, x.L0, x.H2);
    }
    at += total;
    __syncthreads();
  }
}

// T_out[caller id] = T[new id]
__global__ void k_gather(const float* T, const int32_t* iperm, int64_t nv, float* out) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nv) out[i] = T[iperm[i]];
}

// Local-solver test kernel: one thread per element, every corner.
template <int DIM>
__global__ void k_debug_local(const float* T, const float* L, int64_t n, float* out, float large) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  if constexpr (DIM == 3) {
    const float t0 = T[4 * i], t1 = T[4 * i + 1], t2 = T[4 * i + 2], t3 = T[4 * i + 3];
    const float* l = L + 6 * i;
    const float L0 = l[0], L1 = l[1], L2 = l[2], L3 = l[3], L4 = l[4], L5 = l[5];
    out[4 * i + 0] = __builtin_fminf(t0, tet_rotation(0, t0, t1, t2, t3, L0, L1, L2, L3, L4, L5, large));
    out[4 * i + 1] = __builtin_fminf(t1, tet_rotation(1, t0, t1, t2, t3, L0, L1, L2, L3, L4, L5, large));
    out[4 * i + 2] = __builtin_fminf(t2, tet_rotation(2, t0, t1, t2, t3, L0, L1, L2, L3, L4, L5, large));
    out[4 * i + 3] = __builtin_fminf(t3, tet_rotation(3, t0, t1, t2, t3, L0, L1, L2, L3, L4, L5, large));
  } else {
    const float t0 = T[3 * i], t1 = T[3 * i + 1], t2 = T[3 * i + 2];
    const float L0 = L[3 * i], L1 = L[3 * i + 1], L2 = L[3 * i + 2];
    out[3 * i + 0] = __builtin_fminf(t0, tri_rotation(0, t0, t1, t2, L0, L1, L2, large));
    out[3 * i + 1] = __builtin_fminf(t1, tri_rotation(1, t0, t1, t2, L0, L1, L2, large));
    out[3 * i + 2] = __builtin_fminf(t2, tri_rotation(2, t0, t1, t2, L0, L1, L2, large));
  }
}

// ------------------------------------------------------------------------------------------
// Host orchestration
// ------------------------------------------------------------------------------------------
size_t visit_lds_bytes(const Layout& L, int dim, int32_t queue_cap, size_t rec_bytes) {
  // records; times, stamps and halo indices of the local vertices; owned times at the start and
  // (triangles) the owned vertices' dependent masks
  return rec_bytes + sizeof(float) * ((size_t)L.max_local * 3 + L.max_own) +
         (dim == 2 ? sizeof(uint64_t) * ((size_t)L.max_own + 1) : 0) +
         sizeof(uint16_t) * (((size_t)queue_cap + 1) & ~(size_t)1) +
         sizeof(int32_t) * std::max<size_t>(L.max_dep, 2);
}

static int setup_resident(Mesh& m, size_t max_lds);

int upload_layout(Mesh& m) {
  int rc = ensure_stream(m);
  if (rc) return rc;
  if (!m.layout.valid) {
    rc = build_layout(m);
    if (rc) return rc;
  }
  if (!m.device_dirty && m.dev->blocks) return EIK_OK;
  DeviceState* old = m.dev;
  // keep the stream and events, drop the buffers
  DeviceState* d = new DeviceState();
  d->device = old->device;
  d->stream = old->stream;
  d->ev0 = old->ev0;
  d->ev1 = old->ev1;
  d->evA = old->evA;
  d->evB = old->evB;
  old->stream = nullptr;
  old->ev0 = old->ev1 = old->evA = old->evB = nullptr;
  dev_free(old);
  m.dev = d;
  const Layout& L = m.layout;
  hipStream_t s = d->stream;
  d->dim = m.dim;
  d->nblocks = L.nblocks;
  d->nv = m.nv;
  // work queue: all (element, corner) pairs of the largest block if that fits, else chunks of
  // 2048; element records are staged in LDS when the whole visit fits the per-workgroup LDS
  int max_lds = 65536;
  {
    int v = 0;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, d->device) ==
            hipSuccess && v > 0)
      max_lds = v - 1024;  // static shared variables of the kernels
  }
  const int K = m.dim == 3 ? 4 : 3;
  const size_t rb = m.dim == 3 ? sizeof(TetRec) : sizeof(TriRec);
  int32_t qcap = std::min(8192, std::max(256, K * L.max_elem));
  size_t rec_bytes = ((size_t)L.max_elem * rb + 15) & ~(size_t)15;
  size_t lds = visit_lds_bytes(L, m.dim, qcap, rec_bytes);
  d->rec_lds = 1;
  if (lds > (size_t)max_lds) {
    d->rec_lds = 0;
    rec_bytes = 0;
    qcap = std::min(qcap, 2048);
    lds = visit_lds_bytes(L, m.dim, qcap, 0);
  }
  if (lds > (size_t)max_lds)
    return fail(EIK_ERR_CAPACITY, "block too large for LDS staging (" + std::to_string(L.max_local) +
                                      " local vertices); use fewer vertices per block");
  if (lds > 65536) {
    // dynamic LDS beyond 64 KB (MI355X has 160 KB per CU) is opted into per kernel
    const void* ks[] = {(const void*)k_visit_sync<3>, (const void*)k_visit_sync<2>,
                        (const void*)k_visit_general<3>, (const void*)k_visit_general<2>};
    for (const void* k : ks)
      HIP_TRY(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  }
  d->lds_bytes = lds;
  d->lds_bytes_direct = visit_lds_bytes(L, m.dim, qcap, 0);
  d->rec_lds_bytes = rec_bytes;
  d->queue_cap = qcap;
  if ((rc = upload(&d->blocks, L.blocks, s))) return rc;
  if (m.dim == 3) {
    if ((rc = upload(reinterpret_cast<TetRec**>(&d->elems), L.tets, s))) return rc;
  } else {
    if ((rc = upload(reinterpret_cast<TriRec**>(&d->elems), L.tris, s))) return rc;
  }
  if ((rc = upload(&d->halo, L.halo, s))) return rc;
  if ((rc = upload(&d->iperm, L.iperm, s))) return rc;
  if ((rc = upload(&d->dep_start, L.dep_start, s))) return rc;
  if ((rc = upload(&d->dep, L.dep, s))) return rc;
  if ((rc = upload(&d->owner, L.owner, s))) return rc;
  if ((rc = upload(&d->vh_start, L.vh_start, s))) return rc;
  if ((rc = upload(&d->vh_pos, L.vh_pos, s))) return rc;
  if (!L.vmask.empty())
    if ((rc = upload(&d->vmask, L.vmask, s))) return rc;
  if ((rc = upload(&d->rec_elem, L.rec_elem, s))) return rc;
  HIP_TRY(hipMalloc((void**)&d->T, sizeof(float) * m.nv));
  HIP_TRY(hipMalloc((void**)&d->out, sizeof(float) * m.nv));
  d->nseen = m.nv + (int64_t)L.halo.size();
  HIP_TRY(hipMalloc((void**)&d->seen, sizeof(float) * d->nseen));
  HIP_TRY(hipMalloc((void**)&d->stamp[0], sizeof(int32_t) * L.nblocks));
  HIP_TRY(hipMalloc((void**)&d->stamp[1], sizeof(int32_t) * L.nblocks));
  HIP_TRY(hipMalloc((void**)&d->list[0], sizeof(int32_t) * L.nblocks));
  HIP_TRY(hipMalloc((void**)&d->list[1], sizeof(int32_t) * L.nblocks));
  HIP_TRY(hipMalloc((void**)&d->count, sizeof(int32_t) * 4));
  HIP_TRY(hipMalloc((void**)&d->counters, sizeof(unsigned long long) * (kNumCounters + 1)));
  HIP_TRY(hipMalloc((void**)&d->sync_acc, sizeof(unsigned long long) * kSyncSlots * kSyncSlotWords));
  HIP_TRY(hipStreamSynchronize(s));
  rc = setup_resident(m, (size_t)max_lds);
  if (rc) return rc;
  m.device_dirty = false;
  return EIK_OK;
}

struct ResidentKernels {
  const void* loop;  // k_visit_resident
  const void* sync;  // k_visit_sync_resident
};
template <int DIM, int N, int BT, bool CAP = false>
static ResidentKernels resident_pair() {
  return {(const void*)k_visit_resident<DIM, N, BT, CAP>, (const void*)k_visit_sync_resident<DIM, N, BT, CAP>};
}
static ResidentKernels resident_kernels(const DeviceState* d) {
  const int n = d->res_n, bt = d->res_bt;
  if (d->dim == 3)
    return n == 2                   ? resident_pair<3, 2, 512>()
           : n == 4 && bt == 256    ? resident_pair<3, 4, 256>()
           : bt == 256              ? resident_pair<3, kTetN<256>, 256>()
           : bt == 512 && d->res_cap ? resident_pair<3, kTetN<512>, 512, true>()
           : bt == 512              ? resident_pair<3, kTetN<512>, 512>()
                                    : resident_pair<3, kTetN<1024>, 1024>();
  return bt == 256    ? resident_pair<2, 1, 256>()
         : bt == 1024 ? resident_pair<2, 4, 1024>()
         : n == 1     ? resident_pair<2, 1, 512>()
         : n == 2     ? resident_pair<2, 2, 512>()
                      : resident_pair<2, 4, 512>();
}

// The shape of the register-resident visits for this layout, and the triangle items.  A block
// qualifies when one thread can hold each owned vertex and N x BT items (triangles) or elements
// (tets) cover it.  The shapes go from the smallest: few items per thread make the chain of a sweep
// short (64-vertex triangle blocks, 1 per thread of 512 / 2 per thread of 256: level-7 anisotropic
// icosphere 0.49 / 0.56 ms, level 8 1.56 / 1.67, 32^2 square 0.065 / 0.078; 301^2 square with
// obtuse angles, up to 700 items, 2 of 512 / 4 of 256: 0.33 / 0.50).  A tet block keeps 40 KB and a CU
// holds four of 256 threads or two of 512, so the wider workgroup is for meshes whose blocks it holds
// all at once (16^3 cube 0.149 against 0.164 ms, 64^3 0.775 against 0.653).
static int setup_resident(Mesh& m, size_t max_lds) {
  DeviceState* d = m.dev;
  const Layout& L = m.layout;
  d->max_local = L.max_local;
  d->max_elem = L.max_elem;
  d->height_unit = L.height_unit;
  d->res_n = 0;
  if (L.vmask.empty()) return EIK_OK;
  int dev = 0, ncu = 0;
  HIP_TRY(hipGetDevice(&dev));
  HIP_TRY(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
  const int32_t need = m.dim == 3 ? L.max_elem : L.max_items;
  static const int shapes[2][5][2] = {
      {{1, 256}, {1, 512}, {2, 512}, {4, 512}, {4, 1024}},
      {{2, 512}, {4, 256}, {kTetN<256>, 256}, {kTetN<512>, 512}, {kTetN<1024>, 1024}}};
  for (int i = m.dim == 3 && L.nblocks > 2 * ncu ? 1 : 0; i < 5 && d->res_n == 0; ++i) {
    const int* sh = shapes[m.dim == 3 ? 1 : 0][i];
    if (need <= sh[0] * sh[1] && L.max_own <= sh[1]) d->res_n = sh[0], d->res_bt = sh[1];
  }
  if (d->res_n == 0) return EIK_OK;
  if (m.dim == 2 && L.max_local > kItemSlots) {
    d->res_n = 0;
    return EIK_OK;
  }
  d->max_queue = loop_queue(m.dim, d->res_bt, L.max_local, L.max_elem, L.max_items);
  d->res_cap = m.dim == 3 && d->max_queue < L.max_items;
  d->res_lds = loop_lds_bytes(m.dim, L.max_local, L.max_elem, d->max_queue);
  if (d->res_lds > max_lds) {
    d->res_n = 0;
    return EIK_OK;
  }
  if (d->res_lds > 65536)
    for (const void* k : {resident_kernels(d).loop, resident_kernels(d).sync})
      HIP_TRY(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)d->res_lds));
  if (m.dim == 3) return EIK_OK;
  std::vector<int2> range(L.nblocks);
  int64_t n = 0;
  for (int32_t b = 0; b < L.nblocks; ++b) {
    range[b] = make_int2((int)n, L.items[b]);
    n += L.items[b];
  }
  if (n >= INT32_MAX) {
    d->res_n = 0;
    return EIK_OK;
  }
  int rc = upload(&d->item_range, range, d->stream);
  if (rc) return rc;
  HIP_TRY(hipMalloc((void**)&d->item_id, sizeof(uint32_t) * std::max<int64_t>(n, 1)));
  HIP_TRY(hipMalloc((void**)&d->item_len, sizeof(float4) * std::max<int64_t>(n, 1)));
  HIP_TRY(hipMalloc((void**)&d->item_rec, sizeof(uint16_t) * std::max<int64_t>(n, 1)));
  hipLaunchKernelGGL(k_tri_items, dim3(L.nblocks), dim3(256), 0, d->stream, d->blocks,
                     (const uint4*)d->elems, d->item_range, d->item_id, d->item_len,
                     d->item_rec);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(d->stream));  // the host copy of the ranges has been read
  return EIK_OK;
}

// Iterations enqueued beyond the one that has begun last.  The device tells the host which that is
// (SyncArgs::told), so that the stream does not run empty while the host waits to learn whether there is
// another (the reference copies block flags back and forth and synchronises several times per
// iteration, meshFIM3dEikonal.cu:431-531; a wait for every eight iterations left the device idle for 35
// us each).  Iterations enqueued after convergence find no active block and cost one near-empty launch each.
constexpr int kSyncAhead = 5;

// Waits until an iteration has begun.  (The stream is asked only after a while: the question puts a
// marker into it, which costs the device 6 us.)
static int sync_wait(const unsigned long long* told, int64_t it, hipStream_t s) {
  auto begun = [&] { return (int64_t)(uint32_t)__atomic_load_n(told, __ATOMIC_ACQUIRE) >= it; };
  for (;;) {
    const auto t0 = std::chrono::steady_clock::now();
    do {
      for (int spin = 0; spin < 256; ++spin)
        if (begun()) return EIK_OK;
    } while (std::chrono::steady_clock::now() - t0 < std::chrono::milliseconds(20));
    const hipError_t e = hipStreamQuery(s);
    if (e == hipErrorNotReady) continue;
    HIP_TRY(e);
    return begun() ? EIK_OK : fail(EIK_ERR_HIP, "an iteration ended without a sign");
  }
}

static int solve_sync(Mesh& m, const eik_solve_opts_t& o) {
  DeviceState* d = m.dev;
  hipStream_t s = d->stream;
  const int32_t nb = d->nblocks;
  const float large = m.dim == 3 ? EIK_LARGENUM_3D : EIK_LARGENUM_2D;
  // d->count (cleared with the solve's other arrays): the active counts of iterations modulo 3, the
  // last iteration that visited a block
  int32_t* cnt = d->count;
  unsigned long long* told = d->h_cnt + kNumCounters;
  __atomic_store_n(told, 0ull, __ATOMIC_RELEASE);
  SyncArgs a;
  a.snap = nullptr;
  a.v.blocks = d->blocks;
  a.v.elems = d->elems;
  a.v.halo = d->halo;
  a.v.T = d->T;
  a.v.large = large;
  a.v.eps = o.eps;
  a.v.max_inner = default_inner_sweeps(m.dim, o.max_inner);
  a.v.queue_cap = d->queue_cap;
  a.v.seen = d->seen;
  // Every block of an iteration is visited at once, so this kernel is throughput-bound: records
  // read from memory (smaller workgroups, more per CU) were never slower than staged ones and
  // up to 21% faster (96^3 cube 7.53 -> 5.91 ms, 64^3 2.42 -> 2.06, level-7 icospheres 8%);
  // AUTO reads them from memory.
  const bool stage = d->rec_lds && o.stage_records == EIK_STAGE_LDS;
  const size_t lds = stage ? d->lds_bytes : d->lds_bytes_direct;
  a.v.rec_lds = stage ? 1 : 0;
  a.v.vh_start = nullptr;  // the per-iteration activation works on block stamps
  a.v.vh_pos = nullptr;
  a.v.vmask = nullptr;
  a.v.rmult = nullptr;
  a.v.lens = nullptr;
  a.v.dep_start = d->dep_start;
  a.rec_lds_bytes = stage ? d->rec_lds_bytes : 0;
  a.acc = d->sync_acc;
  a.elem_bytes = m.dim == 3 ? kAlgoElemBytes<3> : kAlgoElemBytes<2>;
  a.last = cnt + 3;
  a.told = told;
  a.dep = d->dep;
  a.items = {d->item_range, d->item_id, d->item_len, d->item_rec};
  a.max_local = d->max_local;
  a.max_elem = d->max_elem;
  a.max_queue = d->max_queue;
  a.height_unit = d->height_unit;
  a.nb = nb;
  // values only decrease, so the loop ends; the cap bounds it on pathological inputs
  const int64_t cap = o.max_iterations > 0 ? o.max_iterations : 1000000;
  int64_t it = 0;
  const bool resident = d->res_n != 0 && o.stage_records == EIK_STAGE_AUTO;
  void* args[] = {(void*)&a};
  HIP_TRY(hipEventRecord(d->evA, s));
  while (it < cap) {
    if (it >= kSyncAhead) {
      int rc = sync_wait(told, it + 1 - kSyncAhead, s);
      if (rc) return rc;
    }
    const unsigned long long t = __atomic_load_n(told, __ATOMIC_ACQUIRE);
    if ((t >> 32) < (uint32_t)t) break;  // an iteration without an active block has begun
    ++it;
    a.now = {d->stamp[it & 1], d->list[it & 1], cnt + it % 3};
    a.next = {d->stamp[~it & 1], d->list[~it & 1], cnt + (it + 1) % 3};
    a.count_after = cnt + (it + 2) % 3;
    a.it = (int32_t)it;
    unsigned snap_wgs = 0;
    if (o.record_history) {
      const size_t slot = (size_t)(it - 1);
      while (d->hist.size() <= slot / kHistChunk) {
        float* c = nullptr;
        HIP_TRY(hipMalloc((void**)&c, sizeof(float) * kHistChunk * (size_t)m.nv));
        d->hist.push_back(c);
      }
      a.snap = d->hist[slot / kHistChunk] + (slot % kHistChunk) * (size_t)m.nv;
      snap_wgs = (unsigned)grid1d(nb, kSnapBlocks);
    }
    const dim3 grid((unsigned)nb + snap_wgs);
    if (resident)
      HIP_TRY(hipLaunchKernel(resident_kernels(d).sync, grid, dim3(d->res_bt), args, d->res_lds, s));
    else if (m.dim == 3)
      hipLaunchKernelGGL(k_visit_sync<3>, grid, dim3(kBlockThreads), lds, s, a);
    else
      hipLaunchKernelGGL(k_visit_sync<2>, grid, dim3(kBlockThreads), lds, s, a);
    HIP_TRY(hipGetLastError());
  }
  HIP_TRY(hipEventRecord(d->evB, s));
  hipLaunchKernelGGL(k_sum_slots, dim3(1), dim3(64), 0, s, d->sync_acc, d->counters);
  HIP_TRY(hipGetLastError());
  return EIK_OK;
}

// The visit kernel of the persistent single solve.
struct VisitKernel {
  const void* fn;
  int threads;
  size_t lds;
  bool stage;  // k_visit_general: records staged in LDS
};

// Register-resident visits where the blocks fit them, unless the caller asks for staged records or for
// records read from memory; else the general kernel, its records staged in LDS where they fit.
static VisitKernel visit_kernel(const DeviceState* d, int32_t stage_records) {
  VisitKernel k;
  k.stage = d->rec_lds && stage_records != EIK_STAGE_MEMORY;
  if (d->res_n && stage_records == EIK_STAGE_AUTO) {
    k.threads = d->res_bt;
    k.lds = d->res_lds;
    k.fn = resident_kernels(d).loop;
    return k;
  }
  k.threads = kBlockThreads;
  k.lds = k.stage ? d->lds_bytes : d->lds_bytes_direct;
  k.fn = d->dim == 3 ? (const void*)k_visit_general<3> : (const void*)k_visit_general<2>;
  return k;
}

// Workgroups of the single-solve persistent kernel: one per block while they all fit, so that every
// block stays resident with its owner, else all that fit (64^3 cube, 4,292 blocks: 1.29 ms at 256,
// 0.81 at 512, 0.66 at 768, 0.63 at 1,024; level-8 icosphere, 10,240 blocks of 512 threads: 2.10 at 256,
// 1.73 at 384, 1.57 at 512).  Where a triangle mesh has more blocks than fit and they take 256 threads, of
// which a CU holds more than are of use, the grid is sized to the fronts, which are curves: six workgroups
// per block of a front of sqrt(blocks x sources) blocks, one to three per CU.  Beyond that, workgroups visit
// blocks whose suppliers are still changing, and poll (in registers, 768 workgroups / this rule: level-5
// icosphere at 8 vertices per block 0.56 / 0.27 ms, level 6 at 32 0.60 / 0.34, level 7 at 32 0.79 / 0.73,
// level 8 at 32 1.69 / 1.69; general kernel, records from memory, level 7 with 4 sources at 128 1.93 / 1.65,
// level 7 at 200 1.50 / 1.18).  The other triangle shapes, two to a CU, take all that fit (level 7 with one
// source at 303 / 512: 0.72 / 0.68).
static int persistent_grid(int dim, const VisitKernel& k, int requested, int64_t nblocks, int64_t nseeds,
                           int* out) {
  int dev = 0, ncu = 0, per_cu = 0;
  HIP_TRY(hipGetDevice(&dev));
  HIP_TRY(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
  HIP_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k.fn, k.threads, k.lds));
  int resident = std::max(1, ncu * std::max(per_cu, 1));
  resident = std::min(resident, 64 * ncu);
  if (requested > 0) {
    *out = std::min(requested, resident);
    return EIK_OK;
  }
  int most = dim == 2 ? std::min(resident, 3 * ncu) : resident;
  if (dim == 2 && k.threads == kBlockThreads && nblocks > most) {
    const double front = 6.0 * std::sqrt((double)nblocks * (double)std::max<int64_t>(nseeds, 1));
    most = (int)std::min<double>(most, std::max<double>(ncu, front));
  }
  *out = (int)std::min<int64_t>(most, std::max<int64_t>(nblocks, 1));
  return EIK_OK;
}

// Inner sweeps per visit of the single-solve persistent kernel when the caller leaves the choice: 3 for
// triangles (visits at 2 / 3 / 4 / 5 sweeps, in registers: level-5 icosphere 176 / 167 / 170 / 172 us, level 7
// with 4 sources 476 / 467 / 483 / 503, level 8 1,719 / 1,719 / 1,742 / 1,782; general kernel, level 7 1,063 /
// 1,034 / 1,036 / 1,106); other schedulers and launches keep default_inner_sweeps.
static int32_t async_inner_sweeps(int dim, int32_t requested) {
  return requested > 0 ? requested : (dim == 2 ? 3 : default_inner_sweeps(dim, 0));
}

int check_end(const unsigned char* sctl, hipStream_t s, unsigned long long abandoned) {
  uint32_t done = 0;
  HIP_TRY(hipMemcpyAsync(&done, sctl + kSchedCtlBytes / 2, sizeof(done), hipMemcpyDeviceToHost, s));
  HIP_TRY(hipStreamSynchronize(s));
  if (done) return EIK_OK;
  return fail(EIK_ERR_TIMEOUT, std::to_string(abandoned) +
                                   " queue waits outlasted wait_limit_us and the solve did not "
                                   "finish (incomplete result)");
}

// The block words of the persistent scheduler, allocated on first use: one per block and, since
// every owner has as many, up to one more per workgroup (at most 64 per CU).
static int ensure_words(DeviceState* d) {
  if (d->words) return EIK_OK;
  int dev = 0, ncu = 0;
  HIP_TRY(hipGetDevice(&dev));
  HIP_TRY(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
  d->max_workgroups = 64 * std::max(ncu, 1);
  HIP_TRY(hipMalloc((void**)&d->words, sizeof(unsigned long long) * sched_max_words(d->nblocks, d->max_workgroups)));
  HIP_TRY(hipMalloc((void**)&d->sctl, kSchedCtlBytes));
  return EIK_OK;
}

// Per-solve device state of the persistent scheduler: the mesh's own buffers (eik_solve) or
// carved from the scratch array (eik_solve_noalloc).
struct AsyncBufs {
  float* T;
  float* seen;
  unsigned long long* words;
  unsigned char* sctl;
  unsigned long long* counters;
};

// Enqueues a persistent solve on stream s: the resets, the seeds, and the visits, which write the
// times in caller order to `out` (device memory, or null) when they are done.  A fill kernel
// rather than memsets, so that a caller may capture this into a graph.
static int enqueue_async(const Mesh& m, const eik_solve_opts_t& o, const AsyncBufs& b,
                         const int32_t* seeds, const float* seedvals, int64_t nseeds, float* out,
                         unsigned long long* told, hipStream_t s) {
  const DeviceState* d = m.dev;
  const VisitKernel k = visit_kernel(d, o.stage_records);
  int grid = 0;
  int rc = persistent_grid(m.dim, k, o.workgroups, d->nblocks, nseeds, &grid);
  if (rc) return rc;
  SolveArgs a;
  a.v.blocks = d->blocks;
  a.v.elems = d->elems;
  a.v.halo = d->halo;
  a.v.T = b.T;
  a.v.large = m.dim == 3 ? EIK_LARGENUM_3D : EIK_LARGENUM_2D;
  a.v.eps = o.eps;
  a.v.max_inner = async_inner_sweeps(m.dim, o.max_inner);
  a.v.queue_cap = d->queue_cap;
  a.v.seen = b.seen;
  a.v.rec_lds = k.stage ? 1 : 0;
  a.v.vh_start = d->vh_start;
  a.v.vh_pos = d->vh_pos;
  a.v.vmask = d->vmask;
  a.v.rmult = nullptr;
  a.v.lens = nullptr;
  a.v.dep_start = d->dep_start;
  a.s.word = b.words;
  a.s.ctl = reinterpret_cast<unsigned long long*>(b.sctl);
  a.s.done = reinterpret_cast<uint32_t*>(b.sctl + kSchedCtlBytes / 2);
  sched_shape(a.s, d->nblocks, grid);
  a.s.wait_limit = wait_limit_ticks(d->device, o.wait_limit_us);
  a.items = {d->item_range, d->item_id, d->item_len, d->item_rec};
  a.dep_start = d->dep_start;
  a.dep = d->dep;
  a.iperm = d->iperm;
  a.out = out;
  a.nv = m.nv;
  a.counters = b.counters;
  a.told = told;
  // runaway guard: a workgroup that has made this many visits marks no more blocks (its visits
  // still finish), so a solve ends even if it never converged; the bound is max_iterations
  // outer iterations' worth of visits of every block (1000 without a cap), far above what a
  // converging solve needs
  a.max_visits = (int64_t)(o.max_iterations > 0 ? o.max_iterations : 1000) * d->nblocks;
  a.elem_bytes = m.dim == 3 ? kAlgoElemBytes<3> : kAlgoElemBytes<2>;
  a.max_local = d->max_local;
  a.max_queue = d->max_queue;
  a.max_elem = d->max_elem;
  a.height_unit = d->height_unit;
  a.rec_lds_bytes = k.stage ? d->rec_lds_bytes : 0;
  FillSegs f;
  f.add(b.T, m.nv, (int32_t)__builtin_bit_cast(uint32_t, a.v.large));
  f.add(b.seen, d->nseen, (int32_t)__builtin_bit_cast(uint32_t, EIK_INF));
  f.add(b.counters, 2 * kNumCounters, 0);
  if (told) f.begin = b.counters + kNumCounters;
  f.words[0] = b.words;
  f.nwords[0] = (int64_t)a.s.owners * a.s.stride;
  f.add(b.sctl, kSchedCtlBytes / 4, 0);
  launch_fill(f, s);
  hipLaunchKernelGGL(k_sched_seed, seed_grid(nseeds), dim3(64), 0, s, a.s, seeds, seedvals, nseeds,
                     d->iperm, d->owner, d->dep_start, d->dep, b.T, m.nv);
  HIP_TRY(hipGetLastError());
  void* args[] = {(void*)&a};
  HIP_TRY(hipLaunchKernel(k.fn, dim3(grid), dim3(k.threads), args, k.lds, s));
  return EIK_OK;
}

}  // namespace eik

using namespace eik;

extern "C" {

void eik_solve_opts_default(eik_solve_opts_t* o) {
  if (!o) return;
  std::memset(o, 0, sizeof(*o));
  o->scheduler = EIK_SCHED_ASYNC;
  o->max_iterations = 0;
  o->max_inner = 0;  // per element kind (default_inner_sweeps)
  o->eps = 0.f;
  o->record_history = 0;
  o->workgroups = 0;
  o->wait_limit_us = 0;  // 10 s
}

int eik_mesh_stream(eik_mesh_t h, void** out) {
  Mesh* m = reinterpret_cast<Mesh*>(h);
  if (!m || !out) return fail(EIK_ERR_ARG, "null argument");
  int rc = ensure_stream(*m);
  if (rc) return rc;
  *out = (void*)m->dev->stream;
  return EIK_OK;
}

int eik_mesh_upload(eik_mesh_t h) {
  Mesh* m = reinterpret_cast<Mesh*>(h);
  if (!m) return fail(EIK_ERR_ARG, "null mesh");
  if (m->nblocks <= 0) return fail(EIK_ERR_STATE, "mesh is not partitioned");
  return upload_layout(*m);
}

int eik_solve(eik_mesh_t h, const int32_t* seeds, int64_t nseeds, const float* seed_vals,
              const eik_solve_opts_t* opts, float* T_out, eik_solve_stats_t* stats) {
  Mesh* m = reinterpret_cast<Mesh*>(h);
  if (!m) return fail(EIK_ERR_ARG, "null mesh");
  if (!seeds || nseeds <= 0) return fail(EIK_ERR_ARG, "at least one seed vertex is required");
  for (int64_t i = 0; i < nseeds; ++i) {
    if (seeds[i] < 0 || seeds[i] >= m->nv) return fail(EIK_ERR_ARG, "seed vertex out of range");
    if (seed_vals && !(seed_vals[i] >= 0.f && seed_vals[i] < 1e30f))
      return fail(EIK_ERR_ARG, "seed values must be finite and >= 0");
  }
  if (m->nblocks <= 0) return fail(EIK_ERR_STATE, "mesh is not partitioned");
  eik_solve_opts_t o;
  eik_solve_opts_default(&o);
  if (opts) o = *opts;
  if (o.scheduler != EIK_SCHED_SYNC && o.scheduler != EIK_SCHED_ASYNC)
    return fail(EIK_ERR_ARG, "unknown scheduler");
  if (o.scheduler == EIK_SCHED_ASYNC && o.record_history)
    return fail(EIK_ERR_ARG, "record_history needs the sync scheduler");
  if (o.wait_limit_us < 0) return fail(EIK_ERR_ARG, "wait_limit_us must be >= 0");
  int rc = upload_layout(*m);
  if (rc) return rc;
  DeviceState* d = m->dev;
  hipStream_t s = d->stream;
  auto t0 = std::chrono::steady_clock::now();
  const float large = m->dim == 3 ? EIK_LARGENUM_3D : EIK_LARGENUM_2D;
  // the times are reset below: until this solve succeeds there is no result to read
  d->has_result = false;
  // the staging buffers may still feed a copy of a solve that ended in an error
  HIP_TRY(hipStreamSynchronize(s));
  if (nseeds > d->seed_cap) {
    if (d->seeds) HIP_TRY(hipFree(d->seeds));
    if (d->seedvals) HIP_TRY(hipFree(d->seedvals));
    if (d->h_seed) HIP_TRY(hipHostFree(d->h_seed));
    d->seeds = nullptr;
    d->seedvals = nullptr;
    d->h_seed = nullptr;
    d->seed_cap = 0;
    HIP_TRY(hipMalloc((void**)&d->seeds, sizeof(int32_t) * nseeds));
    HIP_TRY(hipMalloc((void**)&d->seedvals, sizeof(float) * nseeds));
    HIP_TRY(hipHostMalloc((void**)&d->h_seed, sizeof(int32_t) * 2 * nseeds));
    d->seed_cap = nseeds;
  }
  if (!d->h_cnt) {
    HIP_TRY(hipHostMalloc((void**)&d->h_cnt, sizeof(unsigned long long) * (kNumCounters + 3) +
                                                 sizeof(float) * std::min(m->nv, kSmallOut)));
    d->h_out = reinterpret_cast<float*>(d->h_cnt + kNumCounters + 3);
  }
  d->hist_len = 0;
  int32_t* h_vals = d->h_seed + d->seed_cap;
  std::memcpy(d->h_seed, seeds, sizeof(int32_t) * nseeds);
  if (seed_vals) std::memcpy(h_vals, seed_vals, sizeof(float) * nseeds);
  const bool async = o.scheduler == EIK_SCHED_ASYNC;
  // (the persistent kernel tells its times itself: an event is a packet of its own, 2 us)
  if (!async) HIP_TRY(hipEventRecord(d->ev0, s));
  // a few seeds are read where they are, in pinned memory
  const bool direct_seeds = nseeds <= kDirectSeeds;
  if (!direct_seeds) {
    HIP_TRY(hipMemcpyAsync(d->seeds, d->h_seed, sizeof(int32_t) * nseeds, hipMemcpyHostToDevice, s));
    if (seed_vals)
      HIP_TRY(hipMemcpyAsync(d->seedvals, h_vals, sizeof(float) * nseeds, hipMemcpyHostToDevice, s));
  }
  const int32_t* dev_seeds = direct_seeds ? d->h_seed : d->seeds;
  const float* dev_vals = !seed_vals ? nullptr
                          : direct_seeds ? reinterpret_cast<const float*>(h_vals) : d->seedvals;
  // a small result comes back in the solve's one wait, through pinned memory
  const bool small = T_out && m->nv <= kSmallOut;
  eik_solve_stats_t st;
  std::memset(&st, 0, sizeof(st));
  if (async) {
    if ((rc = ensure_words(d))) return rc;
    const AsyncBufs bufs = {d->T, d->seen, d->words, d->sctl, d->counters};
    rc = enqueue_async(*m, o, bufs, dev_seeds, dev_vals, nseeds,
                       small ? d->h_out : T_out ? d->out : nullptr, d->h_cnt, s);
    if (rc) return rc;
  } else {
    FillSegs f;
    f.add(d->T, m->nv, (int32_t)__builtin_bit_cast(uint32_t, large));
    f.add(d->seen, d->nseen, (int32_t)__builtin_bit_cast(uint32_t, EIK_INF));
    f.add(d->stamp[0], d->nblocks, -1);
    f.add(d->stamp[1], d->nblocks, -1);
    f.add(d->counters, 2 * kNumCounters, 0);
    f.add(d->count, 4, 0);
    f.add(d->sync_acc, 2 * kSyncSlots * kSyncSlotWords, 0);
    launch_fill(f, s);
    hipLaunchKernelGGL(k_sync_seed, seed_grid(nseeds), dim3(64), 0, s, dev_seeds, dev_vals, nseeds, d->iperm, d->owner, d->dep_start,
                       d->dep, d->T, Active{d->stamp[1], d->list[1], d->count + 1});
    HIP_TRY(hipGetLastError());
    if ((rc = solve_sync(*m, o))) return rc;
    if (T_out)
      hipLaunchKernelGGL(k_gather, dim3(grid1d(m->nv, 256)), dim3(256), 0, s, d->T, d->iperm, m->nv,
                         d->out);
  }
  if (!async) {
    HIP_TRY(hipEventRecord(d->ev1, s));
    HIP_TRY(hipMemcpyAsync(d->h_cnt, d->counters, sizeof(unsigned long long) * kNumCounters,
                           hipMemcpyDeviceToHost, s));
    if (small)
      HIP_TRY(hipMemcpyAsync(d->h_out, d->out, sizeof(float) * m->nv, hipMemcpyDeviceToHost, s));
  }
  HIP_TRY(hipStreamSynchronize(s));
  const unsigned long long* cnt = d->h_cnt;
  if (!async) {
    float ms = 0.f, vms = 0.f;
    HIP_TRY(hipEventElapsedTime(&ms, d->ev0, d->ev1));
    HIP_TRY(hipEventElapsedTime(&vms, d->evA, d->evB));
    st.kernel_ms = ms;
    st.visit_ms = vms;
  }
  st.outer_iterations = async ? 1 : (int64_t)(d->h_cnt[kNumCounters] >> 32);
  st.visit_launches = st.outer_iterations;
  if (!async && o.record_history) d->hist_len = (decltype(d->hist_len))st.outer_iterations;
  auto t1 = std::chrono::steady_clock::now();
  st.wall_ms = std::chrono::duration<double, std::milli>(t1 - t0).count();
  st.block_visits = (int64_t)cnt[0];
  st.vertex_updates = (int64_t)cnt[1];
  st.inner_sweeps = (int64_t)cnt[2];
  st.local_solves = (int64_t)cnt[3];
  st.algo_bytes = (int64_t)cnt[4];
  st.algo_bytes_loaded = (int64_t)cnt[kCntAlgoLoaded];
  {
    int khz = 0;
    if (hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, d->device) == hipSuccess &&
        khz > 0) {
      if (async) {
        st.kernel_ms = (double)(cnt[kNumCounters + 2] - cnt[kNumCounters]) / khz;
        st.visit_ms = (double)(cnt[kNumCounters + 2] - cnt[kNumCounters + 1]) / khz;
      }
      st.busy_ms = (double)cnt[5] / khz;
      st.wait_ms = (double)cnt[6] / khz;
      st.load_ms = (double)cnt[7] / khz;
      st.sweep_ms = (double)cnt[8] / khz;
      st.writeback_ms = (double)cnt[9] / khz;
      st.queue_ms = (double)cnt[10] / khz;
    }
  }
  st.reruns = (int64_t)cnt[11];
  st.abandoned_waits = (int64_t)cnt[kCntAbandoned];
  st.history_len = d->hist_len;
  if (st.abandoned_waits > 0) {
    if (stats) *stats = st;
    rc = check_end(d->sctl, s, cnt[kCntAbandoned]);
    if (rc) return rc;
  }
  d->has_result = true;
  if (small) {
    std::memcpy(T_out, d->h_out, sizeof(float) * m->nv);
  } else if (T_out) {
    HIP_TRY(hipMemcpyAsync(T_out, d->out, sizeof(float) * m->nv, hipMemcpyDeviceToHost, s));
    HIP_TRY(hipStreamSynchronize(s));
  }
  if (stats) *stats = st;
  return EIK_OK;
}

int eik_get_result(eik_mesh_t h, float* T_out) {
  Mesh* m = reinterpret_cast<Mesh*>(h);
  if (!m || !T_out) return fail(EIK_ERR_ARG, "null argument");
  if (!m->dev || !m->dev->has_result) return fail(EIK_ERR_STATE, "no completed solve (none has run, or the last one failed)");
  DeviceState* d = m->dev;
  hipLaunchKernelGGL(k_gather, dim3(grid1d(m->nv, 256)), dim3(256), 0, d->stream, d->T, d->iperm,
                     m->nv, d->out);
  HIP_TRY(hipMemcpyAsync(T_out, d->out, sizeof(float) * m->nv, hipMemcpyDeviceToHost, d->stream));
  HIP_TRY(hipStreamSynchronize(d->stream));
  return EIK_OK;
}

int eik_get_history(eik_mesh_t h, int64_t i, float* T_out) {
  Mesh* m = reinterpret_cast<Mesh*>(h);
  if (!m || !T_out) return fail(EIK_ERR_ARG, "null argument");
  DeviceState* d = m->dev;
  if (!d || !d->has_result || i < 0 || i >= d->hist_len)
    return fail(EIK_ERR_ARG, "history index out of range");
  const float* snap = d->hist[(size_t)i / kHistChunk] + ((size_t)i % kHistChunk) * (size_t)m->nv;
  hipLaunchKernelGGL(k_gather, dim3(grid1d(m->nv, 256)), dim3(256), 0, d->stream, snap, d->iperm,
                     m->nv, d->out);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipMemcpyAsync(T_out, d->out, sizeof(float) * m->nv, hipMemcpyDeviceToHost, d->stream));
  HIP_TRY(hipStreamSynchronize(d->stream));
  return EIK_OK;
}

int eik_debug_local_solve(int32_t dim, const float* T, const float* L, int64_t n, float* out) {
  if ((dim != 2 && dim != 3) || !T || !L || !out || n <= 0) return fail(EIK_ERR_ARG, "bad argument");
  const int K = dim == 3 ? 4 : 3, NL = dim == 3 ? 6 : 3;
  // the three buffers are freed on every return path
  struct Bufs {
    float *T = nullptr, *L = nullptr, *O = nullptr;
    ~Bufs() {
      for (float* p : {T, L, O})
        if (p) (void)hipFree(p);
    }
  } b;
  HIP_TRY(hipMalloc((void**)&b.T, sizeof(float) * K * n));
  HIP_TRY(hipMalloc((void**)&b.L, sizeof(float) * NL * n));
  HIP_TRY(hipMalloc((void**)&b.O, sizeof(float) * K * n));
  HIP_TRY(hipMemcpy(b.T, T, sizeof(float) * K * n, hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(b.L, L, sizeof(float) * NL * n, hipMemcpyHostToDevice));
  if (dim == 3)
    hipLaunchKernelGGL(k_debug_local<3>, dim3(grid1d(n, 256)), dim3(256), 0, 0, b.T, b.L, n, b.O,
                       EIK_LARGENUM_3D);
  else
    hipLaunchKernelGGL(k_debug_local<2>, dim3(grid1d(n, 256)), dim3(256), 0, 0, b.T, b.L, n, b.O,
                       EIK_LARGENUM_2D);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipMemcpy(out, b.O, sizeof(float) * K * n, hipMemcpyDeviceToHost));
  return EIK_OK;
}

}  // extern "C"

// ------------------------------------------------------------------------------------------
// The solve that allocates nothing
// ------------------------------------------------------------------------------------------
namespace eik {

// Per-solve state of eik_solve_noalloc (times, seen, queue ring, flags, counters), one array per
// device for the life of the process.  Host code never uses the array's name as an address: the
// device address comes from hipGetSymbolAddress, per device, on the first call on that device.
constexpr size_t kScratchBytes = (size_t)64 << 20;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];
constexpr int kMaxDevices = 64;
static void* g_scratch[kMaxDevices];
static std::mutex g_scratch_mu;

static int scratch_address(int dev, unsigned char** out) {
  if (dev < 0 || dev >= kMaxDevices) return fail(EIK_ERR_HIP, "device index out of range");
  std::lock_guard<std::mutex> g(g_scratch_mu);
  if (!g_scratch[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return fail(EIK_ERR_HIP, std::string("scratch address: ") + hipGetErrorString(e));
    g_scratch[dev] = p;
  }
  *out = reinterpret_cast<unsigned char*>(g_scratch[dev]);
  return EIK_OK;
}

static size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

}  // namespace eik

extern "C" {

int eik_solve_noalloc(eik_mesh_t h, const int32_t* seeds_dev, int64_t nseeds, float* T_out_dev,
                      void* stream) {
  Mesh* m = reinterpret_cast<Mesh*>(h);
  if (!m || !seeds_dev || !T_out_dev || nseeds <= 0) return fail(EIK_ERR_ARG, "bad argument");
  DeviceState* d = m->dev;
  if (m->nblocks <= 0 || !d || !d->blocks || m->device_dirty || !m->layout.valid)
    return fail(EIK_ERR_STATE, "the mesh layout must be uploaded first (eik_mesh_upload)");
  int dev = -1;
  HIP_TRY(hipGetDevice(&dev));
  if (dev != d->device)
    return fail(EIK_ERR_STATE, "the current device is not the one the mesh was uploaded to");
  eik_solve_opts_t o;
  eik_solve_opts_default(&o);
  int grid = 0;
  int rc = persistent_grid(m->dim, visit_kernel(d, o.stage_records), o.workgroups, d->nblocks, nseeds, &grid);
  if (rc) return rc;
  Sched words;
  sched_shape(words, d->nblocks, grid);
  // [control words][counters][block words][T][seen], 256-byte aligned
  const size_t o_cnt = align256(kSchedCtlBytes);
  const size_t o_word = o_cnt + align256(sizeof(unsigned long long) * kNumCounters);
  const size_t o_T = o_word + align256(sizeof(unsigned long long) * (size_t)words.owners * words.stride);
  const size_t o_seen = o_T + align256(sizeof(float) * (size_t)m->nv);
  const size_t need = o_seen + align256(sizeof(float) * (size_t)d->nseen);
  if (need > kScratchBytes)
    return fail(EIK_ERR_CAPACITY, "this mesh needs " + std::to_string(need) +
                                      " bytes of solve state; the allocation-free solve has " +
                                      std::to_string(kScratchBytes) + " (use eik_solve)");
  unsigned char* base = nullptr;
  rc = scratch_address(dev, &base);
  if (rc) return rc;
  // the array keeps the previous call's contents: everything the solve reads first is reset
  const AsyncBufs b = {reinterpret_cast<float*>(base + o_T), reinterpret_cast<float*>(base + o_seen),
                       reinterpret_cast<unsigned long long*>(base + o_word), base,
                       reinterpret_cast<unsigned long long*>(base + o_cnt)};
  return enqueue_async(*m, o, b, seeds_dev, nullptr, nseeds, T_out_dev,
                       nullptr, stream ? reinterpret_cast<hipStream_t>(stream) : d->stream);
}

}  // extern "C"
