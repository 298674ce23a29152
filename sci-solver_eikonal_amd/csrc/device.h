// device.h -- device state and the device-side pieces shared by the solve translation units:
// the per-mesh device state, the per-solve resets, LDS carving and visit tallies.
#pragma once

#include <hip/hip_runtime.h>

#include <string>
#include <vector>

#include "eik_internal.h"
#include "fim_kernels.h"

namespace eik {

#define HIP_TRY(expr)                                                                    \
  do {                                                                                   \
    hipError_t _e = (expr);                                                              \
    if (_e != hipSuccess)                                                                \
      return fail(EIK_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(_e));      \
  } while (0)

// counters[0..13]: visits, vertex updates, inner sweeps, local solves, algorithmic bytes,
// wall-clock ticks summed over workgroups: inside visits, waiting for work, then the parts of a
// visit: staging loads, sweeps, write-back, queueing of dependents; visits that followed the
// same workgroup's visit of the same block (re-runs); queue waits abandoned at the wait limit;
// algorithmic bytes without the element data of re-runs whose records were still staged
constexpr int kNumCounters = 14;
constexpr int kCntAbandoned = 12;
constexpr int kCntAlgoLoaded = 13;
// The one-launch-per-iteration kernel adds each visit's counters to one of kSyncSlots lines of
// 128 bytes (workgroup i to line i mod kSyncSlots); they are summed into counters after the
// solve.  Every visit adding to the same line serialised the peak iterations of the 64^3 cube
// (about 4,000 visits each) on that line's atomics.
constexpr int kSyncSlots = 128;
constexpr int kSyncSlotWords = 16;

struct DeviceState {
  int device = -1;
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  hipEvent_t evA = nullptr, evB = nullptr;  // around each block-visit launch
  int dim = 3;
  int32_t nblocks = 0;
  int64_t nv = 0;
  BlockDesc* blocks = nullptr;
  void* elems = nullptr;
  int32_t* halo = nullptr;
  int32_t* iperm = nullptr;
  int32_t* dep_start = nullptr;
  int32_t* dep = nullptr;
  int32_t* owner = nullptr;
  float* T = nullptr;
  float* out = nullptr;
  float* seen = nullptr;
  int64_t nseen = 0;
  int32_t* vh_start = nullptr;
  uint16_t* vh_pos = nullptr;
  uint64_t* vmask = nullptr;
  int32_t* rec_elem = nullptr;
  int32_t rec_lds = 0;
  size_t rec_lds_bytes = 0;
  int32_t* stamp[2] = {nullptr, nullptr};  // synchronous scheduler (Active), by parity of the iteration
  int32_t* list[2] = {nullptr, nullptr};
  int32_t* count = nullptr;  // active counts of iterations modulo 3, last visited iteration
  unsigned long long* counters = nullptr;
  unsigned long long* sync_acc = nullptr;  // kSyncSlots * kSyncSlotWords
  int32_t* seeds = nullptr;
  float* seedvals = nullptr;
  int64_t seed_cap = 0;
  // pinned host staging, so the per-solve copies are plain DMA: the seeds then their values
  // (2 * seed_cap words) on the way in, the counters on the way out
  int32_t* h_seed = nullptr;
  unsigned long long* h_cnt = nullptr;
  // behind h_cnt: a word that the synchronous scheduler's iterations write, a small mesh's times
  // (kSmallOut)
  float* h_out = nullptr;
  // persistent scheduler (block_sched.h): block words and control words
  unsigned long long* words = nullptr;
  unsigned char* sctl = nullptr;
  int32_t max_workgroups = 0;
  size_t lds_bytes = 0;         // a visit with its records staged (when rec_lds)
  size_t lds_bytes_direct = 0;  // a visit reading its records from memory
  int32_t queue_cap = 0;
  // the visits that keep a block's element data in registers (k_visit_resident): items or
  // elements per thread (0: the blocks do not fit), threads, LDS strides and bytes, and for
  // triangles the items (resident.h, TriItems)
  int32_t res_n = 0, res_bt = 0;
  int32_t max_queue = 0;
  bool res_cap = false;  // the work-item queue holds fewer pairs than a block has
  int32_t max_local = 0, max_elem = 0;
  float height_unit = 1.f;
  size_t res_lds = 0;
  int2* item_range = nullptr;
  uint32_t* item_id = nullptr;
  float4* item_len = nullptr;
  uint16_t* item_rec = nullptr;
  bool has_result = false;
  // split element records of the multi-solve visits that read them from memory (ensure_split)
  void* esel = nullptr;
  float* elen = nullptr;
  // per-outer-iteration snapshots of T (block-contiguous order) of the last sync solve with
  // record_history, kHistChunk snapshots per allocation
  std::vector<float*> hist;
  int64_t hist_len = 0;
};

constexpr int kHistChunk = 8;

template <typename T>
inline int upload(T** dst, const std::vector<T>& src, hipStream_t s) {
  size_t n = std::max<size_t>(src.size(), 1);
  HIP_TRY(hipMalloc((void**)dst, n * sizeof(T)));
  if (!src.empty())
    HIP_TRY(hipMemcpyAsync(*dst, src.data(), src.size() * sizeof(T), hipMemcpyHostToDevice, s));
  return EIK_OK;
}

static inline unsigned grid1d(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }


// The per-solve resets in one launch: segment k sets n[k] 32-bit words at p[k] to v[k], and `words`
// block words to clean (a launch per array costs about 5 us each, most of a small solve's set-up).
struct FillSegs {
  static constexpr int kMax = 8;
  int32_t* p[kMax];
  int64_t n[kMax];
  int32_t v[kMax];
  int count = 0;
  unsigned long long* words[2] = {nullptr, nullptr};  // block words (block_sched.h)
  int64_t nwords[2] = {0, 0};
  unsigned long long* begin = nullptr;  // gets the device clock
  void add(void* ptr, int64_t words32, int32_t value) {
    p[count] = reinterpret_cast<int32_t*>(ptr);
    n[count] = words32;
    v[count] = value;
    ++count;
  }
};

// solver.hip
void launch_fill(const FillSegs& f, hipStream_t s);
int ensure_stream(Mesh& m);
int upload_layout(Mesh& m);
size_t visit_lds_bytes(const Layout& L, int dim, int32_t queue_cap, size_t rec_bytes);

// Carves the dynamic LDS of a visit: [records (rec_lds_bytes)] [sT] [sOld] [sChg] [sQ].
struct VisitLds {
  void* rec;
  float* T;
  float* old;
  int* chg;
  int* hidx;
  uint64_t* vm;
  uint16_t* q;
  int* mark;
};

template <int DIM>
__device__ __forceinline__ VisitLds carve_lds(void* base, size_t rec_bytes, int queue_cap,
                                              const BlockDesc& d) {
  VisitLds l;
  char* p = reinterpret_cast<char*>(base);
  l.rec = p;
  l.T = reinterpret_cast<float*>(p + rec_bytes);
  l.old = l.T + (d.nown + d.nhalo);
  l.chg = reinterpret_cast<int*>(l.old + d.nown);
  l.hidx = l.chg + (d.nown + d.nhalo);
  if constexpr (DIM == 2) {  // dependent masks of the owned vertices (triangle visits only)
    l.vm = reinterpret_cast<uint64_t*>((reinterpret_cast<uintptr_t>(l.hidx + d.nhalo) + 7) &
                                       ~static_cast<uintptr_t>(7));
    l.q = reinterpret_cast<uint16_t*>(l.vm + d.nown);
  } else {
    l.vm = nullptr;
    l.q = reinterpret_cast<uint16_t*>(l.hidx + d.nhalo);
  }
  l.mark = reinterpret_cast<int*>(l.q + ((queue_cap + 1) & ~1));
  return l;
}

// Wall-clock ticks of a queue-wait limit given in microseconds (0: 10 s).
inline unsigned long long wait_limit_ticks(int device, int32_t us) {
  int khz = 0;
  if (hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, device) != hipSuccess || khz <= 0)
    khz = 100000;
  const unsigned long long u = us > 0 ? (unsigned long long)us : 10000000ull;
  return u * (unsigned long long)khz / 1000ull;
}

// After a launch whose workgroups gave up waiting: EIK_OK if the solve behind the control words still
// reached its end (the result is complete), else EIK_ERR_TIMEOUT.  Synchronises stream s.
int check_end(const unsigned char* sctl, hipStream_t s, unsigned long long abandoned);

// Algorithmic HBM bytes of one block visit: the element data a visit needs (6 metric values and
// 4 local ids per tet = 32 B, 3 values and 3 ids plus padding per triangle = 20 B), the owned
// and halo times read, the owned times written, and one flag word.  The kernels' records are
// larger (corner heights for pruning) and a visit also touches `seen`, halo ids and its
// descriptor, while a re-run reads no records at all: the bytes actually moved are measured
// with hardware counters, and this figure is the common yardstick.
template <int DIM>
constexpr int kAlgoElemBytes = DIM == 3 ? 32 : 20;
__device__ __forceinline__ unsigned long long visit_algo_bytes(int elem_bytes, const BlockDesc& d) {
  return (unsigned long long)elem_bytes * d.nelem + 4ull * (d.nown + d.nhalo) + 4ull * d.nown + 4ull;
}

// Adds one visit to a workgroup's own tally (thread 0; flushed once when the workgroup exits,
// so the visits of a solve do not contend on shared counter words).  recs_staged: a re-run whose
// element records are still in LDS from the previous visit (it reads none from memory).
__device__ __forceinline__ void tally_visit(unsigned long long* acc, const BlockDesc& d,
                                            const VisitResult& r, unsigned long long solves,
                                            int elem_bytes, unsigned long long busy_ticks,
                                            bool rerun, bool recs_staged) {
  const unsigned long long ab = visit_algo_bytes(elem_bytes, d);
  acc[0] += 1;
  acc[1] += (unsigned long long)d.nown;
  acc[2] += (unsigned long long)r.sweeps;
  acc[3] += solves;
  acc[4] += ab;
  acc[kCntAlgoLoaded] += recs_staged ? ab - (unsigned long long)elem_bytes * d.nelem : ab;
  acc[11] += rerun ? 1ull : 0ull;
  acc[5] += busy_ticks;
  acc[7] += r.t_load;
  acc[8] += r.t_sweep;
  acc[9] += r.t_wb;
}

}  // namespace eik
