// resident.h -- block visits that keep a block's element data in registers (device code).
//
// A persistent workgroup visits the same block several times in a row (a re-run is five of six
// visits of the 64^3 cube), and a visit of a 64-vertex block is a chain of short phases, each a
// few LDS round trips long, not a volume of work.  So what a sweep reads is placed for the
// shortest chain:
//   * triangles: one (target, two others) item per updatable corner, rotated once when the block
//     is loaded, N items per thread in registers with the times they were last solved with.  A
//     sweep is three LDS reads per item, the test, the solve in place and an LDS minimum: one
//     barrier, no work-item queue, no records in LDS.
//   * tets: N elements per thread in registers for the selection (corner slots, heights, the
//     corner times last seen), four LDS reads per element; the selected (element, corner) pairs
//     go through the LDS queue, since a sweep solves one in fifteen of them, and only what the
//     solve reads (corner slots, lengths: 32 bytes) is staged in LDS.
// Freshness is per item: it is solved again only if one of the *other* corners fell since its last
// evaluation by this visit's workgroup (across visits: since the `seen` times).
#pragma once

#include "fim_kernels.h"
#include "lane_ops.h"

namespace eik {

// Items of the triangle blocks: block b's items are [start, start + count) of the arrays.
// id: slots of the two other corners and the target, 10 bits each (a | b << 10 | target << 20);
// len: {|a - target|^2, |b - target|^2, |a - b|^2, height of the target}; rec: the item's element
// record within the block.
struct TriItems {
  const int2* range;
  const uint32_t* id;
  const float4* len;
  const uint16_t* rec;
};
constexpr int kItemSlotBits = 10;
constexpr int kItemSlots = 1 << kItemSlotBits;  // local vertices of a block with items

// Whether a fall counts as a change, after which a visit sweeps again: by more than eps relative (eps = 0:
// at all).
__device__ __forceinline__ bool fell(float last, float now, float eps) {
  return last - now > eps * now;
}

// What a sweep tests first it does for every item, changed or not, and with the instructions issued
// on two thirds of all cycles (96^3 cube) their number counts: so an item holds the LDS offsets of its
// corners' times instead of slots.  A corner counts as fallen if it lies below its last time at all,
// whatever eps: falls within eps are many, and where each had to exceed it alone, with a block's record of
// evaluated times starting anew at every visit, their sum was lost (persistent solves at eps = 0.01,
// largest relative error: 32^3 cube 3e-2, now 1e-5; level-7 icosphere 7e-2, now 9e-3).
__device__ __forceinline__ float time_at(const float* sT, uint32_t offset) {
  return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(sT) + offset);
}

template <int N>
struct TriRegs {
  uint32_t ab[N], t[N];  // LDS offsets of the two other corners, 16 bits each, and of the target
  float la[N], lb[N], lab[N], h[N];
  float pa[N], pb[N];  // the two other corners' times at the last evaluation
};

// The thread index, opaque: what is computed from it is computed where it is used, not hoisted out of
// the loop over the blocks and spilled (a reload waits for every load issued before it).
__device__ __forceinline__ int this_thread() {
  int t = threadIdx.x;
  asm volatile("" : "+v"(t));
  return t;
}

// rmult: a factor per record of the block on its squared lengths, or null (a factor f scales the
// heights by sqrt(f)).
template <int N, int BT>
__device__ __forceinline__ void tri_load(TriRegs<N>& r, const TriItems& t, int2 range,
                                         const float* rmult) {
  const int tid = this_thread();
#pragma unroll
  for (int u = 0; u < N; ++u) {
    const int i = u * BT + tid;
    const bool in = i < range.y;
    const uint32_t id = in ? t.id[range.x + i] : 0u;
    r.ab[u] = (id << 2 & 4 * (kItemSlots - 1)) | (id >> kItemSlotBits & (kItemSlots - 1)) << 18;
    r.t[u] = id >> (2 * kItemSlotBits) << 2;
    const float4 l = in ? t.len[range.x + i] : make_float4(1.f, 1.f, 1.f, EIK_INF);
    r.la[u] = l.x;
    r.lb[u] = l.y;
    r.lab[u] = l.z;
    r.h[u] = l.w;
  }
  if (rmult) {
#pragma unroll
    for (int u = 0; u < N; ++u) {
      const int i = u * BT + tid;
      const float f = i < range.y ? rmult[t.rec[range.x + i]] : 1.f;
      r.la[u] *= f;
      r.lb[u] *= f;
      r.lab[u] *= f;
      r.h[u] *= __builtin_sqrtf(f);
    }
  }
}

template <int N>
__device__ __forceinline__ void tri_seen(TriRegs<N>& r, const float* sP) {
#pragma unroll
  for (int u = 0; u < N; ++u) {
    r.pa[u] = time_at(sP, r.ab[u] & 0xffffu);
    r.pb[u] = time_at(sP, r.ab[u] >> 16);
  }
}

// One sweep over the thread's items.  Returns whether it lowered a time.
template <int N>
__device__ __forceinline__ bool tri_sweep(TriRegs<N>& r, float* sT, float large, float eps,
                                          unsigned& solves) {
  float ta[N], tb[N], tk[N];
  // What a solve computes from the lengths alone stays in registers from sweep to sweep where there
  // is room (N = 2); for more items it would be spilled, so it is computed again.
  if constexpr (N > 2) {
#pragma unroll
    for (int u = 0; u < N; ++u) asm volatile("" : "+v"(r.la[u]), "+v"(r.lb[u]), "+v"(r.lab[u]));
  }
#pragma unroll
  for (int u = 0; u < N; ++u) {
    ta[u] = time_at(sT, r.ab[u] & 0xffffu);
    tb[u] = time_at(sT, r.ab[u] >> 16);
    tk[u] = time_at(sT, r.t[u]);
  }
  bool changed = false;
#pragma unroll
  for (int u = 0; u < N; ++u) {
    if (!(ta[u] < r.pa[u] || tb[u] < r.pb[u])) continue;
    r.pa[u] = ta[u];
    r.pb[u] = tb[u];
    // nothing below the smaller time plus the height; unknown times are `large`, and no time
    // is above that
    if (!(tk[u] > __builtin_fminf(ta[u], tb[u]) + r.h[u])) continue;
    ++solves;
    bool bad = false;
    float cand = tri_corner_solve<kReport>(ta[u], tb[u], r.la[u], r.lb[u], r.lab[u], large, &bad);
    if (__builtin_expect(bad, 0))
      cand = tri_corner_solve_wide(ta[u], tb[u], r.la[u], r.lb[u], r.lab[u], large);
    cand = __builtin_fmaxf(cand, 0.f);
    if (cand < tk[u]) {
      atomicMin(reinterpret_cast<unsigned*>(reinterpret_cast<char*>(sT) + r.t[u]), __float_as_uint(cand));
      changed |= fell(tk[u], cand, eps);
    }
  }
  return changed;
}

// The smallest of three times, which are not negative: as integers, which need no quieting of NaNs.
__device__ __forceinline__ float time_min(float a, float b, float c) {
  const uint32_t x = __float_as_uint(a), y = __float_as_uint(b), z = __float_as_uint(c);
  const uint32_t m = x < y ? x : y;
  return __uint_as_float(m < z ? m : z);
}

template <int N>
struct TetRegs {
  uint32_t v01[N], v23[N];     // LDS offsets of the corners' times, 16 bits each
  // heights in fp16 times `unit`, rounded down (they stay lower bounds of every solve); +inf: not owned.
  // The unit is a power of two that takes the mesh's largest height, or with factors the thread's, to 2^14
  // .. 2^15 units: heights keep 11 bits down to 2^-28 of it, whatever the mesh's scale (in units of 1 a 24^3
  // cube with edges below 1e-7 or above 1e5 ran 3 times as many local solves, 0.18 -> 0.22 ms).
  uint32_t h01[N], h23[N];
  float unit;
  float p0[N], p1[N], p2[N], p3[N];  // the corners' times at the last selection
};

// A sum with the height in the low or high half of h, in one instruction (v_fma_mix_f32), rounded once.
__device__ __forceinline__ float above_lo(float t, uint32_t h, float unit) {
  return __builtin_fmaf(h2f(h & 0xffffu), unit, t);
}
__device__ __forceinline__ float above_hi(float t, uint32_t h, float unit) {
  return __builtin_fmaf(h2f(h >> 16), unit, t);
}

// Loads the thread's records: slots and heights to registers, slots and lengths to LDS.
// unit: of the mesh's heights (Layout::height_unit); rmult as in tri_load.
template <int N, int BT>
__device__ __forceinline__ void tet_load(TetRegs<N>& r, const void* recs, const BlockDesc& d,
                                         uint4* sA, uint4* sB, float unit, const float* rmult) {
  const uint4* p = reinterpret_cast<const uint4*>(recs) + 3 * (int64_t)d.estart;
  const int tid = this_thread();
  const int wave = __builtin_amdgcn_readfirstlane(tid & ~63);
  float h[N][4];
#pragma unroll
  for (int u = 0; u < N; ++u) {
    const int e = u * BT + tid;
    const bool in = e < d.nelem;
    const uint4* q = p + 3 * (in ? e : 0);
    if (in && !rmult) {
      copy_to_lds(q, sA + u * BT + wave);
      copy_to_lds(q + 1, sB + u * BT + wave);
    }
    const uint2 v = *reinterpret_cast<const uint2*>(q);
    const uint4 hq = q[2];
    float h0 = __uint_as_float(hq.x), h1 = __uint_as_float(hq.y);
    float h2 = __uint_as_float(hq.z), h3 = __uint_as_float(hq.w);
    if (rmult && in) {
      const float f = rmult[e], sf = __builtin_sqrtf(f);
      const uint4 a = q[0], b = q[1];
      sA[e] = make_uint4(a.x, a.y, __float_as_uint(__uint_as_float(a.z) * f),
                         __float_as_uint(__uint_as_float(a.w) * f));
      sB[e] = make_uint4(__float_as_uint(__uint_as_float(b.x) * f),
                         __float_as_uint(__uint_as_float(b.y) * f),
                         __float_as_uint(__uint_as_float(b.z) * f),
                         __float_as_uint(__uint_as_float(b.w) * f));
      h0 *= sf;
      h1 *= sf;
      h2 *= sf;
      h3 *= sf;
    }
    const unsigned n = in ? (unsigned)d.nown : 0u;
    h[u][0] = (v.x & 0xffffu) < n ? h0 : EIK_INF;
    h[u][1] = (v.x >> 16) < n ? h1 : EIK_INF;
    h[u][2] = (v.y & 0xffffu) < n ? h2 : EIK_INF;
    h[u][3] = (v.y >> 16) < n ? h3 : EIK_INF;
    r.v01[u] = v.x << 2;  // (the LDS holds fewer than 2^14 times)
    r.v23[u] = v.y << 2;
  }
  if (rmult) {
    float most = 0.f;
#pragma unroll
    for (int u = 0; u < N; ++u)
#pragma unroll
      for (int k = 0; k < 4; ++k) most = __builtin_fmaxf(most, h[u][k] < EIK_INF ? h[u][k] : 0.f);
    unit = height_unit(__builtin_amdgcn_frexp_expf(most));
  }
  r.unit = unit;
  const float per_unit = __uint_as_float((254u << 23) - __float_as_uint(unit));  // 1 / unit, a power of two
#pragma unroll
  for (int u = 0; u < N; ++u) {
    r.h01[u] = half_pair(h[u][0] * per_unit, h[u][1] * per_unit);
    r.h23[u] = half_pair(h[u][2] * per_unit, h[u][3] * per_unit);
  }
}

template <int N>
__device__ __forceinline__ void tet_seen(TetRegs<N>& r, const float* sP) {
#pragma unroll
  for (int u = 0; u < N; ++u) {
    r.p0[u] = time_at(sP, r.v01[u] & 0xffffu);
    r.p1[u] = time_at(sP, r.v01[u] >> 16);
    r.p2[u] = time_at(sP, r.v23[u] & 0xffffu);
    r.p3[u] = time_at(sP, r.v23[u] >> 16);
  }
}

// Inclusive sum over the lanes of a wave, in six DPP steps.
__device__ __forceinline__ int wave_scan(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);  // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);  // row_shr:2
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);  // row_shr:4
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);  // row_shr:8
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast:15
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);  // row_bcast:31
  return x;
}

// Bitwise or over the lanes of a wave (valid in lane 63).
__device__ __forceinline__ uint32_t wave_or(uint32_t v) {
  int x = (int)v;
  x |= __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);  // row_shr:1
  x |= __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);  // row_shr:2
  x |= __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);  // row_shr:4
  x |= __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);  // row_shr:8
  x |= __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast:15
  x |= __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);  // row_bcast:31
  return (uint32_t)x;
}

// A queued pair: thread and, in the low five bits, its element's place u and the corner, 4 u + k.
template <int BT>
__device__ __forceinline__ int item_elem(int item) { return (item >> 2 & 7) * BT + (item >> 5); }

// Appends the (element, corner) pairs of the thread's elements that can improve to the queue.  CAP:
// it may hold fewer than a block has, max_queue; sets *again, and *full to the visit's number, if it did not hold them.
// About 190 vector instructions a wave for N = 4 (350 with slots, last times, quieted minima and
// converted heights): the visits of the 64^3 cube 0.677 -> 0.650 ms, of the 96^3 cube 1.50 -> 1.44.
template <int N, int BT, bool CAP>
__device__ __forceinline__ void tet_select(TetRegs<N>& r, int nelem, const float* sT,
                                           uint16_t* sQ, int max_queue, int* qn, int* again, int* full, int visit) {
  static_assert(N <= 8 && BT <= 2048, "queued pairs have 5 bits for the place, 11 for the thread");
  // places of this wave that hold an element (64^3 cube 0.651 -> 0.633 ms with the others left out)
  const int places = (nelem - __builtin_amdgcn_readfirstlane((int)threadIdx.x & ~63) + BT - 1) / BT;
  float t0[N], t1[N], t2[N], t3[N];
#pragma unroll
  for (int u = 0; u < N; ++u) {
    if (u >= 2 && u >= places) break;
    t0[u] = time_at(sT, r.v01[u] & 0xffffu);
    t1[u] = time_at(sT, r.v01[u] >> 16);
    t2[u] = time_at(sT, r.v23[u] & 0xffffu);
    t3[u] = time_at(sT, r.v23[u] >> 16);
  }
  unsigned sel = 0;
#pragma unroll
  for (int u = 0; u < N; ++u) {
    if (u >= 2 && u >= places) break;
    const bool f0 = t0[u] < r.p0[u], f1 = t1[u] < r.p1[u];
    const bool f2 = t2[u] < r.p2[u], f3 = t3[u] < r.p3[u];
    if (!(f0 || f1 || f2 || f3)) continue;
    r.p0[u] = t0[u];
    r.p1[u] = t1[u];
    r.p2[u] = t2[u];
    r.p3[u] = t3[u];
    // a corner is solved again if another one fell and it lies above the smallest of the others by
    // more than its height
    const bool c0 = t0[u] > above_lo(time_min(t1[u], t2[u], t3[u]), r.h01[u], r.unit);
    const bool c1 = t1[u] > above_hi(time_min(t0[u], t2[u], t3[u]), r.h01[u], r.unit);
    const bool c2 = t2[u] > above_lo(time_min(t0[u], t1[u], t3[u]), r.h23[u], r.unit);
    const bool c3 = t3[u] > above_hi(time_min(t0[u], t1[u], t2[u]), r.h23[u], r.unit);
    sel |= (c0 && (f1 || f2 || f3) ? 1u << 4 * u : 0u) | (c1 && (f0 || f2 || f3) ? 2u << 4 * u : 0u);
    sel |= (c2 && (f0 || f1 || f3) ? 4u << 4 * u : 0u) | (c3 && (f0 || f1 || f2) ? 8u << 4 * u : 0u);
  }
  if (__ballot(sel != 0u) == 0ull) return;
  const int n = __popc(sel);
  const int end = wave_scan(n);
  int base = 0;
  if (__lane_id() == 63) base = lds_take(qn, end);
  base = __builtin_amdgcn_readlane(base, 63);
  const int me = (int)threadIdx.x << 5;
  int q = base + end - n;
  if (!CAP || __builtin_expect(base + __builtin_amdgcn_readlane(end, 63) <= max_queue, 1)) {
    for (; sel; ++q, sel &= sel - 1u) sQ[q] = (uint16_t)(me | (__ffs(sel) - 1));
  } else {
    for (; sel && q < max_queue; ++q, sel &= sel - 1u) sQ[q] = (uint16_t)(me | (__ffs(sel) - 1));
    // what a full queue turns away counts as not evaluated, and another sweep follows
    *again = 1;
    *full = visit;
#pragma unroll
    for (int u = 0; u < N; ++u)
      if (sel >> (4 * u) & 15u) r.p0[u] = r.p1[u] = r.p2[u] = r.p3[u] = EIK_INF;
  }
}

struct TetItem {
  float t0, t1, t2, t3;
  uint4 a, b;  // slots and lengths
  int k;
};

template <int BT>
__device__ __forceinline__ TetItem tet_item(const uint4* sA, const uint4* sB, int item,
                                            const float* sT) {
  TetItem x;
  const int e = item_elem<BT>(item);
  x.k = item & 3;
  x.a = sA[e];
  x.b = sB[e];
  x.t0 = sT[x.a.x & 0xffffu];
  x.t1 = sT[x.a.x >> 16];
  x.t2 = sT[x.a.y & 0xffffu];
  x.t3 = sT[x.a.y >> 16];
  return x;
}

// Lowers the target of an item to a candidate; returns whether it fell.
__device__ __forceinline__ bool tet_lower(const TetItem& x, float cand, float* sT, float eps) {
  const float tk = x.k == 0 ? x.t0 : x.k == 1 ? x.t1 : x.k == 2 ? x.t2 : x.t3;
  const uint32_t pair = x.k < 2 ? x.a.x : x.a.y;
  const int vk = (x.k & 1) ? pair >> 16 : pair & 0xffffu;
  cand = __builtin_fmaxf(cand, 0.f);
  if (!(cand < tk)) return false;
  atomicMin(reinterpret_cast<unsigned*>(&sT[vk]), __float_as_uint(cand));
  return fell(tk, cand, eps);
}

// The queued pairs of ill-conditioned tets, again, in fp64.  What the thread holds of its elements
// goes to memory meanwhile: kept in registers across the calls, the compiler spills most of it on
// every load of a block, whether the block has such tets or not.
template <int N, int BT>
__device__ __forceinline__ bool tet_solve_ill(TetRegs<N>& r, const uint4* sA, const uint4* sB,
                                              const uint16_t* sQ, int nq, float* sT, float large,
                                              float eps) {
  TetRegs<N> keep = r;
  asm volatile("" : : "v"(&keep) : "memory");  // in memory, not in registers
  bool changed = false;
  for (int q = threadIdx.x; q < nq; q += BT) {
    const TetItem x = tet_item<BT>(sA, sB, sQ[q], sT);
    const float cand = tet_rotation_wide(
        x.k, x.t0, x.t1, x.t2, x.t3, __uint_as_float(x.a.z), __uint_as_float(x.a.w),
        __uint_as_float(x.b.x), __uint_as_float(x.b.y), __uint_as_float(x.b.z),
        __uint_as_float(x.b.w), large);
    changed |= tet_lower(x, cand, sT, eps);
  }
  asm volatile("" : : "v"(&keep) : "memory");
  r = keep;
  return changed;
}

// Solves the queued pairs.  Returns whether the thread lowered a time.
template <int N, int BT>
__device__ __forceinline__ bool tet_solve(TetRegs<N>& r, const uint4* sA, const uint4* sB,
                                          const uint16_t* sQ, int nq, float* sT, float large,
                                          float eps, unsigned& solves) {
  bool changed = false, ill = false;
  for (int q = threadIdx.x; q < nq; q += BT) {
    const TetItem x = tet_item<BT>(sA, sB, sQ[q], sT);
    ++solves;
    bool bad = false;
    const float cand = tet_rotation<kReport>(
        x.k, x.t0, x.t1, x.t2, x.t3, __uint_as_float(x.a.z), __uint_as_float(x.a.w),
        __uint_as_float(x.b.x), __uint_as_float(x.b.y), __uint_as_float(x.b.z),
        __uint_as_float(x.b.w), large, &bad);
    ill |= bad;
    if (!bad) changed |= tet_lower(x, cand, sT, eps);
  }
  if (__builtin_expect(__ballot(ill) != 0ull, 0))
    changed |= tet_solve_ill<N, BT>(r, sA, sB, sQ, nq, sT, large, eps);
  return changed;
}

}  // namespace eik
