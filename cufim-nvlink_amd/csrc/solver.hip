// solver.hip -- gfx950 kernels of the FIM activation-time solve and the
// device half of the C ABI (fim_create ... fim_destroy).
//
// Two modes share one pack (host.hpp):
//
//  converge (FP32, exact local solver): per global iteration a persistent
//    kernel (k_conv_band) works through the (instance, submesh) pairs of the
//    iteration's work list, dealt out per XCD in units of a few instances of
//    one submesh.  A work item stages the submesh's vertex times in LDS and
//    runs Jacobi sweeps (capped per activation): sources mark their incident
//    elements through a padded vertex -> element adjacency, the marked
//    elements evaluate exact candidates from 48-byte element records read
//    from L2, and candidates merge with LDS atomicMin on the float bit
//    pattern (times are >= 0, so the IEEE order equals the unsigned order).
//    At its end a work item pushes its lowered interface copies to the other
//    copies of the vertex: global atomicMin into the copy's inbox entry of the
//    next iteration, whose work item merges it when it stages the submesh,
//    and the submesh is queued on the next list.  Inbox, queue flags and wake
//    times exist twice, for even and odd iterations: a kernel reads one set
//    and writes the other, so results are independent of scheduling (atomic
//    min, max and "set" flags commute).  With more instances than a work
//    unit holds, a second kernel (k_conv_plan) cuts the next list into work
//    units; otherwise an iteration is one launch.  Each
//    instance's time window counts from its own start iteration, so a
//    converged instance can be recycled and seeded again mid-run.
//    Iterations are recorded in a hipGraph; the host reads one counter per
//    graph launch.
//
//  compat (FP64, reference local update): one workgroup per submesh runs the
//    reference's per-window phases a-g (src/eikonal/cuda_fim.cu:1992-2334)
//    with vertex times and states in LDS; a separate kernel min-merges the
//    copies of interface vertices (sync_step2, cuda_fim.cu:1752-1787).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "host.hpp"
#include "local_solve.hpp"

#define HIPCHECK(x)                                                                   \
  do {                                                                                \
    hipError_t err_ = (x);                                                            \
    if (err_ != hipSuccess)                                                           \
      throw fim::Error(FIM_EDEVICE, std::string(#x) + ": " + hipGetErrorString(err_)); \
  } while (0)

namespace fim {
namespace {

constexpr float F_INF = __builtin_huge_valf();
constexpr int kHardLocalCap = 4096;  // sweeps per activation before requeue

__device__ inline uint64_t lanes_below() {
  const uint32_t lane = threadIdx.x & 63;
  return lane ? (~0ull >> (64 - lane)) : 0ull;
}

// x as a value of its own: what is computed from it is not kept in registers
// from an earlier phase
__device__ inline uint32_t fresh(uint32_t x) {
  asm volatile("" : "+v"(x));
  return x;
}

__device__ inline bool flag_at(const uint32_t *bits, uint32_t l) {
  return (bits[l >> 5] >> (l & 31)) & 1u;
}

// set bits of the word of l below l
__device__ inline uint32_t bits_below(const uint32_t *bits, uint32_t l) {
  return __popc(bits[l >> 5] & ((1u << (l & 31)) - 1u));
}

// ---------------------------------------------------------------------------
// converge mode
//
// Work lists are bucketed by submesh: bcnt[s] instances of submesh s are
// queued in bins[s * ninst ...].  A (instance, submesh) pair is queued at most
// once per list (the act flag is set on queueing and cleared when the pair is
// processed), so a bucket never holds more than ninst entries.  After the
// list is complete the plan kernel cuts every bucket into work units of up to
// `unit` instances (plan[u] = s * maxch + chunk, submesh-major) and writes the
// unit count.  Units are dealt out XCD-aware: workgroup b runs on XCD b % 8,
// so the unit range is split into 8 contiguous eighths and workgroups of XCD
// x take units of eighth x first (one static unit each, then from the
// eighth's counter), then help the other eighths.  Instances of one submesh
// thus run on one XCD, back to back, and its element data is fetched into
// that XCD's L2 once.
// ---------------------------------------------------------------------------
struct WorkList {
  uint32_t *bcnt;   // nsub: queued instances per submesh
  uint32_t *bins;   // nsub x ninst instance ids
  uint32_t *plan;   // work units
  uint32_t *cnt;    // [0] units, [1] queued pairs, [2] number of the iteration that
                    // works through the list, from kGrab per-XCD unit counters
};

constexpr uint32_t kXcd = 8;
constexpr uint32_t kIterWord = 2;
// A unit counter has a 128 B line to itself: with all eight and the unit count
// in one line, the XCDs' accesses to it limited launches of many small units (357
// maps on 128 submeshes, one instance a unit: 66.2 ms, with lines of their own
// and the own counter asked first 34.6; 395 maps on 127: 77.0 -> 32.5).
constexpr uint32_t kCntLine = 32, kGrab = kCntLine, kCntWords = kGrab + kXcd * kCntLine;

// Queue flags of the items of iteration k: act = 4 (k + 1) + why, so a flag
// needs no clearing; kPushed outranks kQueued.
constexpr uint32_t kQueued = 1, kPushed = 2;
__device__ inline uint32_t act_tag(uint32_t iter) { return 4u * (iter + 1u); }
// Iterations have numbers below this: the last one queues items for the
// iteration after it, and those flags still fit 32 bits.  A context that runs
// on without a reset is renumbered before (k_conv_renumber).
constexpr uint32_t kIterEnd = (1u << 30) - 2u;

// Where items are queued: a list and its iteration's queue flags.
struct Queue {
  WorkList l;
  uint32_t *act;    // n_inst x nsub
  uint32_t tag;     // act_tag of the list's iteration
  uint32_t nsub, ninst;
  uint32_t direct;  // a bucket is one work unit: planned by its first item

  // for kernels between iterations: the list's own iteration number tells the
  // flags' parity and tag
  __device__ void enter() {
    const uint32_t iter = l.cnt[kIterWord];
    act += (iter & 1u) * (size_t)ninst * nsub;
    tag = act_tag(iter);
  }
  __device__ void add(uint32_t inst, uint32_t s, uint32_t why) const {
    if (atomicMax(&act[(size_t)inst * nsub + s], tag + why) >= tag) return;
    const uint32_t j = atomicAdd(&l.bcnt[s], 1u);
    l.bins[(size_t)s * ninst + j] = inst;
    if (direct && j == 0) l.plan[atomicAdd(&l.cnt[0], 1u)] = s;
  }
};

// Builds the work units of a complete list (one workgroup of 1024 threads)
// and clears the buckets of the list the iteration has consumed.
struct PlanArgs {
  const uint32_t *bcnt;
  uint32_t *plan;
  uint32_t *cnt;
  uint32_t *zero_bcnt;  // consumed list, may be null
  uint32_t nsub, unit, maxch;
};

__global__ __launch_bounds__(1024) void k_conv_plan(PlanArgs a) {
  __shared__ uint32_t wsum[16], witems[16];
  __shared__ uint32_t base_sh, items_sh;
  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (tid == 0) {
    base_sh = 0u;
    items_sh = 0u;
  }
  __syncthreads();
  for (uint32_t s0 = 0; s0 < a.nsub; s0 += 1024) {
    const uint32_t s = s0 + tid;
    uint32_t n = 0;
    if (s < a.nsub) {
      n = a.bcnt[s];
      if (a.zero_bcnt) a.zero_bcnt[s] = 0u;
    }
    const uint32_t ch = (n + a.unit - 1) / a.unit;
    uint32_t v = ch, m = n;
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t t = __shfl_up(v, off);
      if (lane >= (uint32_t)off) v += t;
      m += __shfl_xor(m, off);
    }
    if (lane == 63) wsum[wave] = v;
    if (lane == 0) witems[wave] = m;
    __syncthreads();
    uint32_t pre = 0, tot = 0, itot = 0;
    for (uint32_t w = 0; w < 16; ++w) {
      if (w < wave) pre += wsum[w];
      tot += wsum[w];
      itot += witems[w];
    }
    const uint32_t off = base_sh + pre + v - ch;
    for (uint32_t j = 0; j < ch; ++j) a.plan[off + j] = s * a.maxch + j;
    __syncthreads();
    if (tid == 0) {
      base_sh += tot;
      items_sh += itot;
    }
    __syncthreads();
  }
  if (tid == 0) {
    a.cnt[0] = base_sh;
    a.cnt[1] = items_sh;
  }
  if (tid < kXcd) a.cnt[kGrab + kCntLine * tid] = 0u;
}

struct ConvArgs {
  const SubInfo *sub;
  const uint2 *e2n;      // 4 x u16 local ids per element
  const float *geo;      // 6 per element
  const float4 *hgt;     // staged kernel, per element: height of each node above its opposite face
  const uint8_t *ereg;   // region per element
  const float *rscale;   // n_inst x 4 geometry multipliers (1/s^2)
  float *phi;            // n_inst x ncopy
  uint8_t *dirty;        // n_inst x ncopy
  uint32_t *act;         // 2 x n_inst x nsub: queue flags, by iteration parity
  float *wown;           // n_inst x nsub: earliest time the item left dirty
  float *wpush;          // 2 x n_inst x nsub: earliest time pushed to the item
  const uint16_t *if_l;  // per interface entry: local copy id
  const uint2 *ifm;      // per submesh, wps words: interface-copy bits of 32
                         // local copies and the interface entries before them
  uint32_t *inbox;       // 2 x n_inst x n_if: earliest time pushed to an interface copy
  const uint4 *if_fo;    // per entry: first other copy, its submesh, its entry,
  const uint4 *if_os;    // index + 1 in if_os of the next other copy (0 = none)
  WorkList cur;          // work list of this iteration
  WorkList nxt;          // work list of the next iteration (requeues)
  unsigned long long *stats;  // activations, sweeps, element evaluations,
                              // iterations, algorithmic bytes
  uint32_t *old_cnt;     // counters of the list of the last iteration
  const uint32_t *start; // n_inst: iteration an instance was (re)seeded at; its
                         // window is window * (iter - start + 1)
  const uint4 *erec;        // band kernel: 48 B per element (below)
  const uint4 *adj;         // band kernel: per copy, four words of 8 incident local element ids
  const uint32_t *adj_ptr;  // copies of more than 32 elements: offset << 6 | words in adj_more
  const uint4 *adj_more;
  uint32_t nsub, ncopy, ninst, direct;
  float eps;
  const float *winst;    // n_inst: time window added per global iteration of
                         // each instance (us), 0 = off (plain FIM order)
  int32_t max_local;
  uint32_t unit, maxch;  // instances per work unit, units per submesh bucket
  uint32_t n_if, wps;    // interface entries; ifm words per submesh
  uint32_t elcap;        // band kernel: element-list entries per pass
  // LDS carve (bytes)
  uint32_t o_phin, o_flg, o_tch, o_dfr, o_e2n, o_geo, o_list, o_vlist, o_misc, o_wrt, o_ifc;
};

// The kernel's arguments where they lie (scalar loads from the constant
// segment).  The empty asm makes every call a pointer of its own, so that what
// a phase reads through it is loaded in that phase: held from the kernel's
// start, 50 pointers and counts do not fit the scalar registers and were
// spilled to lanes of vector registers (800 v_readlane in a kernel that is
// bound by vector issue).
using KArgs = const __attribute__((address_space(4))) ConvArgs *;
__device__ inline KArgs kargs() {
  KArgs k = (KArgs)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(k));
  return k;
}

struct UnitRange {
  uint32_t b, e, nb;  // units [b, e); nb workgroups of the grid run on this XCD
};

__device__ inline UnitRange xcd_range(uint32_t U, uint32_t y, uint32_t G) {
  UnitRange r;
  r.b = (uint32_t)(((uint64_t)U * y) / kXcd);
  r.e = (uint32_t)(((uint64_t)U * (y + 1)) / kXcd);
  r.nb = G > y ? (G - y + kXcd - 1) / kXcd : 0u;
  return r;
}

// Iterates the (instance, submesh) pairs of a list for one workgroup; every
// thread of the workgroup calls next() together.  `slot` is one LDS word.
struct UnitCursor {
  uint32_t s = 0, base = 0, n_in = 0, i = 0;
  bool first = true;

  // a further unit from the eighths' counters, U if none is left.  The own
  // eighth's counter is asked alone: most units come from it, and eight reads
  // for each unit cost launches of many small units 4 %.  When it has none left,
  // the first wave looks at all eight at once (one after the other took 6 us, at
  // the end of every launch); when no eighth has more units than workgroups, no
  // counter is asked.
  __device__ static uint32_t fetch(const uint32_t *cnt, uint32_t U, uint32_t *slot) {
    const uint32_t G = gridDim.x;
    if ((U + kXcd - 1) / kXcd <= G / kXcd) return U;
    if (threadIdx.x < 64) {
      const uint32_t y = (blockIdx.x + threadIdx.x) % kXcd;
      uint32_t *grab = const_cast<uint32_t *>(cnt) + kGrab + kCntLine * y;
      const UnitRange R = xcd_range(U, y, G);
      const uint32_t dyn = R.b + R.nb;
      uint32_t got = U;
      if (threadIdx.x == 0 && dyn < R.e) {
        const uint32_t v = dyn + atomicAdd(grab, 1u);
        if (v < R.e) got = v;
      }
      got = __builtin_amdgcn_readfirstlane(got);
      while (got == U) {
        // a plain read of the counter skips exhausted eighths without an atomic
        const bool open = threadIdx.x < kXcd && dyn < R.e &&
                          dyn + __hip_atomic_load(grab, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < R.e;
        const uint64_t m = __ballot(open);
        if (m == 0) break;
        const int w = __ffsll((unsigned long long)m) - 1;
        if ((int)threadIdx.x == w) {
          const uint32_t v = dyn + atomicAdd(grab, 1u);
          if (v < R.e) got = v;
        }
        got = __shfl(got, w);
      }
      if (threadIdx.x == 0) *slot = got;
    }
    __syncthreads();
    const uint32_t v = *slot;
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(v);
  }

  __device__ bool next(uint32_t &inst, uint32_t &sub, uint32_t *slot) {
    const KArgs k = kargs();
    if (++i < n_in) {
      inst = k->cur.bins[base + i];
      sub = s;
      return true;
    }
    const uint32_t U = k->cur.cnt[0];
    uint32_t u = U;
    if (first) {
      first = false;
      const UnitRange R = xcd_range(U, blockIdx.x % kXcd, gridDim.x);
      u = R.b + blockIdx.x / kXcd;
      if (u >= R.e) u = fetch(k->cur.cnt, U, slot);
    } else {
      if (k->direct) {  // no plan kernel clears the bucket
        __syncthreads();  // every thread has read its count
        if (threadIdx.x == 0) k->cur.bcnt[s] = 0u;
      }
      u = fetch(k->cur.cnt, U, slot);
    }
    if (u >= U) return false;
    const uint32_t pu = k->cur.plan[u], maxch = k->maxch, unit = k->unit;
    s = maxch == 1 ? pu : pu / maxch;
    const uint32_t j = pu - s * maxch;
    n_in = min(unit, k->cur.bcnt[s] - j * unit);
    base = s * k->ninst + j * unit;
    i = 0;
    inst = k->cur.bins[base];
    sub = s;
    return true;
  }
};

// Start of a kernel of iteration k: the next iteration's number, and, where no
// plan kernel sets them, the counters of the list that was worked through in
// iteration k - 1 and is filled in k + 1.  Returns k.
__device__ inline uint32_t start_iteration() {
  const KArgs k = kargs();
  const uint32_t iter = k->cur.cnt[kIterWord];
  if (blockIdx.x == 0) {
    if (threadIdx.x == 0) {
      k->nxt.cnt[kIterWord] = iter + 1u;
      if (k->cur.cnt[0] > 0) atomicAdd(&k->stats[3], 1ull);
    }
    if (k->direct && threadIdx.x < kIterWord) k->old_cnt[threadIdx.x] = 0u;
    if (k->direct && threadIdx.x < kXcd) k->old_cnt[kGrab + kCntLine * threadIdx.x] = 0u;
  }
  return iter;
}

__device__ inline Queue next_queue(KArgs k, uint32_t iter) {
  return Queue{WorkList{k->nxt.bcnt, k->nxt.bins, k->nxt.plan, k->nxt.cnt},
               k->act + ((iter + 1u) & 1u) * (size_t)k->ninst * k->nsub, act_tag(iter + 1u), k->nsub, k->ninst,
               k->direct};
}

// Pushes the time v of interface entry e (instance inst) to the vertex's other
// copies, for the next iteration.  A copy's time only falls, so a stale read
// of it (its item may run now) lets at most a useless push through, and the
// smallest push to a copy is always below what it reads; min, max and flags
// commute, so the merged times do not depend on any order.
__device__ inline void push_entry(KArgs k, const Queue &nq, uint32_t inst, uint32_t e, uint32_t v,
                                  uint32_t iter) {
  const uint32_t par = (iter + 1u) & 1u;
  const uint32_t *phi = reinterpret_cast<const uint32_t *>(k->phi) + (size_t)inst * k->ncopy;
  uint32_t *inbox = k->inbox + ((size_t)par * k->ninst + inst) * k->n_if;
  uint32_t *wpush = reinterpret_cast<uint32_t *>(k->wpush) + ((size_t)par * k->ninst + inst) * k->nsub;
  const uint32_t *act = nq.act + (size_t)inst * k->nsub;
  uint4 o = k->if_fo[e];  // most entries have one other copy
  for (;;) {
    // three reads in flight together
    const uint32_t cur = __hip_atomic_load(phi + o.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint32_t wcur = __hip_atomic_load(wpush + o.y, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint32_t queued = __hip_atomic_load(act + o.y, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (v < cur) {
      __hip_atomic_fetch_min(inbox + o.z, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (v < wcur) __hip_atomic_fetch_min(wpush + o.y, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (queued < nq.tag + kPushed) nq.add(inst, o.y, kPushed);
    }
    if (o.w == 0u) break;
    o = k->if_os[o.w - 1u];
  }
}

// One item as it is taken from the list.
struct Item {
  bool pushed;    // something was pushed to it
  float own;      // earliest time it left dirty itself
  float wake;     // nothing in it can act before this time
};

// its place in wpush and act of iteration iter's parity; its inbox entries
__device__ inline size_t item_parity(KArgs k, uint32_t inst, uint32_t s, uint32_t iter) {
  return ((iter & 1u) * (size_t)k->ninst + inst) * k->nsub + s;
}
__device__ inline size_t item_inbox(KArgs k, uint32_t ioff, uint32_t inst, uint32_t iter) {
  return ((iter & 1u) * (size_t)k->ninst + inst) * k->n_if + ioff;
}

__device__ inline Item take_item(KArgs k, uint32_t inst, uint32_t s, uint32_t iter) {
  Item t;
  const size_t pe = item_parity(k, inst, s, iter);
  t.own = k->wown[(size_t)inst * k->nsub + s];
  const float wp = k->wpush[pe];
  t.pushed = (k->act[pe] & 3u) == kPushed;
  t.wake = fminf(t.own, wp);
  return t;
}

// End of an item: the earliest time it left dirty itself; one thread.
__device__ inline void end_item(KArgs k, const Queue &nq, uint32_t inst, uint32_t s, uint32_t iter, bool pushed,
                                float wake) {
  k->wown[(size_t)inst * k->nsub + s] = wake;
  if (pushed) k->wpush[item_parity(k, inst, s, iter)] = F_INF;
  if (wake < F_INF) nq.add(inst, s, kQueued);
}

// An item that cannot act in this iteration stays queued.  What was pushed to
// it goes into the copies' times now (the inbox of this parity is written
// again in the next iteration); pushes that lower nothing leave no trace.
// low: one LDS word.  Every thread of the workgroup calls it.
template <int BS>
__device__ inline void defer_item(const SubInfo &si, const Item &t, uint32_t inst, uint32_t s, uint32_t iter,
                                  uint32_t *low) {
  const KArgs k = kargs();
  const Queue nq = next_queue(k, iter);
  if (!t.pushed) {
    if (threadIdx.x == 0) nq.add(inst, s, kQueued);
    return;
  }
  __syncthreads();  // the LDS word is free
  if (threadIdx.x == 0) *low = __float_as_uint(t.own);
  __syncthreads();
  uint32_t *phi = reinterpret_cast<uint32_t *>(k->phi) + (size_t)inst * k->ncopy + si.coff;
  uint32_t *inbox = k->inbox + item_inbox(k, si.ioff, inst, iter);
  for (uint32_t j = threadIdx.x; j < si.ni; j += BS) {
    const uint32_t v = inbox[j];
    if (v == __float_as_uint(F_INF)) continue;
    inbox[j] = __float_as_uint(F_INF);
    const uint32_t l = k->if_l[si.ioff + j];
    if (v < phi[l]) {
      phi[l] = v;
      k->dirty[(size_t)inst * k->ncopy + si.coff + l] = 1;
      atomicMin(low, v);
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) end_item(k, nq, inst, s, iter, true, __uint_as_float(*low));
}

// the time of an interface copy of an item that was pushed to: the smaller of
// its own v and its inbox entry's, which is emptied; true if lowered
__device__ inline bool merge_inbox(uint32_t *entry, float *phi, float &v) {
  const float x = __uint_as_float(*entry);
  if (!(x < F_INF)) return false;
  *entry = __float_as_uint(F_INF);
  if (!(x < v)) return false;
  v = x;
  *phi = x;
  return true;
}

// Pushes the interface copies lowered by this activation (bits in tch), found
// through the interface list.
template <int BS>
__device__ inline void push_lowered_scan(const Queue &nq, const SubInfo &si, uint32_t inst, uint32_t iter,
                                         const uint32_t *tch, const float *phi_l) {
  const KArgs k = kargs();
  for (uint32_t j = threadIdx.x; j < si.ni; j += BS) {
    const uint32_t l = k->if_l[si.ioff + j];
    if (flag_at(tch, l)) push_entry(k, nq, inst, si.ioff + j, __float_as_uint(phi_l[l]), iter);
  }
}

// The staged converge kernel (fim_opts.staged): one workgroup per work item
// (instance, submesh) copies the submesh's elements (nodes + geometry) into
// LDS and finds the active elements by scanning them every sweep.
template <int BS>
__global__ __launch_bounds__(BS) void k_conv_compute(ConvArgs a) {
  extern __shared__ __align__(16) unsigned char lds[];
  float *phi_l = reinterpret_cast<float *>(lds);
  uint32_t *phi_n = reinterpret_cast<uint32_t *>(lds + a.o_phin);
  uint32_t *flg = reinterpret_cast<uint32_t *>(lds + a.o_flg);
  uint32_t *tch = reinterpret_cast<uint32_t *>(lds + a.o_tch);
  uint32_t *dfr = reinterpret_cast<uint32_t *>(lds + a.o_dfr);
  uint2 *el = reinterpret_cast<uint2 *>(lds + a.o_e2n);
  float *gl = reinterpret_cast<float *>(lds + a.o_geo);
  uint16_t *elist = reinterpret_cast<uint16_t *>(lds + a.o_list);
  uint32_t *misc = reinterpret_cast<uint32_t *>(lds + a.o_misc);
  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

  UnitCursor cursor;
  const uint32_t iter_now = start_iteration();
  unsigned long long sweeps = 0, evals = 0, acts = 0, abytes = 0, vupd = 0;

  uint32_t inst, s;
  while (cursor.next(inst, s, &misc[4])) {
    const float wi = a.winst[inst];
    // time window of this iteration: flagged vertices later than W wait
    const float W = wi > 0.0f ? wi * (float)(iter_now - a.start[inst] + 1u) : F_INF;
    const SubInfo si = a.sub[s];
    const Item item = take_item(kargs(), inst, s, iter_now);
    const size_t cb = (size_t)inst * a.ncopy + si.coff;
    const uint32_t nn = si.nn, ne = si.ne;
    const uint32_t nv64 = (nn + 63u) & ~63u;
    // nothing in this submesh can act before the window reaches its wake
    // time: keep it queued without staging anything
    if (item.wake > W) {
      defer_item<BS>(si, item, inst, s, iter_now, &misc[5]);
      continue;
    }
    // stage vertex times and dirty flags
    for (uint32_t l0 = 0; l0 < nv64; l0 += BS) {
      const uint32_t l = l0 + tid;
      bool d = false, late = false;
      if (l < nn) {
        float v = a.phi[cb + l];
        d = a.dirty[cb + l] != 0;
        if (d) a.dirty[cb + l] = 0;
        if (item.pushed) {
          const uint2 w = a.ifm[(size_t)s * a.wps + (l >> 5)];
          if ((w.x >> (l & 31)) & 1u)
            d |= merge_inbox(a.inbox + item_inbox(kargs(), si.ioff, inst, iter_now) + w.y +
                                 __popc(w.x & ((1u << (l & 31)) - 1u)),
                             a.phi + cb + l, v);
        }
        phi_l[l] = v;
        phi_n[l] = __float_as_uint(v);
        late = d && v > W;
        d = d && !late;
      }
      const uint64_t m = __ballot(d), md = __ballot(late);
      const uint32_t wb = l0 + wave * 64;
      if (wb < nv64) {
        if (lane == 0) flg[wb >> 5] = (uint32_t)m;
        if (lane == 1) flg[(wb >> 5) + 1] = (uint32_t)(m >> 32);
        if (lane == 2) tch[wb >> 5] = 0u;
        if (lane == 3) tch[(wb >> 5) + 1] = 0u;
        if (lane == 4) dfr[wb >> 5] = (uint32_t)md;
        if (lane == 5) dfr[(wb >> 5) + 1] = (uint32_t)(md >> 32);
      }
    }
    const float *rs = a.rscale + 4 * (size_t)inst;
    // stage elements (geometry scaled by the instance's regional factor)
    for (uint32_t e = tid; e < ne; e += BS) {
      const size_t ge = (size_t)si.eoff + e;
      el[e] = a.e2n[ge];
      const float sc = rs[a.ereg[ge] & 3];
      const float2 *g2 = reinterpret_cast<const float2 *>(a.geo + 6 * ge);
      const float2 x0 = g2[0], x1 = g2[1], x2 = g2[2];
      float *o = gl + 6 * e;
      o[0] = x0.x * sc;
      o[1] = x0.y * sc;
      o[2] = x1.x * sc;
      o[3] = x1.y * sc;
      o[4] = x2.x * sc;
      o[5] = x2.y * sc;
    }
    __syncthreads();

    int it = 0;
    bool capped = false;
    for (;;) {
      if (tid == 0) misc[0] = 0u;
      __syncthreads();
      // active elements: any node flagged (wave ballot + per-wave base)
      for (uint32_t e0 = 0; e0 < ne; e0 += BS) {
        const uint32_t e = e0 + tid;
        bool on = false;
        if (e < ne) {
          const uint2 q = el[e];
          on = flag_at(flg, q.x & 0xffffu) || flag_at(flg, q.x >> 16) ||
               flag_at(flg, q.y & 0xffffu) || flag_at(flg, q.y >> 16);
        }
        const uint64_t m = __ballot(on);
        uint32_t base = 0;
        if (lane == 0 && m) base = atomicAdd(&misc[0], (uint32_t)__popcll(m));
        base = __shfl(base, 0);
        if (on) elist[base + __popcll(m & lanes_below())] = (uint16_t)e;
      }
      __syncthreads();
      const uint32_t nact = misc[0];
      if (nact == 0) break;
      if ((a.max_local > 0 && it >= a.max_local) || it >= kHardLocalCap) {
        capped = true;
        break;
      }
      ++it;
      evals += nact;
      // candidates of the active elements
      for (uint32_t i = tid; i < nact; i += BS) {
        const uint32_t e = elist[i];
        const uint2 q = el[e];
        float g[6];
#pragma unroll
        for (int k = 0; k < 6; ++k) g[k] = gl[6 * e + k];
        const uint32_t nd[4] = {q.x & 0xffffu, q.x >> 16, q.y & 0xffffu, q.y >> 16};
        float ph[4];
        int f[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          ph[k] = phi_l[nd[k]];
          f[k] = flag_at(flg, nd[k]) ? 1 : 0;
        }
        const int nf = f[0] + f[1] + f[2] + f[3];
        // every candidate of a target is at least the earliest other node
        // plus the target's metric height above the opposite face: evaluate
        // only targets with a flagged other node that can still improve
        const size_t gh = (size_t)si.eoff + e;
        const float hs = csqrt(rs[a.ereg[gh] & 3]);
        const float4 hh = a.hgt[gh];
        const float h[4] = {hh.x * hs, hh.y * hs, hh.z * hs, hh.w * hs};
        if (nf - f[0] > 0 && ph[0] > fminf(ph[1], fminf(ph[2], ph[3])) + h[0]) {
          const float c = cand_exact<0, float>(g, ph, F_INF);
          ++vupd;
          if (c < ph[0]) atomicMin(&phi_n[nd[0]], __float_as_uint(c));
        }
        if (nf - f[1] > 0 && ph[1] > fminf(ph[0], fminf(ph[2], ph[3])) + h[1]) {
          const float c = cand_exact<1, float>(g, ph, F_INF);
          ++vupd;
          if (c < ph[1]) atomicMin(&phi_n[nd[1]], __float_as_uint(c));
        }
        if (nf - f[2] > 0 && ph[2] > fminf(ph[0], fminf(ph[1], ph[3])) + h[2]) {
          const float c = cand_exact<2, float>(g, ph, F_INF);
          ++vupd;
          if (c < ph[2]) atomicMin(&phi_n[nd[2]], __float_as_uint(c));
        }
        if (nf - f[3] > 0 && ph[3] > fminf(ph[0], fminf(ph[1], ph[2])) + h[3]) {
          const float c = cand_exact<3, float>(g, ph, F_INF);
          ++vupd;
          if (c < ph[3]) atomicMin(&phi_n[nd[3]], __float_as_uint(c));
        }
      }
      __syncthreads();
      // accept: new flags = significant decreases (reference criterion
      // |old-new| >= eps (1 + (old+new)/2), cuda_fim.cu:2154)
      for (uint32_t l0 = 0; l0 < nv64; l0 += BS) {
        const uint32_t l = l0 + tid;
        bool sig = false, dec = false, late = false;
        if (l < nn) {
          const float ov = phi_l[l];
          const float nv = __uint_as_float(phi_n[l]);
          if (nv < ov) {
            phi_l[l] = nv;
            dec = true;
            sig = (ov - nv) >= a.eps * (1.0f + 0.5f * (ov + nv));
            late = sig && nv > W;
            sig = sig && !late;
          }
        }
        const uint64_t m = __ballot(sig), mt = __ballot(dec), md = __ballot(late);
        const uint32_t wb = l0 + wave * 64;
        if (wb < nv64) {
          if (lane == 0) flg[wb >> 5] = (uint32_t)m;
          if (lane == 1) flg[(wb >> 5) + 1] = (uint32_t)(m >> 32);
          if (lane == 2) tch[wb >> 5] |= (uint32_t)mt;
          if (lane == 3) tch[(wb >> 5) + 1] |= (uint32_t)(mt >> 32);
          // a deferred vertex that is now a source leaves the deferred set
          if (lane == 4) dfr[wb >> 5] = (dfr[wb >> 5] & ~(uint32_t)m) | (uint32_t)md;
          if (lane == 5) dfr[(wb >> 5) + 1] = (dfr[(wb >> 5) + 1] & ~(uint32_t)(m >> 32)) | (uint32_t)(md >> 32);
        }
      }
      __syncthreads();
    }
    sweeps += it;
    acts += it > 0;
    // algorithmic bytes of the activation: copies read and written (phi 4+4,
    // flag 1+1), interface entries (index 4, read 4, write 4) and the
    // element data (nodes 8 + geometry 24)
    if (it > 0) abytes += 32ull * ne + 10ull * nn + 12ull * si.ni;
    // write back decreased copies and push the lowered interface copies.
    // Deferred vertices (and sources left by the sweep cap) stay dirty and
    // the submesh is queued for the next iteration.
    if (tid == 0) misc[1] = __float_as_uint(F_INF);
    __syncthreads();
    for (uint32_t l = tid; l < nn; l += BS) {
      if (flag_at(tch, l)) a.phi[cb + l] = phi_l[l];
      if (flag_at(dfr, l) || (capped && flag_at(flg, l))) {
        a.dirty[cb + l] = 1;
        atomicMin(&misc[1], __float_as_uint(phi_l[l]));
      }
    }
    const Queue nq = next_queue(kargs(), iter_now);
    push_lowered_scan<BS>(nq, si, inst, iter_now, tch, phi_l);
    __syncthreads();
    if (tid == 0) end_item(kargs(), nq, inst, s, iter_now, item.pushed, __uint_as_float(misc[1]));
    __syncthreads();
  }
  if (tid == 0 && acts) {
    atomicAdd(&a.stats[0], acts);
    atomicAdd(&a.stats[1], sweeps);
    atomicAdd(&a.stats[2], evals);
    atomicAdd(&a.stats[4], abytes);
  }
  for (int off = 32; off > 0; off >>= 1) vupd += __shfl_xor(vupd, off);
  if (lane == 0 && vupd) atomicAdd(&a.stats[5], vupd);
}

// Element record of the band kernel, three 16-byte words per element:
//   [0] nodes 0,1 (u16 each; bit 15 and bit 31 carry the region id's bits 0
//       and 1), nodes 2,3 (u16 each), geometry e12 e13 (f32)
//   [1] geometry e23 e14 e24 e34 (f32)
//   [2] candidate bounds: for the targets T = 0..3, n . (x_T - x_i) of the
//       nodes i = T+1, T+2, T+3 (ElementBounds), their scale (f32)
// Local copy ids are below 2^15, so the two region bits are free.

// The targets with a source among the other nodes whose candidates can still
// lower them: a candidate is at least min_i (p_i + n . u_i).  With n along the
// target's distance from the centroid of the opposite face this keeps 33 % of
// the targets of a settled slab; the plane's height over that face (n
// perpendicular to it, four floats, the bound before) 50 %, two directions
// 23 %, three 20 %.  One direction in bytes is what fits the record's 48 B: the
// records of the fronts that an XCD works on just about fill its L2, and a
// record of 80 B for two directions lost in L2 misses (twice as many) what
// fewer candidates saved.  Three directions from the squared lengths, without
// a table, take 100 instructions and 30 more registers (28 % slower).
__device__ inline uint32_t live_targets(const uint4 b, float hs, const float ph[4], const int f[4]) {
  const uint32_t w[3] = {b.x, b.y, b.z};
  float v[4];
  cand_bounds32(w, __uint_as_float(b.w) * hs, ph, v);
  const int nf = f[0] + f[1] + f[2] + f[3];
  uint32_t tm = 0;
#pragma unroll
  for (int T = 0; T < 4; ++T) tm |= (nf - f[T] > 0 && ph[T] > v[T]) ? 1u << T : 0u;
  return tm;
}

// marks the two local elements of one adjacency word in the LDS bitmask; the
// atomics return nothing, the list is built from the bitmask
__device__ inline void mark_word(uint32_t *emark, uint32_t w) {
  atomicOr(&emark[(w & 0xffffu) >> 5], 1u << (w & 31u));
  atomicOr(&emark[w >> 21], 1u << ((w >> 16) & 31u));
}

__device__ inline void mark_chunk(uint32_t *emark, const uint4 q) {
  mark_word(emark, q.x);
  mark_word(emark, q.y);
  mark_word(emark, q.z);
  mark_word(emark, q.w);
}

// marks the incident elements of local copy c.  Every copy has four 16-byte
// words of eight ids in a row, found without a pointer (a dependent load from
// L2 less per sweep) and filled up with its first element, which may be marked
// any number of times; a wave skips words that only repeat.  A copy of more
// than 32 elements has kAdjMore in place of the last id and lists the others
// through adj_ptr.
constexpr uint32_t kAdjMore = 0xffffu;
__device__ inline void mark_incident(const uint4 *adj, const uint32_t *adj_ptr, const uint4 *adj_more, uint32_t c,
                                     uint32_t *emark) {
  const uint4 *ch = adj + 4 * (size_t)c;
  const uint4 q0 = ch[0], q1 = ch[1], q2 = ch[2];
  uint4 q3 = ch[3];
  const uint32_t first = q0.x & 0xffffu;
  mark_chunk(emark, q0);
  mark_chunk(emark, q1);
  if (__any((q2.x & 0xffffu) != first)) mark_chunk(emark, q2);
  if (__any((q3.x & 0xffffu) != first)) {
    const bool more = q3.w >> 16 == kAdjMore;
    if (more) q3.w = (q3.w & 0xffffu) | first << 16;
    mark_chunk(emark, q3);
    if (more) {
      const uint32_t ap = adj_ptr[c];
      for (uint32_t k = 0; k < (ap & 63u); ++k) mark_chunk(emark, adj_more[(ap >> 6) + k]);
    }
  }
}

// sum over the wave of n < 2^BITS, one ballot per bit; every lane of the
// wave must be active
template <int BITS>
__device__ inline uint32_t wave_sum_small(uint32_t n) {
  uint32_t s = 0;
#pragma unroll
  for (int b = 0; b < BITS; ++b) s += (uint32_t)__popcll(__ballot((n >> b) & 1u)) << b;
  return s;
}

// appends the lanes with `pred` (vertex l) to list[*cnt ...], one LDS atomic
// per wave
__device__ inline void wave_append(bool pred, uint32_t l, uint16_t *list, uint32_t *cnt) {
  const uint64_t m = __ballot(pred);
  uint32_t base = 0;
  if ((threadIdx.x & 63) == 0 && m) base = atomicAdd(cnt, (uint32_t)__popcll(m));
  base = __builtin_amdgcn_readfirstlane(base);  // every lane of the wave is active
  if (pred) list[base + __popcll(m & lanes_below())] = (uint16_t)l;
}

// Unstaged converge kernel.  Per sweep it touches only the band that is
// active, in three steps, a barrier after each:
//   mark: the sources (a compact list) mark their incident elements through
//     the vertex -> element adjacency in an LDS bitmask (atomics without
//     return);
//   evaluate: each wave lists the marked elements of its words of the bitmask
//     and computes their candidates from L2-resident element records; LDS
//     atomicMin winners set a "written" bit;
//   accept: each written vertex takes its new time; a significant decrease
//     (reference criterion, cuda_fim.cu:2154) makes it a source of the next
//     sweep, or a deferred vertex if it lies beyond the window.
// Element data never enters LDS.  PAIRS evaluates (element, target) pairs
// in full rounds of 64 instead of an element's four targets per lane (local
// element ids below 2^14).  WPE is the number of waves per SIMD the register
// budget is sized for (512 / WPE VGPRs): the launch picks the one that the LDS
// carve allows anyway, so registers left over by a large submesh's LDS footprint
// are used instead of spilled; with WPE <= 4 a wave works on two rounds of
// pairs side by side (ILP).
//
// What bounds it: at 512 instances a launch, vector issue (75 % of one wave
// instruction per SIMD and 4 cycles, 5.2e8 instructions in 1,120 us, 10.5 per
// candidate), while waves wait 60 % of their cycles; with 128 instances, or a
// single one, those waits (65-70 %: L2 misses of records and times, LDS round
// trips, barriers), vector issue being 41-50 %.  Cycles per item of the 2M slab (256 x 2
// instances, 2816 copies; a single solve, 1024 copies): staging 24k / 6.9k,
// mark 13k / 7k, list and evaluate 79k / 27k, accept 17k / 5k, write-back 6k /
// 3k, push 3k / 2.5k, next item 6k / 2.6k; 155k / 63k in all before the lists
// were split over the waves, blocks with nothing to do were skipped by whole
// waves and the adjacency lost its pointer.  A single solve's iteration lasts
// as long as its longest item (107k cycles), a batch's launch is 1,450 items
// deep.  Loading the next 64 listed elements ahead of the current ones gained
// nothing.
//
// GATHER: a sweep of few sources marks too few elements to give every wave a
// full round, and eight nearly empty rounds cost as many instructions as eight
// full ones.  Where the CUs are busy (the units fill half of the workgroups or
// more), submeshes of up to kGatherFull elements a wave have such a sweep
// listed by one wave for every 32 sources (about 20 elements each): 271 maps of
// a 44k-tet mesh in submeshes of 769 copies, workgroups of 512, 16.6 ms against
// 20.8 with all waves; 423 maps of a 180k-tet shell in two contexts 74 against
// 93.  With the line at 1,280 elements a wave some batches gained another 10 %,
// others lost 20 % (149 maps on 42 submeshes 42 against 34 ms): their sweeps are
// a chain of rounds, and 512 maps of the 2M-tet slab take 228 instead of 205 ms
// with few waves.  So do launches that leave the CUs half empty.  Up to
// kGatherAlways elements a wave, a wave has hardly a word of the bitmask, and
// few waves list at any load (a single solve on 3,534 submeshes of 256 copies:
// 9.0 against 10.2 ms).
template <int BS, int WPE, bool PAIRS, bool GATHER>
__global__ __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(WPE, 8))) void k_conv_band(ConvArgs) {
  extern __shared__ __align__(16) unsigned char lds[];
  const KArgs k0 = kargs();
  float *phi_l = reinterpret_cast<float *>(lds);
  uint32_t *phi_n = reinterpret_cast<uint32_t *>(lds + k0->o_phin);
  uint32_t *flg = reinterpret_cast<uint32_t *>(lds + k0->o_flg);  // sources of the sweep
  uint32_t *tch = reinterpret_cast<uint32_t *>(lds + k0->o_tch);  // decreased this activation
  uint32_t *dfr = reinterpret_cast<uint32_t *>(lds + k0->o_dfr);  // flagged, beyond the window
  uint32_t *wrt = reinterpret_cast<uint32_t *>(lds + k0->o_wrt);  // lowered in this sweep
  uint32_t *ifc = reinterpret_cast<uint32_t *>(lds + k0->o_ifc);  // interface copies
  uint32_t *ipre = ifc + k0->wps;  // interface entries before each word
  uint32_t *emark = reinterpret_cast<uint32_t *>(lds + k0->o_e2n);
  uint32_t *eseen = reinterpret_cast<uint32_t *>(lds + k0->o_geo);
  uint16_t *elist = reinterpret_cast<uint16_t *>(lds + k0->o_list);
  uint16_t *vlist = reinterpret_cast<uint16_t *>(lds + k0->o_vlist);
  // misc: [0] element evaluations, [2] listed sources, [3] distinct elements,
  // [4] work cursor, [5] earliest deferred time, [6], [7] lowered interface copies,
  // [8..11] the instance's region factors, [12..19] launch counters
  uint32_t *misc = reinterpret_cast<uint32_t *>(lds + k0->o_misc);
  const float *rsl = reinterpret_cast<const float *>(misc + 8);
  constexpr uint32_t NW = BS / 64, LNW = NW == 8 ? 3 : NW == 4 ? 2 : NW == 2 ? 1 : 0;
  constexpr int ILP = WPE <= 4 ? 2 : 1;
  uint32_t tid = threadIdx.x;
  const uint32_t lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  UnitCursor cursor;
  const uint32_t iter_now = start_iteration();
  const bool full = GATHER && 2u * k0->cur.cnt[0] >= gridDim.x;
  // counters of the launch (thread 0): activations, sweeps, element
  // evaluations, algorithmic bytes
  unsigned long long *ctr = reinterpret_cast<unsigned long long *>(misc + 12);
  if (tid == 0) ctr[0] = ctr[1] = ctr[2] = ctr[3] = 0ull;
  uint32_t vupd = 0;  // candidates of the lane in this launch

  uint32_t npush = 6;  // misc word of the push count, 6 and 7 in turn
  uint32_t inst, s;
  while (cursor.next(inst, s, &misc[4])) {
    const KArgs ks = kargs();
    tid = fresh(tid);
    const float wi = ks->winst[inst];
    // time window of this iteration: flagged vertices later than W wait
    const float W = wi > 0.0f ? wi * (float)(iter_now - ks->start[inst] + 1u) : F_INF;
    const SubInfo si = ks->sub[s];
    const Item item = take_item(ks, inst, s, iter_now);
    const uint32_t nn = si.nn, ne = si.ne;
    const uint32_t nv64 = (nn + 63u) & ~63u;
    const uint32_t new32 = (ne + 31u) >> 5;  // element bitmask words
    const bool gather = GATHER && ne <= (full ? kGatherFull : kGatherAlways) * NW;
    if (item.wake > W) {
      defer_item<BS>(si, item, inst, s, iter_now, &misc[5]);
      continue;
    }
    const uint2 *ifm_g = ks->ifm + (size_t)s * ks->wps;
    for (uint32_t k = tid; k < new32; k += BS) {
      emark[k] = 0u;
      eseen[k] = 0u;
    }
    if (tid == 0) {
      misc[0] = 0u;
      misc[2] = 0u;
      misc[3] = 0u;
      misc[5] = __float_as_uint(F_INF);
      misc[npush] = 0u;
    }
    for (uint32_t q = tid; q < nv64 / 32; q += BS) {
      const uint2 fw = ifm_g[q];
      ifc[q] = fw.x;
      ipre[q] = fw.y;
    }
    if (tid < 4) misc[8 + tid] = __float_as_uint(ks->rscale[4 * (size_t)inst + tid]);
    __syncthreads();
    // stage vertex times; dirty flags split into sources and deferred
    float *phi_g = ks->phi + (size_t)inst * ks->ncopy + si.coff;
    uint8_t *dirty_g = ks->dirty + (size_t)inst * ks->ncopy + si.coff;
    uint32_t *inbox_g = ks->inbox + item_inbox(ks, si.ioff, inst, iter_now);
    // the loads of a wave's next block of 64 copies are issued before the
    // current one is used
    struct Staged {
      float v, x;  // time, time pushed
      uint32_t d;
    };
    auto fetch = [&](uint32_t l) {
      Staged g{F_INF, F_INF, 0u};
      if (l < nn) {
        g.v = phi_g[l];
        g.d = dirty_g[l];
        if (item.pushed && flag_at(ifc, l)) g.x = __uint_as_float(inbox_g[ipre[l >> 5] + bits_below(ifc, l)]);
      }
      return g;
    };
    Staged next = fetch(tid);
    for (uint32_t l0 = 0; l0 < nv64; l0 += BS) {
      const uint32_t l = l0 + tid;
      const uint32_t wb = l0 + wave * 64;
      if (wb < nv64) {
        const Staged g = next;
        next = fetch(l + BS);
        bool d = g.d != 0;
        float v = g.v;
        if (d) dirty_g[l] = 0;
        if (g.x < F_INF) {  // merged into the time, and emptied
          inbox_g[ipre[l >> 5] + bits_below(ifc, l)] = __float_as_uint(F_INF);
          if (g.x < v) {
            v = g.x;
            phi_g[l] = v;
            d = true;
          }
        }
        if (l < nn) {
          phi_l[l] = v;
          phi_n[l] = __float_as_uint(v);
        }
        const bool late = d && v > W;
        d = d && !late;
        const uint64_t m = __ballot(d), md = __ballot(late);
        const uint32_t k = wb >> 5;
        if (lane == 0) {
          flg[k] = (uint32_t)m;
          flg[k + 1] = (uint32_t)(m >> 32);
          dfr[k] = (uint32_t)md;
          dfr[k + 1] = (uint32_t)(md >> 32);
        }
        if (lane == 1) {
          tch[k] = 0u;
          tch[k + 1] = 0u;
          wrt[k] = 0u;
          wrt[k + 1] = 0u;
        }
        wave_append(d, l, vlist, &misc[2]);
      }
    }
    __syncthreads();

    uint32_t it = 0, evals = 0;
    tid = fresh(tid);
    bool capped = false;
    const KArgs kw = kargs();
    const uint32_t wcap = kw->elcap / NW;
    uint16_t *wlist = elist + wave * wcap;
    const int32_t max_local = kw->max_local;
    const float eps = kw->eps;
    const uint4 *erec = kw->erec + 3 * (size_t)si.eoff, *adj = kw->adj + 4 * (size_t)si.coff, *adj_more = kw->adj_more;
    const uint32_t *adj_ptr = kw->adj_ptr + si.coff;
    for (;;) {
      const uint32_t nsrc = misc[2];
      if (nsrc == 0) break;
      if ((max_local > 0 && it >= (uint32_t)max_local) || it >= (uint32_t)kHardLocalCap) {
        capped = true;
        break;
      }
      ++it;
      // mark the elements incident to the sources
      for (uint32_t i = tid; i < nsrc; i += BS) mark_incident(adj, adj_ptr, adj_more, vlist[i], emark);
      __syncthreads();
      if (tid == 0) misc[2] = 0u;  // every thread has read the source count
      // Each wave, or each of a few, lists and evaluates the marked elements of
      // its own words of the bitmask (every NW-th: neighbours go to different
      // waves), without a barrier in between.  Lane i holds word i: offsets from a wave prefix sum
      // of the word counts (<= 32, six bits) with one ballot per bit, then two
      // words at a time, a lane per bit.  A pass lists at most wcap elements;
      // what is left of the words stays marked for the next pass (the sweep
      // still evaluates every marked element against the same times).
      uint32_t lw = LNW;  // 2^lw waves
      if (GATHER && gather && nsrc < 128u)
        lw = __builtin_amdgcn_readfirstlane(min(LNW, nsrc < 32u ? 0u : nsrc < 64u ? 1u : 2u));
      const uint32_t nw = 1u << lw, nww = wave < min(nw, new32) ? (new32 - wave + nw - 1) >> lw : 0u;
      for (uint32_t i0 = 0; i0 < nww;) {
        const uint32_t kw = wave + ((i0 + lane) << lw);
        const uint32_t rest = i0 + lane < nww ? emark[kw] : 0u;
        const uint32_t n = __popc(rest);
        uint32_t pos = 0, tot = 0;
#pragma unroll
        for (int b = 0; b < 6; ++b) {
          const uint64_t m = __ballot((n >> b) & 1u);
          pos += (uint32_t)__popcll(m & lanes_below()) << b;
          tot += (uint32_t)__popcll(m) << b;
        }
        const uint32_t word0 = i0;
        uint32_t take = rest;
        if (tot > wcap) {  // uniform: the list is full after some word's first bits
          uint32_t room = pos < wcap ? wcap - pos : 0u;
          take = 0u;
          for (uint32_t left = rest; left && room; --room) {
            take |= left & (0u - left);
            left &= left - 1u;
          }
        } else {
          i0 += 64;
        }
        if (tot == 0) continue;  // uniform
        if (rest) {
          emark[kw] = rest & ~take;
          eseen[kw] |= take;
        }
        for (uint64_t some = __ballot(take != 0u); some;) {
          const int i1 = __ffsll((unsigned long long)some) - 1;
          some &= some - 1;
          const bool two = some != 0;
          const int i2 = two ? __ffsll((unsigned long long)some) - 1 : i1;
          some &= some - 1;  // 0 stays 0
          const uint32_t t1 = __builtin_amdgcn_readlane(take, i1), t2 = __builtin_amdgcn_readlane(take, i2);
          const uint32_t p1 = __builtin_amdgcn_readlane(pos, i1), p2 = __builtin_amdgcn_readlane(pos, i2);
          const bool hi = lane >= 32;
          const uint32_t bit = lane & 31u, tw = hi ? (two ? t2 : 0u) : t1;
          if ((tw >> bit) & 1u)
            wlist[(hi ? p2 : p1) + __popc(tw & ((1u << bit) - 1u))] =
                (uint16_t)((wave + ((word0 + (hi ? i2 : i1)) << lw)) * 32 + bit);
        }
        __builtin_amdgcn_wave_barrier();
        const uint32_t nact = min(tot, wcap);
        evals += nact;
        // candidates of the listed elements
        if constexpr (PAIRS) {
          // (element, target) pairs: a pass over 64 listed elements per wave
          // keeps the targets that pass the bound test and queues them in a
          // wave-private ring (LDS, in the source list's space, idle until the
          // accept step); full rounds of 64 pairs then evaluate one target
          // per lane, so no lane idles on a pruned target
          constexpr uint32_t kRing = pair_ring(ILP);
          uint16_t *pq = vlist + wave * kRing;
          uint32_t qh = 0, qn = 0;  // ring head and fill, uniform across the wave
          for (uint32_t c0 = 0;; c0 += 64) {
            const bool more = c0 < nact;  // uniform across the wave
            if (more) {
              const uint32_t i = c0 + lane;
              uint32_t tm = 0, e = 0;
              if (i < nact) {
                e = wlist[i];
                const uint4 *rec = erec + 3 * e;
                const uint4 r0 = rec[0], r2 = rec[2];
                const float hs = csqrt(rsl[((r0.x >> 15) & 1u) | ((r0.x >> 30) & 2u)]);
                const uint32_t nd[4] = {r0.x & 0x7fffu, (r0.x >> 16) & 0x7fffu, r0.y & 0xffffu,
                                        r0.y >> 16};
                float ph[4];
                int f[4];
  #pragma unroll
                for (int k = 0; k < 4; ++k) {
                  ph[k] = phi_l[nd[k]];
                  f[k] = flag_at(flg, nd[k]) ? 1 : 0;
                }
                tm = live_targets(r2, hs, ph, f);
              }
  #pragma unroll
              for (uint32_t T = 0; T < 4; ++T) {
                const bool p = (tm >> T) & 1u;
                const uint64_t m = __ballot(p);
                if (p) {
                  uint32_t pos = qh + qn + (uint32_t)__popcll(m & lanes_below());
                  if (pos >= kRing) pos -= kRing;
                  pq[pos] = (uint16_t)(e | (T << 14));
                }
                qn += (uint32_t)__popcll(m);
              }
              __builtin_amdgcn_wave_barrier();
            }
            while (qn >= 64u * ILP || (!more && qn > 0u)) {
              const uint32_t take = min(qn, 64u * ILP);
              float gp[ILP][6], pp[ILP][4];
              uint32_t nt[ILP];
              auto load = [&](int u) {
                uint32_t pos = qh + 64u * u + lane;
                if (pos >= kRing) pos -= kRing;
                // a lane without a pair works on element 0 and drops the result
                const uint32_t code = 64u * u + lane < take ? pq[pos] : 0u;
                const uint32_t e = code & 0x3fffu, T = code >> 14;
                const uint4 *rec = erec + 3 * e;
                const uint4 r0 = rec[0], r1 = rec[1];
                const float sc = rsl[((r0.x >> 15) & 1u) | ((r0.x >> 30) & 2u)];
                const float g[6] = {__uint_as_float(r0.z) * sc, __uint_as_float(r0.w) * sc,
                                    __uint_as_float(r1.x) * sc, __uint_as_float(r1.y) * sc,
                                    __uint_as_float(r1.z) * sc, __uint_as_float(r1.w) * sc};
                // relabel so that the target is node 3 (others T+1, T+2, T+3):
                // the same candidate as for node position T.  The node ids
                // rotate as one 64-bit word.
                const uint64_t ids = (uint64_t)r0.y << 32 | (r0.x & 0x7fff7fffu);
                const uint64_t rot = ids >> (16u * T) | ids << ((64u - 16u * T) & 63u);
                const bool t1 = T & 1u, t2 = T & 2u;
                auto sel = [&](float x0, float x1, float x2, float x3) {
                  return t2 ? (t1 ? x3 : x2) : (t1 ? x1 : x0);
                };
                // edge (i,j) of the relabelled element for T = 0, 1, 2, 3
                gp[u][0] = sel(g[2], g[5], g[3], g[0]);
                gp[u][1] = t1 ? g[1] : g[4];
                gp[u][2] = sel(g[5], g[3], g[0], g[2]);
                gp[u][3] = sel(g[0], g[2], g[5], g[3]);
                gp[u][4] = t1 ? g[4] : g[1];
                gp[u][5] = sel(g[3], g[0], g[2], g[5]);
                nt[u] = (uint32_t)rot & 0xffffu;
                pp[u][0] = phi_l[(uint32_t)rot >> 16];
                pp[u][1] = phi_l[(uint32_t)(rot >> 32) & 0xffffu];
                pp[u][2] = phi_l[(uint32_t)(rot >> 48)];
                pp[u][3] = phi_l[nt[u]];
              };
              auto value = [&](int u) {
                float sq[6], rc[6];
  #pragma unroll
                for (int k = 0; k < 3; ++k) {
                  rc[k] = __builtin_amdgcn_rcpf(gp[u][k]);
                  sq[k + 3] = csqrt(gp[u][k + 3]);
                  sq[k] = 0.0f;
                  rc[k + 3] = 0.0f;
                }
                return cand_exact_sh<3, float>(gp[u], sq, rc, pp[u], F_INF);
              };
              auto commit = [&](int u, float c) {
                ++vupd;
                if (c < pp[u][3]) {
                  // below the staged time: the minimum ends below it too, so the
                  // written bit needs no returned value
                  atomicMin(&phi_n[nt[u]], __float_as_uint(c));
                  atomicOr(&wrt[nt[u] >> 5], 1u << (nt[u] & 31));
                }
              };
              if constexpr (ILP == 1) {
                if (lane < take) {
                  load(0);
                  commit(0, value(0));
                }
              } else {
                load(0);
                load(1);
                const float c0 = value(0), c1 = value(1);
                if (lane < take) commit(0, c0);
                if (64u + lane < take) commit(1, c1);
              }
              qh += take;
              if (qh >= kRing) qh -= kRing;
              qn -= take;
              __builtin_amdgcn_wave_barrier();
            }
            if (!more) break;
          }
        } else {
          for (uint32_t i = lane; i < nact; i += 64) {
            const uint32_t e = wlist[i];
            const uint4 r0 = erec[3 * e], r1 = erec[3 * e + 1];
            const float sc = rsl[((r0.x >> 15) & 1u) | ((r0.x >> 30) & 2u)];
            const float g[6] = {__uint_as_float(r0.z) * sc, __uint_as_float(r0.w) * sc,
                                __uint_as_float(r1.x) * sc, __uint_as_float(r1.y) * sc,
                                __uint_as_float(r1.z) * sc, __uint_as_float(r1.w) * sc};
            // square roots (edge candidates) and reciprocals (triangle bases) of
            // the six squared lengths, shared by the element's four targets
            float sq[6], rc[6];
    #pragma unroll
            for (int k = 0; k < 6; ++k) {
              sq[k] = csqrt(g[k]);
              rc[k] = __builtin_amdgcn_rcpf(g[k]);
            }
            const uint32_t nd[4] = {r0.x & 0x7fffu, (r0.x >> 16) & 0x7fffu, r0.y & 0xffffu,
                                    r0.y >> 16};
            float ph[4];
            int f[4];
    #pragma unroll
            for (int k = 0; k < 4; ++k) {
              ph[k] = phi_l[nd[k]];
              f[k] = flag_at(flg, nd[k]) ? 1 : 0;
            }
            const uint32_t tm = live_targets(erec[3 * e + 2], csqrt(sc), ph, f);
    #define FIM_TARGET(T)                                                                 \
            if (tm & (1u << T)) {                                                             \
              const float c = cand_exact_sh<T, float>(g, sq, rc, ph, F_INF);                 \
              ++vupd;                                                                         \
              if (c < ph[T]) {                                                                \
                const uint32_t cbits = __float_as_uint(c);                                    \
                if (cbits < atomicMin(&phi_n[nd[T]], cbits))                                  \
                  atomicOr(&wrt[nd[T] >> 5], 1u << (nd[T] & 31));                             \
              }                                                                               \
            }
            FIM_TARGET(0)
            FIM_TARGET(1)
            FIM_TARGET(2)
            FIM_TARGET(3)
    #undef FIM_TARGET
          }
        }
        __builtin_amdgcn_wave_barrier();
      }
      __syncthreads();
      // accept the written vertices: the sources of the next sweep
      // lane i of a wave looks at its block i of 64 copies: blocks with nothing
      // written have no sources, the others are gone through
      for (uint32_t b0 = wave; b0 < nv64 / 64; b0 += BS) {
        const uint32_t bl = b0 + lane * (BS / 64);
        uint2 wr = make_uint2(0u, 0u);
        if (bl < nv64 / 64) {
          wr = reinterpret_cast<const uint2 *>(wrt)[bl];
          if ((wr.x | wr.y) == 0u) reinterpret_cast<uint2 *>(flg)[bl] = make_uint2(0u, 0u);
        }
        for (uint64_t some = __ballot((wr.x | wr.y) != 0u); some; some &= some - 1) {
          const int i = __ffsll((unsigned long long)some) - 1;
          const uint32_t k = 2 * (b0 + (uint32_t)i * (BS / 64)), l = 32 * k + lane;
          const uint64_t w = (uint64_t)(uint32_t)__builtin_amdgcn_readlane(wr.y, i) << 32 |
                             (uint32_t)__builtin_amdgcn_readlane(wr.x, i);
          bool sg = false, lt = false, dc = false;
          if ((w >> lane) & 1u) {
            const float ov = phi_l[l];
            const float nv = __uint_as_float(phi_n[l]);
            if (nv < ov) {
              phi_l[l] = nv;
              dc = true;
              if ((ov - nv) >= eps * (1.0f + 0.5f * (ov + nv))) {
                lt = nv > W;
                sg = !lt;
              }
            }
          }
          const uint64_t msg = __ballot(sg), mlt = __ballot(lt), mdc = __ballot(dc);
          if (lane == 0) {
            flg[k] = (uint32_t)msg;
            flg[k + 1] = (uint32_t)(msg >> 32);
            wrt[k] = 0u;
            wrt[k + 1] = 0u;
          }
          if (lane == 1) {
            tch[k] |= (uint32_t)mdc;
            tch[k + 1] |= (uint32_t)(mdc >> 32);
          }
          if (lane == 2) {
            dfr[k] = (dfr[k] & ~(uint32_t)msg) | (uint32_t)mlt;
            dfr[k + 1] = (dfr[k + 1] & ~(uint32_t)(msg >> 32)) | (uint32_t)(mlt >> 32);
          }
          wave_append(sg, l, vlist, &misc[2]);
        }
      }
      __syncthreads();
    }
    // algorithmic bytes: copies (phi 4+4, flag 1+1), interface entries
    // (4+4+4) and the distinct elements evaluated (32 B: 24 B of FP32
    // geometry + 8 B of node ids; the record's 16 B of candidate bounds and
    // their scale are pruning data of this kernel, not algorithmic bytes)
    uint32_t cnt = 0;
    for (uint32_t k = tid; k < new32; k += BS) cnt += __popc(eseen[k]);
    // up to 65,535 elements, so 2,048 / BS words of 32 per thread (8 with 256)
    cnt = wave_sum_small<BS >= 256 ? 9 : BS == 128 ? 10 : 11>(cnt);
    if (lane == 0 && cnt) atomicAdd(&misc[3], cnt);
    if (lane == 0 && evals) atomicAdd(&misc[0], evals);
    // write back decreased copies and list the lowered interface copies
    // (interface entry << 16 | copy, in the space of the candidate minima);
    // deferred vertices (and sources left by the sweep cap) stay dirty and the
    // submesh is queued again.  Lane i of a wave looks at its block i of 64
    // copies; blocks with nothing lowered or left dirty are skipped.
    const KArgs ke = kargs();
    tid = fresh(tid);
    float *phi_e = ke->phi + (size_t)inst * ke->ncopy + si.coff;
    uint8_t *dirty_e = ke->dirty + (size_t)inst * ke->ncopy + si.coff;
    uint32_t dmin = 0xffffffffu;  // earliest time left dirty, per lane
    for (uint32_t b0 = wave; b0 < nv64 / 64; b0 += BS) {
      const uint32_t bl = b0 + lane * (BS / 64);
      uint2 tc = make_uint2(0u, 0u), df = tc;
      if (bl < nv64 / 64) {
        tc = reinterpret_cast<const uint2 *>(tch)[bl];
        df = reinterpret_cast<const uint2 *>(dfr)[bl];
        if (capped) {
          const uint2 fl = reinterpret_cast<const uint2 *>(flg)[bl];
          df.x |= fl.x;
          df.y |= fl.y;
        }
      }
      for (uint64_t some = __ballot((tc.x | tc.y | df.x | df.y) != 0u); some; some &= some - 1) {
        const int i = __ffsll((unsigned long long)some) - 1;
        const uint32_t l = 64 * (b0 + (uint32_t)i * (BS / 64)) + lane;
        const uint64_t t = (uint64_t)(uint32_t)__builtin_amdgcn_readlane(tc.y, i) << 32 |
                           (uint32_t)__builtin_amdgcn_readlane(tc.x, i);
        const uint64_t q = (uint64_t)(uint32_t)__builtin_amdgcn_readlane(df.y, i) << 32 |
                           (uint32_t)__builtin_amdgcn_readlane(df.x, i);
        const float v = phi_l[l];
        bool p = false;
        if ((t >> lane) & 1u) {
          phi_e[l] = v;
          p = flag_at(ifc, l);
        }
        if ((q >> lane) & 1u) {
          dirty_e[l] = 1;
          dmin = min(dmin, __float_as_uint(v));
        }
        const uint64_t m = __ballot(p);
        if (m == 0) continue;
        uint32_t at = 0;
        if (lane == 0) at = atomicAdd(&misc[npush], (uint32_t)__popcll(m));
        at = __builtin_amdgcn_readfirstlane(at);
        if (p) phi_n[at + (uint32_t)__popcll(m & lanes_below())] = (ipre[l >> 5] + bits_below(ifc, l)) << 16 | l;
      }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) dmin = min(dmin, (uint32_t)__shfl_xor(dmin, off));
    if (lane == 0 && dmin != 0xffffffffu) atomicMin(&misc[5], dmin);
    __syncthreads();
    const Queue nq = next_queue(ke, iter_now);
    if (tid == 0) {
      if (it > 0) {  // pushes that lowered nothing make no activation
        ctr[0] += 1ull;
        ctr[1] += it;
        ctr[2] += misc[0];
        ctr[3] += 32ull * misc[3] + 10ull * nn + 12ull * si.ni;
      }
      end_item(ke, nq, inst, s, iter_now, item.pushed, __uint_as_float(misc[5]));
    }
    // the last waves first: the first wave, which ends the item, is free to
    // fetch the next one meanwhile
    for (uint32_t i = BS - 1 - tid, n = misc[npush]; i < n; i += BS) {
      const uint32_t q = phi_n[i];
      push_entry(ke, nq, inst, si.ioff + (q >> 16), __float_as_uint(phi_l[q & 0xffffu]), iter_now);
    }
    // no barrier: what the push reads (times, list) is written again only after
    // the next item's first barrier, its count is another word
    npush ^= 1u;
  }
  unsigned long long *stats = kargs()->stats;
  if (tid == 0 && ctr[0]) {
    atomicAdd(&stats[0], ctr[0]);
    atomicAdd(&stats[1], ctr[1]);
    atomicAdd(&stats[2], ctr[2]);
    atomicAdd(&stats[4], ctr[3]);
  }
  unsigned long long vsum = vupd;
  for (int off = 32; off > 0; off >>= 1) vsum += __shfl_xor(vsum, off);
  if (lane == 0 && vsum) atomicAdd(&stats[5], vsum);
}

// Merges what is left in the inbox (the run stopped before the items it was
// pushed to were worked through) into the copies' times, so that a context's
// state is in its times, flags and list alone.
struct DrainArgs {
  const uint32_t *ifc;  // per interface entry: its copy
  const uint32_t *c2s;
  uint32_t *inbox;
  float *phi, *wown;
  uint8_t *dirty;
  const uint32_t *iter;
  uint32_t n_if, ncopy, nsub, ninst;
};

__global__ __launch_bounds__(256) void k_conv_drain(DrainArgs a) {
  uint32_t *inbox = a.inbox + (*a.iter & 1u) * (size_t)a.ninst * a.n_if;
  for (uint32_t inst = blockIdx.y; inst < a.ninst; inst += gridDim.y)
    for (uint32_t e = blockIdx.x * blockDim.x + threadIdx.x; e < a.n_if; e += gridDim.x * blockDim.x) {
      const size_t i = (size_t)inst * a.n_if + e;
      const uint32_t v = inbox[i];
      if (v == __float_as_uint(F_INF)) continue;
      inbox[i] = __float_as_uint(F_INF);
      const uint32_t c = a.ifc[e];
      const size_t gc = (size_t)inst * a.ncopy + c;
      if (__uint_as_float(v) < a.phi[gc]) {
        a.phi[gc] = __uint_as_float(v);
        a.dirty[gc] = 1;
        atomicMin(reinterpret_cast<uint32_t *>(a.wown) + (size_t)inst * a.nsub + a.c2s[c], v);
      }
    }
}

// seeds: (instance, copy) pairs get min(phi, t0), are flagged, and their
// submesh is queued on the current list
__global__ void k_conv_seed(const uint2 *ic, uint32_t n, float t0, const uint32_t *c2s, float *phi,
                            uint8_t *dirty, float *wake, Queue q, uint32_t ncopy) {
  const uint32_t nsub = q.nsub;
  q.enter();
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const uint32_t inst = ic[i].x, c = ic[i].y;
    const size_t gc = (size_t)inst * ncopy + c;
    atomicMin(reinterpret_cast<uint32_t *>(phi + gc), __float_as_uint(t0));
    dirty[gc] = 1;
    const uint32_t s = c2s[c];
    atomicMin(reinterpret_cast<uint32_t *>(wake + (size_t)inst * nsub + s), __float_as_uint(t0));
    q.add(inst, s, kQueued);
  }
}

// per instance: 1 if any (instance, submesh) pair is queued
__global__ __launch_bounds__(256) void k_inst_active(Queue q, uint32_t *out) {
  __shared__ uint32_t any;
  if (threadIdx.x == 0) any = 0u;
  q.enter();
  __syncthreads();
  const uint32_t *row = q.act + (size_t)blockIdx.x * q.nsub;
  uint32_t v = 0u;
  for (uint32_t s = threadIdx.x; s < q.nsub; s += blockDim.x) v |= row[s] >= q.tag ? 1u : 0u;
  if (v) atomicOr(&any, 1u);
  __syncthreads();
  if (threadIdx.x == 0) out[blockIdx.x] = any;
}

// Gives the next iteration the number `to` (to + 1 if its parity differs: inbox,
// wake times and flags exist by parity), between runs.  What is queued
// for it stays queued, for the same reason; flags of earlier iterations are
// cleared; the instances' windows go on from where they are.
__device__ inline uint32_t renumbered(uint32_t now, uint32_t to) { return to + ((now ^ to) & 1u); }
__global__ __launch_bounds__(256) void k_conv_renumber(const uint32_t *iter, uint32_t to, uint32_t *act, size_t nss,
                                                       uint32_t *start, uint32_t ninst) {
  const uint32_t now = *iter, next = renumbered(now, to), tag = act_tag(now);
  uint32_t *cur = act + (now & 1u) * nss, *other = act + (~now & 1u) * nss;
  const size_t first = blockIdx.x * (size_t)256 + threadIdx.x, step = (size_t)gridDim.x * 256;
  for (size_t i = first; i < nss; i += step) {
    const uint32_t f = cur[i];
    cur[i] = f >= tag ? act_tag(next) + (f & 3u) : 0u;
    other[i] = 0u;
  }
  for (size_t i = first; i < ninst; i += step) start[i] += next - now;
}
__global__ void k_iter_set(uint32_t *iter, uint32_t to) { *iter = renumbered(*iter, to); }

// recycles finished instances: times to +inf, flags and wake times cleared,
// and the instance's window restarts at the current iteration
__global__ void k_inst_reset(const uint32_t *insts, uint32_t n, float *phi, uint8_t *dirty, float *wake,
                             uint32_t *start, const uint32_t *iter, uint32_t ncopy, uint32_t nsub) {
  const size_t per = (size_t)ncopy + nsub;
  const size_t total = per * n;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
    const uint32_t inst = insts[i / per];
    const size_t k = i % per;
    if (k < ncopy) {
      phi[(size_t)inst * ncopy + k] = F_INF;
      dirty[(size_t)inst * ncopy + k] = 0;
    } else {
      wake[(size_t)inst * nsub + (k - ncopy)] = F_INF;
    }
    if (k == 0) start[inst] = *iter;
  }
}

// warm start: every copy of the instance takes the global field value,
// everything flagged, every submesh queued
__global__ void k_conv_init(const float *phi0, const uint32_t *c2g, uint32_t inst, float *phi,
                            uint8_t *dirty, uint32_t ncopy, int flag) {
  for (uint32_t c = blockIdx.x * blockDim.x + threadIdx.x; c < ncopy; c += gridDim.x * blockDim.x) {
    const size_t gc = (size_t)inst * ncopy + c;
    phi[gc] = phi0[c2g[c]];
    dirty[gc] = (uint8_t)flag;
  }
}

__global__ void k_conv_queue_all(uint32_t inst, float *wake, Queue q) {
  q.enter();
  for (uint32_t s = blockIdx.x * blockDim.x + threadIdx.x; s < q.nsub; s += gridDim.x * blockDim.x) {
    wake[(size_t)inst * q.nsub + s] = 0.0f;
    q.add(inst, s, kQueued);
  }
}

template <class T>
__global__ void k_fill(T *p, size_t n, T v) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    p[i] = v;
}

// Several arrays filled in one launch (a context's reset was ten, at about 4 us
// each on a small mesh): 16 bytes of each array's pattern at a time, and
// the bytes left at its end.
struct FillArgs {
  struct {
    void *p;       // 16-byte aligned
    size_t bytes;
    uint4 v;       // the pattern (of 1, 4 or 8 bytes, repeated)
  } seg[10];
  int n = 0;
  template <class T>
  void add(T *p, size_t count, T v) {
    static_assert(sizeof(T) <= 8, "pattern");
    unsigned char b[16];
    for (size_t i = 0; i < 16; i += sizeof(T)) std::memcpy(b + i, &v, sizeof(T));
    seg[n].p = p;
    seg[n].bytes = count * sizeof(T);
    std::memcpy(&seg[n++].v, b, 16);
  }
};

__global__ __launch_bounds__(256) void k_fill_all(FillArgs a) {
  const size_t first = blockIdx.x * (size_t)256 + threadIdx.x, step = (size_t)gridDim.x * 256;
  for (int k = 0; k < a.n; ++k) {
    const size_t n16 = a.seg[k].bytes / 16;
    const uint4 v = a.seg[k].v;
    uint4 *p = static_cast<uint4 *>(a.seg[k].p);
    for (size_t i = first; i < n16; i += step) p[i] = v;
    if (first < a.seg[k].bytes % 16) {
      const uint32_t w[4] = {v.x, v.y, v.z, v.w};
      reinterpret_cast<unsigned char *>(p + n16)[first] = (unsigned char)(w[first / 4] >> 8 * (first % 4));
    }
  }
}

// Before a run: speed factors and windows from pinned memory, counters cleared
// (two copies, a wait and a clear before)
__global__ __launch_bounds__(256) void k_run_begin(const float *src, uint32_t nr, float *rscale, uint32_t nw,
                                                   float *winst, unsigned long long *stats) {
  for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < nr + nw; i += gridDim.x * 256) {
    if (i < nr)
      rscale[i] = src[i];
    else
      winst[i - nr] = src[i];
  }
  if (stats && blockIdx.x == 0 && threadIdx.x < 8) stats[threadIdx.x] = 0ull;
}

// After a chunk of iterations: queued units and counters to pinned memory
// (word 0; words 2..17)
__global__ void k_chunk_end(const uint32_t *left, const uint32_t *stats, uint32_t *pin) {
  if (threadIdx.x == 0) pin[0] = *left;
  if (threadIdx.x < 16) pin[2 + threadIdx.x] = stats[threadIdx.x];
}

// min over copies of each global vertex
__global__ void k_conv_gather(const float *phi, const uint32_t *g2c_dsp, const uint32_t *g2c,
                              uint32_t nn, size_t ib, float *out) {
  for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < nn; v += gridDim.x * blockDim.x) {
    float m = F_INF;
    for (uint32_t k = g2c_dsp[v]; k < g2c_dsp[v + 1]; ++k) m = fminf(m, phi[ib + g2c[k]]);
    out[v] = m;
  }
}

// residual sweep: max relative amount any copy could still be lowered
__global__ __launch_bounds__(256) void k_conv_residual(const SubInfo *sub, uint32_t nsub,
                                                       const uint2 *e2n, const float *geo,
                                                       const uint8_t *ereg, const float *rscale,
                                                       const float *phi, size_t ib, uint32_t inst,
                                                       uint32_t *res_bits) {
  float worst = 0.0f;
  for (uint32_t s = blockIdx.x; s < nsub; s += gridDim.x) {
    const SubInfo si = sub[s];
    for (uint32_t e = threadIdx.x; e < si.ne; e += blockDim.x) {
      const size_t ge = (size_t)si.eoff + e;
      const uint2 q = e2n[ge];
      const uint32_t nd[4] = {q.x & 0xffffu, q.x >> 16, q.y & 0xffffu, q.y >> 16};
      const float sc = rscale[4 * (size_t)inst + (ereg[ge] & 3)];
      float g[6], ph[4];
      for (int k = 0; k < 6; ++k) g[k] = geo[6 * ge + k] * sc;
      for (int k = 0; k < 4; ++k) ph[k] = phi[ib + si.coff + nd[k]];
      float c[4] = {cand_exact<0, float>(g, ph, F_INF), cand_exact<1, float>(g, ph, F_INF),
                    cand_exact<2, float>(g, ph, F_INF), cand_exact<3, float>(g, ph, F_INF)};
      for (int k = 0; k < 4; ++k)
        if (c[k] < ph[k]) worst = fmaxf(worst, ph[k] == F_INF ? F_INF : (ph[k] - c[k]) / (1.0f + ph[k]));
    }
  }
  if (worst > 0.0f) atomicMax(res_bits, __float_as_uint(worst));
}

// support sweep: for every vertex the smallest candidate its elements give
// (global vertex, float bits, atomicMin); seeds and unreached vertices are
// judged by the caller
__global__ __launch_bounds__(256) void k_conv_support(const SubInfo *sub, uint32_t nsub,
                                                      const uint2 *e2n, const float *geo,
                                                      const uint8_t *ereg, const float *rscale,
                                                      const float *phi, const uint32_t *c2g,
                                                      size_t ib, uint32_t inst, uint32_t *best) {
  for (uint32_t s = blockIdx.x; s < nsub; s += gridDim.x) {
    const SubInfo si = sub[s];
    for (uint32_t e = threadIdx.x; e < si.ne; e += blockDim.x) {
      const size_t ge = (size_t)si.eoff + e;
      const uint2 q = e2n[ge];
      const uint32_t nd[4] = {q.x & 0xffffu, q.x >> 16, q.y & 0xffffu, q.y >> 16};
      const float sc = rscale[4 * (size_t)inst + (ereg[ge] & 3)];
      float g[6], ph[4];
      for (int k = 0; k < 6; ++k) g[k] = geo[6 * ge + k] * sc;
      for (int k = 0; k < 4; ++k) ph[k] = phi[ib + si.coff + nd[k]];
      const float c[4] = {cand_exact<0, float>(g, ph, F_INF), cand_exact<1, float>(g, ph, F_INF),
                          cand_exact<2, float>(g, ph, F_INF), cand_exact<3, float>(g, ph, F_INF)};
      for (int k = 0; k < 4; ++k)
        if (c[k] < F_INF) atomicMin(&best[c2g[si.coff + nd[k]]], __float_as_uint(c[k]));
    }
  }
}

// worst relative amount by which a reached, non-seed vertex lies below the
// best candidate of its elements (a field that is not a fixed point from
// below: an initial field that was not an upper bound)
__global__ void k_support_check(const float *phi_g, const uint32_t *best, uint32_t nn,
                                uint32_t *worst_bits) {
  float worst = 0.0f;
  for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < nn; v += gridDim.x * blockDim.x) {
    const float p = phi_g[v];
    if (!(p > 0.0f) || !(p < F_INF)) continue;
    const float b = __uint_as_float(best[v]);
    if (b > p) worst = fmaxf(worst, (b - p) / (1.0f + p));
  }
  if (worst > 0.0f) atomicMax(worst_bits, __float_as_uint(worst));
}

// ---------------------------------------------------------------------------
// compat mode (reference time windows, FP64)
// ---------------------------------------------------------------------------
constexpr uint32_t kNoVertex = 0xffffffffu;

// A submesh of k_compat_small: its constant data is one block of 16-byte
// words (blob + boff): slot chunk offsets of the copies (nn + 1 u16), node ids
// of the elements (8 B each), slots (u16, element << 2 | position, each copy's
// padded to chunks of four with kNoSlot) and, if it is to be in LDS, the FP64
// geometry (48 B per element).
struct CompatSub {
  uint32_t coff, nn, eoff, ne, ioff, boff, nw, nch;  // nw words, nch chunks of slots
};
constexpr uint16_t kNoSlot = 0xffffu;

struct CompatArgs {
  const SubInfo *sub;
  const uint2 *e2n;
  const double *geo;
  const uint32_t *n2e_dsp;
  const uint16_t *n2e_le;
  const uint8_t *n2e_pos;
  const uint32_t *n2n_dsp;
  const uint16_t *n2n_lv;
  double *phi;
  int8_t *st;
  double *nexte;              // per submesh: earliest window time its copies change
  const uint32_t *list;       // submeshes of this window (k_compat_sync), *nlist of them
  const uint32_t *nlist;
  const uint32_t *cshared;    // per copy: its vertex if it has other copies, else kNoVertex
  uint32_t *vrec, *vcnt;      // per submesh (at ioff): shared vertices whose copy changed, their number
  unsigned long long *done;   // finished workgroups << 32 | pending copies
  uint32_t *out;              // pinned host word: copies left narrow/next after the window
  uint32_t nsub;
  int32_t exact;
  double fw, cur, phi_start, dt, apd;
  uint32_t o_tphi, o_st, o_tst, o_snap, o_misc;
  // k_compat_small
  const CompatSub *csub;
  const uint4 *blob;
  uint32_t o_tmin, o_lp, o_lq, o_blob;
};

__device__ inline uint32_t block_sum(uint32_t v, uint32_t *slot) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  if (threadIdx.x == 0) *slot = 0u;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) atomicAdd(slot, v);
  __syncthreads();
  const uint32_t r = *slot;
  __syncthreads();
  return r;
}

// FP64 bit pattern -> unsigned key of the same order (no NaN) and back
__device__ inline unsigned long long dkey(double d) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(d);
  return (b >> 63) ? ~b : (b | (1ull << 63));
}
__device__ inline double dkey_inv(unsigned long long k) {
  return __longlong_as_double((long long)((k >> 63) ? (k & ~(1ull << 63)) : ~k));
}

// minimum over the block, valid in thread 0 only (the slot is reset by
// thread 0 before its first barrier, so back-to-back calls need no third one)
__device__ inline double block_min0(double v, unsigned long long *slot) {
  for (int off = 32; off > 0; off >>= 1) v = fmin(v, __shfl_xor(v, off));
  if (threadIdx.x == 0) *slot = ~0ull;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) atomicMin(slot, dkey(v));
  __syncthreads();
  return threadIdx.x == 0 ? dkey_inv(*slot) : 0.0;
}

// A workgroup is through with its submeshes (one thread calls this): the last
// of the min(max(n, 1), gridDim) workgroups that take part knows the window's
// pending count from the one counter all of them add to, hands it to the host
// and clears the counter, so a window needs no fill and no copy for it.
__device__ inline void compat_finish(const CompatArgs &a, uint32_t nlist, uint32_t pend) {
  const uint32_t part = min(max(nlist, 1u), gridDim.x);
  if (blockIdx.x >= part) return;
  const unsigned long long add = (1ull << 32) | pend;
  const unsigned long long now = atomicAdd(a.done, add) + add;
  if ((uint32_t)(now >> 32) == part) {
    __hip_atomic_store(a.out, (uint32_t)now, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(a.done, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// Records the shared vertices whose copies (c, of the lanes with `changed`)
// the pass has changed in the submesh's range of vrec; cnt is one LDS word.
// Lane 0 of a wave is active whenever another lane is.
__device__ inline void compat_record(const CompatArgs &a, uint32_t ioff, bool changed, uint32_t c, uint32_t *cnt) {
  const uint32_t v = changed ? a.cshared[c] : kNoVertex;
  const uint64_t m = __ballot(v != kNoVertex);
  if (m == 0) return;
  uint32_t at = 0;
  if ((threadIdx.x & 63) == 0) at = atomicAdd(cnt, (uint32_t)__popcll(m));
  at = __builtin_amdgcn_readfirstlane(at);
  if (v != kNoVertex) a.vrec[ioff + at + (uint32_t)__popcll(m & lanes_below())] = v;
}

// one (vertex, element) slot: src/eikonal/cuda_fim.h:1362-1411.  The slot's
// element nodes nd (local ids) and the owner's position t are given.
__device__ inline double compat_slot(const CompatArgs &a, const SubInfo &si, const double *phi_l,
                                     const int8_t *st_l, size_t ge, const uint32_t nd[4], int t) {
  double ph[4], g[6];
  const double lo = a.phi_start - a.fw;
  for (int j = 0; j < 4; ++j) {
    const uint32_t n = nd[j];
    ph[j] = (j != t && st_l[n] >= FIM_NARROW && phi_l[n] > lo) ? phi_l[n] : DBL_MAX;
  }
  for (int j = 0; j < 6; ++j) g[j] = a.geo[6 * ge + j];
  if (!a.exact) return cand_ref(g, ph, t);
  switch (t) {
    case 0: return cand_exact<0, double>(g, ph, DBL_MAX);
    case 1: return cand_exact<1, double>(g, ph, DBL_MAX);
    case 2: return cand_exact<2, double>(g, ph, DBL_MAX);
    default: return cand_exact<3, double>(g, ph, DBL_MAX);
  }
}

constexpr unsigned long long kDmaxBits = 0x7fefffffffffffffull;  // DBL_MAX

// The candidates of every slot k0 <= k < k1 whose owner has state `want`,
// merged into the owner's minimum (FP64 bits, LDS integer min).
__device__ inline void compat_slots(const CompatArgs &a, const SubInfo &si, const double *phi_l, const int8_t *st_l,
                                    uint32_t k0, uint32_t k1, int8_t want, unsigned long long *tmin) {
  for (uint32_t k = k0 + threadIdx.x; k < k1; k += blockDim.x) {
    const int t = a.n2e_pos[k];
    const size_t ge = (size_t)si.eoff + a.n2e_le[k];
    const uint2 q = a.e2n[ge];
    const uint32_t nd[4] = {q.x & 0xffffu, q.x >> 16, q.y & 0xffffu, q.y >> 16};
    const uint32_t owner = nd[t];
    if (st_l[owner] != want) continue;
    const double v = compat_slot(a, si, phi_l, st_l, ge, nd, t);
    atomicMin(&tmin[owner], (unsigned long long)__double_as_longlong(v));
  }
}

template <int BS>
__global__ __launch_bounds__(BS) void k_compat_compute(CompatArgs a) {
#pragma clang fp contract(off)
  extern __shared__ __align__(16) unsigned char lds[];
  double *phi_l = reinterpret_cast<double *>(lds);
  double *tphi = reinterpret_cast<double *>(lds + a.o_tphi);
  int8_t *st_l = reinterpret_cast<int8_t *>(lds + a.o_st);
  int8_t *tst = reinterpret_cast<int8_t *>(lds + a.o_tst);
  int8_t *snap = reinterpret_cast<int8_t *>(lds + a.o_snap);
  uint32_t *misc = reinterpret_cast<uint32_t *>(lds + a.o_misc);
  const uint32_t tid = threadIdx.x;
  unsigned long long *evslot = reinterpret_cast<unsigned long long *>(misc + 2);
  const uint32_t nlist = *a.nlist;
  uint32_t pend_wg = 0;  // thread 0
  for (uint32_t i = blockIdx.x; i < nlist; i += gridDim.x) {
    const uint32_t s = a.list[i];
    const SubInfo si = a.sub[s];
    const uint32_t nn = si.nn;
    // update_states (cuda_fim.cu:1790-1845), applied to every submesh
    uint32_t cnt = 0;
    double p0 = 0.0;  // the copy as loaded (one copy per thread when nn <= BS)
    int8_t st0 = 0;
    for (uint32_t l = tid; l < nn; l += BS) {
      double p = a.phi[si.coff + l];
      int8_t st = a.st[si.coff + l];
      p0 = p;
      st0 = st;
      if (st == FIM_NARROW) {
        ++cnt;
      } else if (st == FIM_NEXT) {
        ++cnt;
        st = FIM_NARROW;
      } else if (st == FIM_FROZEN) {
        if (!(p + a.apd > a.cur)) st = FIM_TAIL;
      } else if (st == FIM_TAIL) {
        if (!(p + a.apd / 0.91 > a.cur)) {
          p = DBL_MAX;
          st = FIM_FAR;
        }
      }
      phi_l[l] = p;
      st_l[l] = st;
    }
    uint32_t active = block_sum(cnt, misc);
    const bool idle = active == 0;
    // the submesh's (vertex, element) slots, contiguous in the copy-major CSR
    const uint32_t k0 = a.n2e_dsp[si.coff], k1 = a.n2e_dsp[si.coff + nn];
    unsigned long long *tmin = reinterpret_cast<unsigned long long *>(tphi);
    while (active > 0) {
      // a: candidates of narrow vertices, one thread per slot; times are
      // >= 0, so the minimum of the FP64 bit patterns as integers is the
      // minimum of the values and does not depend on the order
      for (uint32_t l = tid; l < nn; l += BS) tmin[l] = kDmaxBits;
      __syncthreads();
      compat_slots(a, si, phi_l, st_l, k0, k1, FIM_NARROW, tmin);
      __syncthreads();
      // b: reduce, window test, convergence test
      for (uint32_t l = tid; l < nn; l += BS) {
        tst[l] = FIM_FAR;
        if (st_l[l] != FIM_NARROW) continue;
        const double old = phi_l[l];
        const double nw = tphi[l] < old ? tphi[l] : old;
        phi_l[l] = nw;
        if (nw - a.phi_start > a.dt)
          st_l[l] = FIM_NEXT;
        else if (fabs(old - nw) < (1e-6 * (1 + (old + nw) * .5)))
          tst[l] = FIM_FROZEN;
      }
      __syncthreads();
      // c: downwind neighbours of just-frozen vertices (flags as after b)
      for (uint32_t l = tid; l < nn; l += BS) snap[l] = tst[l];
      __syncthreads();
      for (uint32_t l = tid; l < nn; l += BS) {
        if (st_l[l] == FIM_NARROW) continue;
        const uint32_t c = si.coff + l;
        for (uint32_t k = a.n2n_dsp[c]; k < a.n2n_dsp[c + 1]; ++k) {
          const uint32_t n = a.n2n_lv[k];
          if (snap[n] == FIM_FROZEN && phi_l[n] < phi_l[l]) {
            tst[l] = st_l[l];
            st_l[l] = FIM_NEIG;
            break;
          }
        }
      }
      __syncthreads();
      // d: candidates of marked vertices, one thread per slot
      for (uint32_t l = tid; l < nn; l += BS) tmin[l] = kDmaxBits;
      __syncthreads();
      compat_slots(a, si, phi_l, st_l, k0, k1, FIM_NEIG, tmin);
      __syncthreads();
      // e: accept improvements
      for (uint32_t l = tid; l < nn; l += BS) {
        if (st_l[l] != FIM_NEIG) continue;
        const double old = phi_l[l];
        const double nw = tphi[l] < old ? tphi[l] : old;
        phi_l[l] = nw;
        st_l[l] = (nw < old) ? (int8_t)FIM_NARROW : tst[l];
      }
      __syncthreads();
      // f: freeze / count
      cnt = 0;
      for (uint32_t l = tid; l < nn; l += BS) {
        if (st_l[l] == FIM_NARROW) {
          if (tst[l] == FIM_FROZEN)
            st_l[l] = FIM_FROZEN;
          else
            ++cnt;
        } else if (st_l[l] == FIM_NEIG) {
          st_l[l] = FIM_NARROW;
          ++cnt;
        }
      }
      active = block_sum(cnt, misc);
    }
    // write back; when nothing was narrow only update_states' time-driven
    // transitions can have changed a copy, and nothing is pending (narrow and
    // next copies are what `active` counted).  ev: the earliest window time
    // at which update_states would change a copy (frozen: p + apd, tail:
    // p + apd / 0.91, as update_states computes them; narrow or next: now)
    const bool lean = idle && nn <= BS;
    uint32_t pend = 0;
    double ev = INFINITY;
    if (tid == 0) misc[1] = 0u;
    __syncthreads();
    for (uint32_t l = tid; l < nn; l += BS) {
      const double p = phi_l[l];
      const int8_t st = st_l[l];
      compat_record(a, si.ioff, !lean || p != p0, si.coff + l, &misc[1]);
      if (!lean || p != p0 || st != st0) {
        a.phi[si.coff + l] = p;
        a.st[si.coff + l] = st;
      }
      if (st == FIM_NARROW || st == FIM_NEXT) {
        ++pend;
        ev = -INFINITY;
      } else if (st == FIM_FROZEN) {
        ev = fmin(ev, p + a.apd);
      } else if (st == FIM_TAIL) {
        ev = fmin(ev, p + a.apd / 0.91);
      }
    }
    if (!lean) {
      pend = block_sum(pend, misc);
      pend_wg += pend;
    }
    ev = block_min0(ev, evslot);
    if (tid == 0) {
      a.nexte[s] = ev;
      a.vcnt[s] = misc[1];
    }
  }
  if (tid == 0) compat_finish(a, nlist, pend_wg);
}

// geometry index of e12 e13 e23 e14 e24 e34 after relabelling for target t
// (3 bits each, e12 lowest)
__device__ inline uint32_t compat_relabel(int t) {
  constexpr auto pack = [](int t) {
    const int q1 = (t + 1) & 3, q2 = (t + 2) & 3, q3 = (t + 3) & 3;
    return (uint32_t)(edge_idx(q1, q2) | edge_idx(q1, q3) << 3 | edge_idx(q2, q3) << 6 | edge_idx(q1, t) << 9 |
                      edge_idx(q2, t) << 12 | edge_idx(q3, t) << 15);
  };
  constexpr uint32_t r0 = pack(0), r1 = pack(1), r2 = pack(2), r3 = pack(3);
  return t & 2 ? (t & 1 ? r3 : r2) : (t & 1 ? r1 : r0);
}

// The window's pass for submeshes of at most BS copies: one thread per copy
// keeps the copy's time and states in registers, the submesh's (vertex,
// element) slots, node ids and (GEO) FP64 geometry are in LDS for all sweeps
// of the window.  The pass is a chain of short sweeps, so what a sweep costs
// is its latency: barriers, memory round trips and rounds of the ~3,000-cycle
// FP64 candidate.  Here
//   - a phase's slots are appended to an LDS list by the threads that decide
//     on them, four at a time, so a candidate round has live lanes and no slot
//     is looked at in vain (the scan of every slot cost most of a sweep);
//   - `up` holds the time a copy offers to others (DBL_MAX if it may not act),
//     so a slot reads three words and no states;
//   - the downwind neighbours of just-frozen copies are found through the
//     elements (copies are neighbours when they share one);
//   - a sweep in which nothing froze has three barriers, any other five or six;
//   - the submesh's data comes straight into LDS, in flight together with the
//     copies' times, so a submesh waits for memory three times in all.
// Full slab, 10,152 submeshes of at most 128 copies, 150 windows of 2 ms: a
// map takes 11.7 ms against 25.0 with the general kernel (k_compat_compute)
// and the sync over all shared vertices; the pass 46 us per window against
// 109.  Workgroups of 256 beat 128 (12.8 ms) and 512 (13.2 ms); registers for
// five waves per SIMD spill (13.0 ms); submeshes taken from a counter instead
// of in turn gain nothing (11.9 ms).
template <int BS, bool GEO>
__global__ __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(4, 8))) void k_compat_small(CompatArgs a) {
#pragma clang fp contract(off)
  extern __shared__ __align__(16) unsigned char lds[];
  double *phi_l = reinterpret_cast<double *>(lds);
  double *up = reinterpret_cast<double *>(lds + a.o_tphi);
  unsigned long long *tmin = reinterpret_cast<unsigned long long *>(lds + a.o_tmin);
  int8_t *st_l = reinterpret_cast<int8_t *>(lds + a.o_st);
  uint2 *lp = reinterpret_cast<uint2 *>(lds + a.o_lp);  // slot chunks of narrow copies
  uint2 *lq = reinterpret_cast<uint2 *>(lds + a.o_lq);  // slot chunks of marked neighbours
  uint4 *blob = reinterpret_cast<uint4 *>(lds + a.o_blob);
  // misc: [0,1] chunks in lp (by sweep parity), [2] chunks in lq, [4,5]
  // block_min0's slot, [6] shared vertices recorded, [8..] just-frozen bits,
  // [8 + BS / 32 ..] marked-neighbour bits
  uint32_t *misc = reinterpret_cast<uint32_t *>(lds + a.o_misc);
  uint32_t *fz = misc + 8, *mk = fz + BS / 32;
  unsigned long long *evslot = reinterpret_cast<unsigned long long *>(misc + 4);
  const uint32_t tid = threadIdx.x, lane = tid & 63;
  const uint32_t l = tid;
  const double lo = a.phi_start - a.fw;
  const uint32_t nlist = *a.nlist;
  uint32_t s = a.list[blockIdx.x];  // gridDim <= nsub entries; read with nlist
  uint32_t pend_wg = 0;  // thread 0
  auto offer = [&](int8_t st, double p) { return (st >= FIM_NARROW && p > lo) ? p : DBL_MAX; };
  for (uint32_t i = blockIdx.x; i < nlist; i += gridDim.x) {
    if (i != blockIdx.x) s = a.list[i];
    const CompatSub si = a.csub[s];
    const uint32_t nn = si.nn, ne = si.ne;
    const bool own = l < nn;
    const uint16_t *dsp = reinterpret_cast<const uint16_t *>(blob);
    const uint2 *el = reinterpret_cast<const uint2 *>(blob + (2 * (nn + 1) + 15) / 16);
    const uint2 *sw = reinterpret_cast<const uint2 *>(reinterpret_cast<const uint4 *>(el) + (8 * ne + 15) / 16);
    const double *gl = reinterpret_cast<const double *>(reinterpret_cast<const uint4 *>(sw) + (8 * si.nch + 15) / 16);
    // chunks of the slots of copy v appended to a list
    auto append = [&](uint2 *list, uint32_t *cnt, uint32_t v) {
      const uint32_t b = dsp[v], n = dsp[v + 1] - b, at = atomicAdd(cnt, n);
      for (uint32_t k = 0; k < n; k += 3) {
        const uint2 w0 = sw[b + k], w1 = sw[b + min(k + 1, n - 1)], w2 = sw[b + min(k + 2, n - 1)];
        list[at + k] = w0;
        list[at + min(k + 1, n - 1)] = w1;
        list[at + min(k + 2, n - 1)] = w2;
      }
    };
    // the submesh's block into LDS: a wave's 64 lanes take 64 consecutive words
    for (uint32_t k0 = tid & ~63u; k0 < si.nw; k0 += BS)
      if (k0 + lane < si.nw)
        __builtin_amdgcn_global_load_lds(
            reinterpret_cast<const __attribute__((address_space(1))) uint32_t *>(
                reinterpret_cast<uintptr_t>(a.blob + si.boff + k0 + lane)),
            (__attribute__((address_space(3))) uint32_t *)(blob + k0), 16, 0, 0);
    // update_states (cuda_fim.cu:1790-1845)
    double p = DBL_MAX, p0 = 0.0;
    int8_t st = FIM_FAR, st0 = FIM_FAR;
    if (own) {
      p = a.phi[si.coff + l];
      st = a.st[si.coff + l];
      p0 = p;
      st0 = st;
      if (st == FIM_NEXT) {
        st = FIM_NARROW;
      } else if (st == FIM_FROZEN) {
        if (!(p + a.apd > a.cur)) st = FIM_TAIL;
      } else if (st == FIM_TAIL) {
        if (!(p + a.apd / 0.91 > a.cur)) {
          p = DBL_MAX;
          st = FIM_FAR;
        }
      }
    }
    if (tid < 8) misc[tid] = 0u;
    if (tid < 2 * (BS / 32)) fz[tid] = 0u;
    if (own) {
      phi_l[l] = p;
      up[l] = offer(st, p);
      st_l[l] = st;
      tmin[l] = kDmaxBits;
    }
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): the block is in LDS
    __syncthreads();
    if (own && st == FIM_NARROW) append(lp, &misc[0], l);
    {
      // candidates of the listed slots: times are >= 0, so the minimum of the
      // FP64 bit patterns as integers is the minimum of the values.  A slot's
      // reference candidate is worked out by two lanes of different waves
      // (the tet face and a triangle; two triangles and the edges): half the
      // chain, at half the slots per round.
      auto evaluate = [&](const uint2 *chunks, uint32_t nch) {
        const uint16_t *list = reinterpret_cast<const uint16_t *>(chunks);
        const uint32_t n = 4 * nch;
        const bool split = !a.exact && BS > 64;
        const bool second = split && tid >= BS / 2;
        for (uint32_t j = second ? tid - BS / 2 : tid; j < n; j += split ? BS / 2 : BS) {
          const uint32_t w = list[j], le = w >> 2;
          if (w == kNoSlot) continue;
          const int t = (int)(w & 3u);
          const uint2 q = el[le];
          const unsigned long long nd = (unsigned long long)q.y << 32 | q.x;
          auto node = [&](int k) { return (uint32_t)(nd >> (16 * (k & 3))) & 0xffffu; };
          const double p1 = up[node(t + 1)], p2 = up[node(t + 2)], p3 = up[node(t + 3)];
          const double *g = GEO ? gl + 6 * le : a.geo + 6 * ((size_t)si.eoff + le);
          const uint32_t ix = compat_relabel(t);
          const double e12 = g[ix & 7u], e13 = g[(ix >> 3) & 7u], e23 = g[(ix >> 6) & 7u], e14 = g[(ix >> 9) & 7u],
                       e24 = g[(ix >> 12) & 7u], e34 = g[ix >> 15];
          double v;
          if (a.exact)
            v = cand_core<double>(e12, e13, e23, e14, e24, e34, p1, p2, p3, DBL_MAX);
          else if (!split)
            v = fmin(cand_ref_a(e12, e13, e23, e14, e24, e34, p1, p2, p3),
                     cand_ref_b(e12, e23, e14, e24, e34, p1, p2, p3));
          else if (second)
            v = cand_ref_b(e12, e23, e14, e24, e34, p1, p2, p3);
          else
            v = cand_ref_a(e12, e13, e23, e14, e24, e34, p1, p2, p3);
          atomicMin(&tmin[node(t)], (unsigned long long)__double_as_longlong(v));
        }
      };
      for (uint32_t par = 0;; par ^= 1u) {
        __syncthreads();
        const uint32_t n = misc[par];
        if (n == 0) break;  // uniform
        // a: candidates of narrow copies
        evaluate(lp, n);
        __syncthreads();
        // b: reduce, window test, convergence test; a copy that stays narrow
        // is listed for the next sweep
        bool froze = false;
        int8_t prev = FIM_FAR;  // state before being marked (c)
        if (own && st == FIM_NARROW) {
          const double c = __longlong_as_double((long long)tmin[l]), old = p;
          const double nw = c < old ? c : old;
          tmin[l] = kDmaxBits;
          p = nw;
          phi_l[l] = nw;
          if (nw - a.phi_start > a.dt) {
            st = FIM_NEXT;
            st_l[l] = st;
          } else if (fabs(old - nw) < (1e-6 * (1 + (old + nw) * .5))) {
            froze = true;
          } else {
            append(lp, &misc[par ^ 1u], l);
          }
          up[l] = offer(st, p);
        }
        const uint64_t fm = __ballot(froze);
        if (lane == 0) {
          fz[tid >> 5] = (uint32_t)fm;
          if (BS > 32) fz[(tid >> 5) + 1] = (uint32_t)(fm >> 32);
        }
        __syncthreads();
        if (tid == 0) misc[par] = 0u;  // every thread has read it
        uint32_t any = 0;
#pragma unroll
        for (int k = 0; k < BS / 32; ++k) any |= fz[k];
        if (any == 0u) continue;  // uniform
        // c: copies that are not narrow and lie downwind of a just-frozen
        // neighbour are marked
        for (uint32_t e = tid; e < ne; e += BS) {
          const uint2 q = el[e];
          const uint32_t nd[4] = {q.x & 0xffffu, q.x >> 16, q.y & 0xffffu, q.y >> 16};
          double first = DBL_MAX;  // earliest just-frozen node
          bool f = false;
#pragma unroll
          for (int k = 0; k < 4; ++k)
            if (flag_at(fz, nd[k])) {
              f = true;
              first = fmin(first, phi_l[nd[k]]);
            }
          if (!f) continue;
#pragma unroll
          for (int k = 0; k < 4; ++k)
            if (st_l[nd[k]] != FIM_NARROW && first < phi_l[nd[k]]) atomicOr(&mk[nd[k] >> 5], 1u << (nd[k] & 31u));
        }
        __syncthreads();
        // d: candidates of marked copies (a marked copy offers nothing)
        const bool marked = own && flag_at(mk, l);
        if (marked) {
          prev = st;
          up[l] = DBL_MAX;
          append(lq, &misc[2], l);
        }
        __syncthreads();
        const uint32_t nq = misc[2];
        if (nq) {  // uniform
          evaluate(lq, nq);
          __syncthreads();
        }
        // e, f: accept improvements; freeze
        if (froze) {
          st = FIM_FROZEN;
          st_l[l] = st;
          up[l] = offer(st, p);
        }
        if (marked) {
          const double c = __longlong_as_double((long long)tmin[l]), old = p;
          tmin[l] = kDmaxBits;
          const double nw = c < old ? c : old;
          p = nw;
          phi_l[l] = nw;
          st = prev;
          if (nw < old) {
            // accepted; a copy that was frozen freezes again (phase f)
            st = prev == FIM_FROZEN ? (int8_t)FIM_FROZEN : (int8_t)FIM_NARROW;
            if (st == FIM_NARROW) append(lp, &misc[par ^ 1u], l);
          }
          st_l[l] = st;
          up[l] = offer(st, p);
          atomicAnd(&mk[l >> 5], ~(1u << (l & 31u)));
        }
        if (tid == 0) misc[2] = 0u;
      }
    }
    // write back what changed; ev: the earliest window time at which
    // update_states would change a copy (frozen: p + apd, tail: p + apd /
    // 0.91, as update_states computes them; narrow or next: now)
    bool pend = false;
    double ev = INFINITY;
    compat_record(a, si.ioff, own && p != p0, si.coff + l, &misc[6]);
    if (own) {
      if (p != p0) a.phi[si.coff + l] = p;
      if (st != st0) a.st[si.coff + l] = st;
      pend = st == FIM_NARROW || st == FIM_NEXT;
      if (pend)
        ev = -INFINITY;
      else if (st == FIM_FROZEN)
        ev = p + a.apd;
      else if (st == FIM_TAIL)
        ev = p + a.apd / 0.91;
    }
    pend_wg += (uint32_t)__syncthreads_count(pend);
    ev = block_min0(ev, evslot);
    if (tid == 0) {
      a.nexte[s] = ev;
      a.vcnt[s] = misc[6];
    }
  }
  if (tid == 0) compat_finish(a, nlist, pend_wg);
}

// Assembles the submeshes' blocks (CompatSub), one workgroup per submesh, from
// the plain arrays.  On the host, and copied from there, the 144 MB of the 2M-tet
// slab took 10 ms more of a context's creation (20 against 9 to 10; 8.2 with the
// general kernel alone; this kernel takes 0.1).
struct CompatBlockArgs {
  const CompatSub *csub;
  const uint2 *e2n;
  const uint32_t *n2e_dsp;
  const uint16_t *n2e_le;
  const uint8_t *n2e_pos;
  const uint4 *geo;  // FP64 geometry, three words an element; null: not in the blocks
  uint4 *blob;
  uint32_t nsub;
};
__global__ __launch_bounds__(256) void k_compat_block(CompatBlockArgs a) {
  __shared__ uint32_t off[512 + 1];  // chunks before each copy; at most 512 copies (k_compat_small)
  const uint32_t tid = threadIdx.x;
  for (uint32_t s = blockIdx.x; s < a.nsub; s += gridDim.x) {
    const CompatSub q = a.csub[s];
    const uint32_t nd = (2 * (q.nn + 1) + 15) / 16, nel = (8 * q.ne + 15) / 16, nsl = (8 * q.nch + 15) / 16;
    uint4 *block = a.blob + q.boff;
    const uint32_t *dsp = a.n2e_dsp + q.coff;
    if (tid < 3) block[(tid == 0 ? nd : tid == 1 ? nd + nel : nd + nel + nsl) - 1] = make_uint4(0u, 0u, 0u, 0u);  // ends
    if (tid < 64) {
      uint32_t before = 0;
      for (uint32_t l0 = 0; l0 < q.nn; l0 += 64) {
        const uint32_t l = l0 + tid, n = l < q.nn ? (dsp[l + 1] - dsp[l] + 3) / 4 : 0u;
        uint32_t sum = n;
        for (int d = 1; d < 64; d <<= 1) {
          const uint32_t x = __shfl_up(sum, d);
          if (tid >= (uint32_t)d) sum += x;
        }
        if (l < q.nn) off[l] = before + sum - n;
        before += __shfl(sum, 63);
      }
      if (tid == 0) off[q.nn] = before;
    }
    __syncthreads();
    uint16_t *o = reinterpret_cast<uint16_t *>(block);
    for (uint32_t l = tid; l <= q.nn; l += 256) o[l] = (uint16_t)off[l];
    uint2 *en = reinterpret_cast<uint2 *>(block + nd);
    for (uint32_t e = tid; e < q.ne; e += 256) en[e] = a.e2n[(size_t)q.eoff + e];
    uint16_t *sl = reinterpret_cast<uint16_t *>(block + nd + nel);
    for (uint32_t l = tid; l < q.nn; l += 256) {
      const uint32_t kb = dsp[l], n = dsp[l + 1] - kb;
      for (uint32_t k = 0; k < (n + 3) / 4 * 4; ++k)
        sl[4 * off[l] + k] = k < n ? (uint16_t)((uint32_t)a.n2e_le[kb + k] << 2 | a.n2e_pos[kb + k]) : kNoSlot;
    }
    if (a.geo)
      for (uint32_t i = tid; i < 3 * q.ne; i += 256) block[nd + nel + nsl + i] = a.geo[3 * (size_t)q.eoff + i];
    __syncthreads();  // off is free
  }
}

// per copy: its vertex if it has other copies, else kNoVertex
__global__ __launch_bounds__(256) void k_compat_shared(const uint32_t *c2g, const uint32_t *g2c_dsp, uint32_t *cshared,
                                                       uint32_t ncopy) {
  for (uint32_t c = blockIdx.x * 256 + threadIdx.x; c < ncopy; c += gridDim.x * 256) {
    const uint32_t v = c2g[c];
    cshared[c] = g2c_dsp[v + 1] - g2c_dsp[v] > 1u ? v : kNoVertex;
  }
}

// Start of a window.  sync_step2 (min over the copies of each shared vertex)
// and the list of submeshes the window's pass has to run on: those whose
// copies' own clocks are due (nexte; -inf when something is narrow or next)
// and those a shared vertex was lowered in.  A submesh left out would come out
// of the pass unchanged: nothing narrow or next, and its frozen and tail
// copies all stay put at this window time.
// The copies of a vertex are equal after a sync and a seed sets all of them,
// so only the vertices that the last window's pass recorded can differ: one
// wave per submesh of that window's list goes through its records.  A vertex
// recorded by several submeshes is merged by each of them: all find the same
// minimum and write nothing else.
struct CompatSyncArgs {
  const SubInfo *sub;
  const uint32_t *last, *nlast;  // the last window's list
  const uint32_t *vrec, *vcnt;
  const uint32_t *g2c_dsp, *g2c, *c2s;
  double *phi;
  int8_t *st;
  const double *nexte;
  uint32_t nsub;
  double cur;
  uint32_t *list, *cnt, *next_cnt;  // this window's list; the next one's count, cleared
  uint32_t *mark, stamp;            // mark[s] == stamp: s is on this window's list
};

__global__ __launch_bounds__(256) void k_compat_sync(CompatSyncArgs a) {
  auto queue = [&](uint32_t s) {
    if (a.mark[s] != a.stamp && atomicExch(&a.mark[s], a.stamp) != a.stamp) a.list[atomicAdd(a.cnt, 1u)] = s;
  };
  const uint32_t t0 = blockIdx.x * blockDim.x + threadIdx.x, nt = gridDim.x * blockDim.x;
  if (t0 == 0) *a.next_cnt = 0u;
  for (uint32_t s = t0; s < a.nsub; s += nt)
    if (!(a.nexte[s] > a.cur)) queue(s);
  const uint32_t nlast = *a.nlast;
  for (uint32_t i = t0 >> 6; i < nlast; i += nt >> 6) {
    const uint32_t s = a.last[i], n = a.vcnt[s], off = a.sub[s].ioff;
    for (uint32_t r = threadIdx.x & 63; r < n; r += 64) {
      const uint32_t v = a.vrec[off + r], b = a.g2c_dsp[v], e = a.g2c_dsp[v + 1];
      double mn = DBL_MAX;
      for (uint32_t k = b; k < e; ++k) {
        const double c = a.phi[a.g2c[k]];
        if (c < mn) mn = c;
      }
      for (uint32_t k = b; k < e; ++k) {
        const uint32_t c = a.g2c[k];
        if (mn < a.phi[c]) {
          a.phi[c] = mn;
          a.st[c] = FIM_NARROW;
          queue(a.c2s[c]);
        }
      }
    }
  }
}

__global__ void k_compat_seed(const uint2 *ic, uint32_t n, double t0, const uint32_t *c2s, double *phi,
                              int8_t *st, double *nexte) {
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    phi[ic[i].y] = t0;
    st[ic[i].y] = FIM_NARROW;
    nexte[c2s[ic[i].y]] = -INFINITY;
  }
}

__global__ void k_compat_gather(const double *phi, const int8_t *st, const uint32_t *g2c_dsp,
                                const uint32_t *g2c, uint32_t nn, double *out_phi, int32_t *out_st) {
  for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < nn; v += gridDim.x * blockDim.x) {
    double m = DBL_MAX;
    int32_t s = FIM_FAR;
    for (uint32_t k = g2c_dsp[v]; k < g2c_dsp[v + 1]; ++k) {
      const uint32_t c = g2c[k];
      if (phi[c] < m) m = phi[c];
      if (st[c] > s) s = st[c];
    }
    out_phi[v] = m;
    out_st[v] = s;
  }
}

uint32_t al16(uint32_t x) { return (x + 15u) & ~15u; }

template <class T>
T *dalloc(size_t n, std::vector<void *> &owned) {
  void *p = nullptr;
  if (n == 0) n = 1;
  HIPCHECK(hipMalloc(&p, n * sizeof(T)));
  owned.push_back(p);
  return static_cast<T *>(p);
}

template <class T>
T *dupload(const std::vector<T> &v, std::vector<void *> &owned) {
  T *p = dalloc<T>(v.size(), owned);
  if (!v.empty()) HIPCHECK(hipMemcpy(p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
  return p;
}

// device buffers of a scope
struct Buffers {
  std::vector<void *> v;
  ~Buffers() {
    for (void *p : v) (void)hipFree(p);
  }
};

}  // namespace
}  // namespace fim

// Scratch of fim_support_noalloc: the best candidate time (float bits) of
// every vertex, for meshes of up to kNoAllocMaxVertices vertices (4 MiB).
// One copy per device, held until the process ends.  Host code never uses
// this name as an address: fim_create looks the device address up once per
// device (noalloc_scratch) and the kernels get that pointer.
constexpr uint32_t kNoAllocMaxVertices = 1u << 20;
static __device__ __align__(256) uint32_t scratch[kNoAllocMaxVertices];

using namespace fim;

struct fim_ctx {
  int dev = 0;
  hipStream_t stream = nullptr;
  fim_opts o{};
  uint32_t nsub = 0, ncopy = 0, ninst = 1, nn = 0, n_if = 0;
  int64_t ne = 0;
  int32_t nn_max = 0, ne_max = 0;
  std::vector<void *> owned;
  // host copies for seeding
  std::vector<uint32_t> g2c_dsp, g2c;
  // pack
  SubInfo *d_sub = nullptr;
  uint2 *d_e2n = nullptr;
  float *d_geo32 = nullptr;
  float4 *d_hgt = nullptr;
  double *d_geo64 = nullptr;
  uint8_t *d_ereg = nullptr;
  uint32_t *d_c2g = nullptr, *d_c2s = nullptr, *d_g2c_dsp = nullptr, *d_g2c = nullptr;
  uint16_t *d_if_l = nullptr;
  uint4 *d_if_fo = nullptr, *d_if_os = nullptr;
  uint32_t *d_n2e_dsp = nullptr, *d_n2n_dsp = nullptr;
  uint16_t *d_n2e_le = nullptr, *d_n2n_lv = nullptr;
  uint8_t *d_n2e_pos = nullptr;
  uint4 *d_erec = nullptr, *d_adj = nullptr, *d_adj_more = nullptr;
  uint32_t *d_adj_ptr = nullptr;
  // converge state
  float *d_phi = nullptr, *d_rscale = nullptr;
  uint8_t *d_dirty = nullptr;
  uint32_t *d_act = nullptr, *d_cnt = nullptr;
  uint32_t *d_start = nullptr;  // n_inst: iteration each instance was (re)seeded at
  float *d_winst = nullptr;     // n_inst: time window per iteration (us), 0 = off
  // per-instance region factors and windows as set on the host
  // (fim_set_scaling, fim_set_window), uploaded together before the next
  // launch that reads them: setting up a batch costs no device round trip
  // per instance
  std::vector<float> h_rscale, h_winst;
  float *h_par = nullptr, *d_par = nullptr;  // the two on their way: pinned, and its device address
  bool params_dirty = false;
  uint32_t *d_flag = nullptr;   // n_inst: scratch for instance queries / lists
  uint32_t *d_inbox = nullptr;  // 2 x n_inst x interface entries
  uint32_t *d_ifc = nullptr;    // per interface entry: its copy
  bool inbox_left = false;      // the last run stopped with pushes in the inbox
  bool direct_plan = false;     // a bucket is one work unit
  uint32_t next_iter = 0;       // the next iteration's number, or one more
  uint2 *d_ifm = nullptr;
  uint32_t wps = 1;
  WorkList wl[3] = {};
  uint32_t unit = 2, maxch = 1;
  float *d_wake = nullptr, *d_wpush = nullptr;
  // compat state
  double *d_phi64 = nullptr;
  int8_t *d_st = nullptr;
  double *d_nexte = nullptr;  // per submesh: earliest window time a copy changes
  // submesh lists of this and the last window (two in turn), their counts
  // (three in turn), the stamps of the last window that listed a submesh (0:
  // none), the pass's end counter and its records of changed shared vertices
  uint32_t *d_list = nullptr, *d_lcnt = nullptr, *d_mark = nullptr;
  CompatSub *d_csub = nullptr;
  uint4 *d_blob = nullptr;
  uint32_t *d_cshared = nullptr, *d_vrec = nullptr, *d_vcnt = nullptr;
  unsigned long long *d_done = nullptr;
  uint32_t stamp = 0, turn = 0;  // of the last window
  bool compat_small = false, compat_geo = false;  // k_compat_small, with geometry in LDS
  // shared
  unsigned long long *d_stats = nullptr;
  uint32_t *h_pin = nullptr, *d_pin = nullptr;  // pinned host words and their device address
  // (instance, copy) pairs to seed: pinned, and the device address
  uint2 *h_seed = nullptr, *d_seed = nullptr;
  size_t seed_cap = 0;
  float *d_tmpf = nullptr;
  // a downloaded map on its way out: pinned, written by the gather kernel
  // (float32 times; in compat mode float64 times, then int32 states)
  unsigned char *h_map = nullptr, *d_map = nullptr;
  uint32_t *d_tmpu = nullptr;
  hipGraph_t graph = nullptr;
  hipGraphExec_t gexec = nullptr;
  hipGraphNode_t node = nullptr;  // the last one, while the graph is built
  bool building = false;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  hipEvent_t evc = nullptr;  // end of an iteration chunk's read-back
  std::vector<hipEvent_t> kev;  // profile: events around each compute launch
  ConvArgs ca{};
  CompatArgs xa{};
  uint32_t lds_conv = 0, lds_compat = 0;
  int grid = 0, block = 256, graph_iters = 8;
  int band_wpe = 8;  // waves per SIMD the band kernel's registers are sized for
  bool band_pairs = false;  // band kernel evaluates (element, target) pairs
  bool band_gather = false; // its GATHER variant
  bool direct = false;      // launch iterations directly instead of replaying the graph
  fim_stats_t stats{};
};

namespace {

template <bool GATHER>
const void *band_pairs_ptr(int block, int wpe) {
  if (block == 512) return (const void *)k_conv_band<512, 8, true, GATHER>;
  if (wpe == 5) return (const void *)k_conv_band<256, 5, true, GATHER>;
  if (wpe == 6) return (const void *)k_conv_band<256, 6, true, GATHER>;
  if (wpe == 7) return (const void *)k_conv_band<256, 7, true, GATHER>;
  return (const void *)k_conv_band<256, 8, true, GATHER>;
}

const void *conv_kernel_ptr(const fim_ctx *c) {
  const int block = c->block, wpe = c->band_wpe;
  if (c->o.staged) switch (block) {
      case 64: return (const void *)k_conv_compute<64>;
      case 128: return (const void *)k_conv_compute<128>;
      case 512: return (const void *)k_conv_compute<512>;
      default: return (const void *)k_conv_compute<256>;
    }
  if (c->band_pairs) {
    if (wpe <= 4)
      return block == 512 ? (const void *)k_conv_band<512, 4, true, false> : (const void *)k_conv_band<256, 4, true, false>;
    return c->band_gather ? band_pairs_ptr<true>(block, wpe) : band_pairs_ptr<false>(block, wpe);
  }
  switch (block) {
    case 64: return (const void *)k_conv_band<64, 8, false, false>;
    case 128: return (const void *)k_conv_band<128, 8, false, false>;
    case 512: return (const void *)k_conv_band<512, 8, false, false>;
    default:
      if (wpe <= 5) return (const void *)k_conv_band<256, 5, false, false>;
      if (wpe == 6) return (const void *)k_conv_band<256, 6, false, false>;
      if (wpe == 7) return (const void *)k_conv_band<256, 7, false, false>;
      return (const void *)k_conv_band<256, 8, false, false>;
  }
}

// a kernel of an iteration: into the context's stream or, while its graph is
// built, as the graph's next node
void launch(fim_ctx *c, const void *f, dim3 grid, dim3 block, void **args, uint32_t lds) {
  if (!c->building) {
    HIPCHECK(hipLaunchKernel(f, grid, block, args, lds, c->stream));
    return;
  }
  hipKernelNodeParams n{};
  n.func = const_cast<void *>(f);
  n.gridDim = grid;
  n.blockDim = block;
  n.kernelParams = args;  // copied by the call
  n.sharedMemBytes = lds;
  hipGraphNode_t node;
  HIPCHECK(hipGraphAddKernelNode(&node, c->graph, c->node ? &c->node : nullptr, c->node ? 1 : 0, &n));
  c->node = node;
}

void launch_conv_compute(fim_ctx *c, const ConvArgs &a) {
  void *args[] = {const_cast<ConvArgs *>(&a)};
  launch(c, conv_kernel_ptr(c), dim3(c->grid), dim3(c->block), args, c->lds_conv);
}

void set_lds_attr(fim_ctx *c) {
  const void *f = conv_kernel_ptr(c);
  HIPCHECK(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)c->lds_conv));
}

const void *compat_kernel_ptr(const fim_ctx *c) {
  const bool geo = c->compat_geo;
  if (c->compat_small) switch (c->block) {
      case 64: return geo ? (const void *)k_compat_small<64, true> : (const void *)k_compat_small<64, false>;
      case 128: return geo ? (const void *)k_compat_small<128, true> : (const void *)k_compat_small<128, false>;
      case 512: return geo ? (const void *)k_compat_small<512, true> : (const void *)k_compat_small<512, false>;
      default: return geo ? (const void *)k_compat_small<256, true> : (const void *)k_compat_small<256, false>;
    }
  switch (c->block) {
    case 64: return (const void *)k_compat_compute<64>;
    case 128: return (const void *)k_compat_compute<128>;
    case 512: return (const void *)k_compat_compute<512>;
    default: return (const void *)k_compat_compute<256>;
  }
}

void launch_compat_compute(fim_ctx *c, const CompatArgs &a) {
  void *args[] = {const_cast<CompatArgs *>(&a)};
  HIPCHECK(hipLaunchKernel(compat_kernel_ptr(c), dim3(c->grid), dim3(c->block), args, c->lds_compat, c->stream));
}

int blocks_for(size_t n, int bs) { return (int)std::max<size_t>(1, std::min<size_t>((n + bs - 1) / bs, 65536)); }

// work units of list l; the buckets of list z (consumed), if any, are cleared
void launch_plan(fim_ctx *c, int l, int z) {
  PlanArgs pa{c->wl[l].bcnt, c->wl[l].plan, c->wl[l].cnt, z >= 0 ? c->wl[z].bcnt : nullptr,
              c->nsub, c->unit, c->maxch};
  void *args[] = {&pa};
  launch(c, (const void *)k_conv_plan, dim3(1), dim3(1024), args, 0);
}

// one global iteration k: work lists rotate over three buffers; iteration k
// reads list k%3 and appends to (k+1)%3, whose units are planned then (by the
// items themselves when a bucket is one unit) and the buckets of list k%3
// cleared
void enqueue_iteration(fim_ctx *c, int k, bool timed) {
  const int p = k % 3, q = (k + 1) % 3;
  if (timed) HIPCHECK(hipEventRecord(c->kev[2 * k], c->stream));
  ConvArgs a = c->ca;
  a.cur = c->wl[p];
  a.nxt = c->wl[q];
  a.old_cnt = c->wl[(k + 2) % 3].cnt;
  launch_conv_compute(c, a);
  if (timed) HIPCHECK(hipEventRecord(c->kev[2 * k + 1], c->stream));
  if (!c->direct_plan) launch_plan(c, q, p);
}

// The iterations as a chain of kernel nodes.  (Captured from the stream, they
// failed, and so did the other's call, where another thread used the null
// stream meanwhile, for instance to create a context.)
void build_graph(fim_ctx *c) {
  HIPCHECK(hipGraphCreate(&c->graph, 0));
  c->building = true;
  c->node = nullptr;
  try {
    for (int i = 0; i < c->graph_iters; ++i) enqueue_iteration(c, i, false);
    c->building = false;
    HIPCHECK(hipGraphInstantiate(&c->gexec, c->graph, nullptr, nullptr, 0));
  } catch (...) {
    c->building = false;
    (void)hipGraphDestroy(c->graph);
    c->graph = nullptr;
    c->gexec = nullptr;
    throw;
  }
}

// the list that the next run starts on, for kernels between runs
Queue list0(const fim_ctx *c) {
  return Queue{c->wl[0], c->d_act, 0u, c->nsub, c->ninst, c->direct_plan ? 1u : 0u};
}

// before a call reads or replaces times while pushes may be in the inbox
void settle(fim_ctx *c) {
  if (!c->inbox_left) return;
  c->inbox_left = false;
  if (c->n_if == 0) return;
  const DrainArgs a{c->d_ifc, c->d_c2s, c->d_inbox, c->d_phi, c->d_wake, c->d_dirty, c->wl[0].cnt + kIterWord,
                    c->n_if, c->ncopy, c->nsub, c->ninst};
  k_conv_drain<<<dim3(std::min(blocks_for(c->n_if, 256), 256), std::min<uint32_t>(c->ninst, 1024u)), 256, 0,
                 c->stream>>>(a);
  HIPCHECK(hipGetLastError());
}

// continues the numbering of the iterations at `to`, or to + 1
void renumber(fim_ctx *c, uint32_t to) {
  const size_t nss = (size_t)c->ninst * c->nsub;
  uint32_t *iter = c->wl[0].cnt + kIterWord;
  k_conv_renumber<<<std::min(blocks_for(std::max<size_t>(nss, c->ninst), 256), 2048), 256, 0, c->stream>>>(
      iter, to, c->d_act, nss, c->d_start, c->ninst);
  k_iter_set<<<1, 1, 0, c->stream>>>(iter, to);
  HIPCHECK(hipGetLastError());
  c->next_iter = to + 1u;
}

void check_inst(const fim_ctx *c, int32_t inst) {
  if (inst < 0 || (uint32_t)inst >= c->ninst) throw Error(FIM_EINVAL, "instance index out of range");
}

std::vector<uint32_t> copies_of(const fim_ctx *c, const int64_t *vtx, int64_t n) {
  std::vector<uint32_t> out;
  for (int64_t i = 0; i < n; ++i) {
    if (vtx[i] < 0 || vtx[i] >= (int64_t)c->nn) throw Error(FIM_EINVAL, "seed vertex out of range");
    for (uint32_t k = c->g2c_dsp[vtx[i]]; k < c->g2c_dsp[vtx[i] + 1]; ++k) out.push_back(c->g2c[k]);
  }
  return out;
}

void destroy_ctx(fim_ctx *c) {
  if (!c) return;
  if (c->gexec) (void)hipGraphExecDestroy(c->gexec);
  if (c->graph) (void)hipGraphDestroy(c->graph);
  if (c->ev0) (void)hipEventDestroy(c->ev0);
  if (c->ev1) (void)hipEventDestroy(c->ev1);
  if (c->evc) (void)hipEventDestroy(c->evc);
  for (hipEvent_t e : c->kev)
    if (e) (void)hipEventDestroy(e);
  for (void *p : c->owned) (void)hipFree(p);
  if (c->h_pin) (void)hipHostFree(c->h_pin);
  if (c->h_map) (void)hipHostFree(c->h_map);
  if (c->h_par) (void)hipHostFree(c->h_par);
  if (c->h_seed) (void)hipHostFree(c->h_seed);
  if (c->stream) (void)hipStreamDestroy(c->stream);
  delete c;
}

template <class F>
int guarded(F &&f) {
  try {
    f();
    return FIM_OK;
  } catch (const Error &e) {
    set_last_error(e.what());
    return e.code;
  } catch (const std::exception &e) {
    set_last_error(e.what());
    return FIM_EINVAL;
  } catch (...) {
    set_last_error("unknown error");
    return FIM_EINVAL;
  }
}

}  // namespace

namespace fim {

void *ctx_stream(fim_ctx *c) { return c->stream; }
int32_t ctx_device(const fim_ctx *c) { return c->dev; }
uint32_t ctx_vertices(const fim_ctx *c) { return c->nn; }
int32_t ctx_instances(const fim_ctx *c) { return (int32_t)c->ninst; }
bool ctx_converge(const fim_ctx *c) { return c->o.mode == FIM_MODE_CONVERGE; }

const float *ctx_gather(fim_ctx *c, int32_t inst) {
  check_inst(c, inst);
  k_conv_gather<<<blocks_for(c->nn, 256), 256, 0, c->stream>>>(c->d_phi, c->d_g2c_dsp, c->d_g2c, c->nn,
                                                               (size_t)inst * c->ncopy, c->d_tmpf);
  HIPCHECK(hipGetLastError());
  return c->d_tmpf;
}

float *ctx_field_buffer(fim_ctx *c) { return c->d_tmpf; }

void ctx_init_field(fim_ctx *c, int32_t inst, bool all_active) {
  check_inst(c, inst);
  settle(c);
  k_conv_init<<<blocks_for(c->ncopy, 256), 256, 0, c->stream>>>(c->d_tmpf, c->d_c2g, (uint32_t)inst,
                                                                 c->d_phi, c->d_dirty, c->ncopy,
                                                                 all_active ? 1 : 0);
  if (all_active)
    k_conv_queue_all<<<blocks_for(c->nsub, 256), 256, 0, c->stream>>>((uint32_t)inst, c->d_wake, list0(c));
  HIPCHECK(hipGetLastError());
}

// device address of `scratch` on the current device `dev`, looked up once
// per device (hipGetSymbolAddress) and kept
uint32_t *noalloc_scratch(int dev) {
  static std::mutex mu;
  static std::vector<uint32_t *> ptr;
  std::lock_guard<std::mutex> lock(mu);
  if (dev < 0) throw Error(FIM_EINVAL, "bad device ordinal");
  if ((size_t)dev >= ptr.size()) ptr.resize((size_t)dev + 1, nullptr);
  if (!ptr[dev]) {
    void *p = nullptr;
    HIPCHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) throw Error(FIM_EDEVICE, "no device address for the support scratch");
    ptr[dev] = static_cast<uint32_t *>(p);
  }
  return ptr[dev];
}

// uploads the per-instance factors and windows set since the last upload
// (the device must be current)
void flush_params(fim_ctx *c, bool clear_stats = false) {
  if (!c->params_dirty && !clear_stats) return;
  const uint32_t nr = c->params_dirty ? (uint32_t)c->h_rscale.size() : 0u;
  const uint32_t nw = c->params_dirty ? (uint32_t)c->h_winst.size() : 0u;
  if (c->params_dirty) {
    HIPCHECK(hipStreamSynchronize(c->stream));  // a kernel may still read the last ones (idle but after an error)
    std::memcpy(c->h_par, c->h_rscale.data(), nr * sizeof(float));
    std::memcpy(c->h_par + nr, c->h_winst.data(), nw * sizeof(float));
  }
  k_run_begin<<<blocks_for(nr + nw, 256), 256, 0, c->stream>>>(c->d_par, nr, c->d_rscale, nw, c->d_winst,
                                                              clear_stats ? c->d_stats : nullptr);
  HIPCHECK(hipGetLastError());
  c->params_dirty = false;
}

// support check of one instance with `best` (nn words of device memory) as
// the per-vertex candidate minimum
double support_into(fim_ctx *c, int32_t inst, uint32_t *best) {
  flush_params(c);
  settle(c);
  k_fill<uint32_t><<<blocks_for(c->nn, 256), 256, 0, c->stream>>>(best, c->nn, 0x7f800000u);
  k_conv_support<<<(int)std::min<uint32_t>(c->nsub, 4096u), 256, 0, c->stream>>>(
      c->d_sub, c->nsub, c->d_e2n, c->d_geo32, c->d_ereg, c->d_rscale, c->d_phi, c->d_c2g,
      (size_t)inst * c->ncopy, (uint32_t)inst, best);
  k_conv_gather<<<blocks_for(c->nn, 256), 256, 0, c->stream>>>(c->d_phi, c->d_g2c_dsp, c->d_g2c, c->nn,
                                                               (size_t)inst * c->ncopy, c->d_tmpf);
  k_fill<uint32_t><<<1, 64, 0, c->stream>>>(c->d_tmpu, 1, 0u);
  k_support_check<<<blocks_for(c->nn, 256), 256, 0, c->stream>>>(c->d_tmpf, best, c->nn, c->d_tmpu);
  HIPCHECK(hipGetLastError());
  HIPCHECK(hipMemcpyAsync(c->h_pin, c->d_tmpu, 4, hipMemcpyDeviceToHost, c->stream));
  HIPCHECK(hipStreamSynchronize(c->stream));
  float r;
  std::memcpy(&r, c->h_pin, 4);
  return r;
}

}  // namespace fim

extern "C" {

int fim_create(const fim_pack *pk, const fim_opts *o, fim_ctx **out) {
  return guarded([&] {
    if (!pk || !o || !out) throw Error(FIM_EINVAL, "null argument");
    *out = nullptr;
    const Pack &p = pk->p;
    fim_ctx *c = new fim_ctx();
    try {
      c->o = *o;
      c->dev = o->device;
      HIPCHECK(hipSetDevice(c->dev));
      (void)noalloc_scratch(c->dev);  // once per device: fim_support_noalloc's scratch
      // CUFIM_DIRECT_LAUNCH=1 launches the iterations' kernels directly instead
      // of replaying the graph of them (the same kernel sequence): for tools
      // that cannot trace graph launches
      {
        const char *dl = std::getenv("CUFIM_DIRECT_LAUNCH");
        c->direct = dl && dl[0] == '1';
      }
      HIPCHECK(hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking));
      HIPCHECK(hipEventCreate(&c->ev0));
      HIPCHECK(hipEventCreate(&c->ev1));
      HIPCHECK(hipEventCreate(&c->evc));
      if (o->mode != FIM_MODE_CONVERGE && o->mode != FIM_MODE_COMPAT)
        throw Error(FIM_EINVAL, "unknown mode");
      c->block = o->block ? o->block : (o->mode == FIM_MODE_CONVERGE ? 512 : 256);
      if (c->block != 64 && c->block != 128 && c->block != 256 && c->block != 512)
        throw Error(FIM_EINVAL, "block must be 64, 128, 256 or 512");
      if (o->waves < 0 || o->waves > 8) throw Error(FIM_EINVAL, "waves must be 0..8");
      c->ninst = o->mode == FIM_MODE_CONVERGE ? (uint32_t)std::max(1, o->n_instances) : 1u;
      // a multiple of 3 so every graph launch starts on list 0
      c->graph_iters = o->graph_iters > 0 ? 3 * ((o->graph_iters + 2) / 3) : 6;
      c->nsub = (uint32_t)p.nsub;
      c->ncopy = (uint32_t)p.ncopy;
      c->nn = (uint32_t)p.nn_global;
      c->ne = p.ne_global;
      c->nn_max = p.nn_max;
      c->ne_max = p.ne_max;
      if ((uint64_t)c->ninst * c->nsub >= (1ull << 32) || (uint64_t)c->ninst * c->ncopy >= (1ull << 40))
        throw Error(FIM_ELIMIT, "too many instances for this mesh");
      c->g2c_dsp = p.g2c_dsp;
      c->g2c = p.g2c;
      auto &ow = c->owned;
      Buffers tmp;  // what only kernels of this call read: until the stream is past them
      c->d_sub = dupload(p.sub, ow);
      {
        std::vector<uint2> e2(p.ne_global);
        for (int64_t e = 0; e < p.ne_global; ++e) {
          e2[e].x = (uint32_t)p.e2n_l[4 * e] | ((uint32_t)p.e2n_l[4 * e + 1] << 16);
          e2[e].y = (uint32_t)p.e2n_l[4 * e + 2] | ((uint32_t)p.e2n_l[4 * e + 3] << 16);
        }
        c->d_e2n = dupload(e2, ow);
      }
      c->d_ereg = dupload(p.ereg, ow);
      c->d_c2g = dupload(p.c2g, ow);
      c->d_c2s = dupload(p.c2s, ow);
      c->d_g2c_dsp = dupload(p.g2c_dsp, ow);
      c->d_g2c = dupload(p.g2c, ow);
      c->d_stats = dalloc<unsigned long long>(8, ow);
      HIPCHECK(hipHostMalloc((void **)&c->h_pin, 128, hipHostMallocDefault));
      HIPCHECK(hipHostGetDevicePointer((void **)&c->d_pin, c->h_pin, 0));
      const size_t per = o->mode == FIM_MODE_CONVERGE ? sizeof(float) : sizeof(double) + sizeof(int32_t);
      HIPCHECK(hipHostMalloc((void **)&c->h_map, std::max<size_t>(c->nn * per, 64), hipHostMallocDefault));
      HIPCHECK(hipHostGetDevicePointer((void **)&c->d_map, c->h_map, 0));
      c->d_tmpu = dalloc<uint32_t>(4, ow);
      HIPCHECK(hipMemset(c->d_stats, 0, 8 * sizeof(unsigned long long)));
      if (o->mode == FIM_MODE_CONVERGE) {
        c->lds_conv = 0;
        c->unit = o->unit > 0 ? (uint32_t)o->unit : 2u;
        c->maxch = (c->ninst + c->unit - 1) / c->unit;
        if ((uint64_t)c->nsub * c->maxch >= (1ull << 32)) throw Error(FIM_ELIMIT, "too many work units");
        // a bucket that fits one unit is planned by its first item; only
        // batches of more instances need the plan kernel (4 us, and as much
        // again between two launches, out of 60 for an iteration of a single
        // solve on the 2M-tet slab)
        c->direct_plan = c->maxch == 1;
        int ncu = 256;
        HIPCHECK(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, c->dev));
        c->band_pairs = !o->staged && band_with_pairs(c->block, c->ne_max);
        const bool few = c->band_pairs && c->direct_plan && o->waves == 0 && few_submeshes(c->nsub, ncu);
        if (few) c->band_wpe = 4;
        const ConvergeCarve lds = converge_carve(c->nn_max, c->ne_max, c->block, o->staged != 0,
                                                 !c->band_pairs ? 0 : few ? 2 : 1);
        c->lds_conv = lds.bytes;
        if (c->lds_conv > 160 * 1024)
          throw Error(FIM_ELIMIT, "largest submesh needs " + std::to_string(c->lds_conv) +
                                      " B of LDS (limit 163840); use a smaller partition budget");
        c->d_geo32 = dupload(p.geo32, ow);
        if (o->staged) {  // the band kernel's records have bounds of their own
          std::vector<float4> hg(p.ne_global);
          for (int64_t e = 0; e < p.ne_global; ++e)
            hg[e] = make_float4(p.hgt32[4 * e], p.hgt32[4 * e + 1], p.hgt32[4 * e + 2], p.hgt32[4 * e + 3]);
          c->d_hgt = dupload(hg, ow);
        }
        if (!o->staged) {
          if (c->nn_max > 32768) throw Error(FIM_ELIMIT, "submeshes above 32768 copies");
          std::call_once(pk->bounds_once, [&] { pk->bounds = element_bounds(p); });
          const ElementBounds &eb = pk->bounds;
          std::vector<uint4> rec(3 * (size_t)p.ne_global);
          parallel_ranges((size_t)p.ne_global, 65536, [&](size_t b, size_t end) {
            for (size_t e = b; e < end; ++e) {
              const uint16_t *n = &p.e2n_l[4 * e];
              const uint32_t r = p.ereg.empty() ? 0u : (p.ereg[e] & 3u);
              const float *g = &p.geo32[6 * e];
              auto fb = [](float x) { uint32_t u; std::memcpy(&u, &x, 4); return u; };
              rec[3 * e] = make_uint4((uint32_t)n[0] | ((uint32_t)n[1] << 16) | ((r & 1u) << 15) | ((r & 2u) << 30),
                                      (uint32_t)n[2] | ((uint32_t)n[3] << 16), fb(g[0]), fb(g[1]));
              rec[3 * e + 1] = make_uint4(fb(g[2]), fb(g[3]), fb(g[4]), fb(g[5]));
              uint32_t w[3];
              std::memcpy(w, &eb.b[12 * e], 12);
              rec[3 * e + 2] = make_uint4(w[0], w[1], w[2], fb(eb.scale[e]));
            }
          });
          c->d_erec = dupload(rec, ow);
          // four words of eight element ids per copy (mark_incident)
          std::vector<uint4> adj(4 * (size_t)p.ncopy), more;
          std::vector<uint32_t> aptr(p.ncopy, 0u);
          for (int64_t cc = 0; cc < p.ncopy; ++cc) {
            const uint32_t kb = p.n2e_dsp[cc], n = p.n2e_dsp[cc + 1] - kb;
            if (n == 0 || n > 504) throw Error(FIM_ELIMIT, "vertex with no or over 504 incident elements");
            uint16_t *q = reinterpret_cast<uint16_t *>(&adj[4 * (size_t)cc]);
            for (uint32_t k = 0; k < 32; ++k) q[k] = p.n2e_le[kb + (k < n ? k : 0u)];
            if (n <= 32) continue;
            q[31] = (uint16_t)kAdjMore;
            const size_t off = more.size(), words = (n - 31 + 7) / 8;
            if (off >= (1u << 26)) throw Error(FIM_ELIMIT, "adjacency above 2^26 chunks");
            aptr[cc] = (uint32_t)(off << 6 | words);
            more.resize(off + words);
            uint16_t *o = reinterpret_cast<uint16_t *>(&more[off]);
            for (uint32_t k = 0; k < 8 * words; ++k) o[k] = p.n2e_le[kb + (31 + k < n ? 31 + k : 0u)];
          }
          c->d_adj = dupload(adj, ow);
          c->d_adj_ptr = dupload(aptr, ow);
          c->d_adj_more = dupload(more, ow);
        }
        c->d_if_l = dupload(p.if_l, ow);
        {
          // interface entry of a copy
          std::vector<uint32_t> ifc(p.if_l.size()), ent(p.ncopy, 0u);
          for (const SubInfo &si : p.sub)
            for (uint32_t e = si.ioff; e < si.ioff + si.ni; ++e) {
              ifc[e] = si.coff + p.if_l[e];
              ent[ifc[e]] = e;
            }
          c->d_ifc = dupload(ifc, ow);
          std::vector<uint4> os(p.if_other.size()), fo(p.if_l.size());
          for (size_t e = 0; e < fo.size(); ++e) {
            const uint32_t k0 = p.if_dsp[e], k1 = p.if_dsp[e + 1];
            if (k1 <= k0) throw Error(FIM_EINVAL, "interface entry without another copy");
            for (uint32_t k = k0; k < k1; ++k) {
              const uint32_t o = p.if_other[k];
              os[k] = make_uint4(o, p.c2s[o], ent[o], k + 1 < k1 ? k + 2 : 0u);
            }
            fo[e] = os[k0];
          }
          c->d_if_os = dupload(os, ow);
          c->d_if_fo = dupload(fo, ow);
        }
        const size_t ncs = (size_t)c->ninst * c->ncopy, nss = (size_t)c->ninst * c->nsub;
        if (nss >= (1ull << 32)) throw Error(FIM_ELIMIT, "instances x submeshes exceed 2^32");
        c->d_phi = dalloc<float>(ncs, ow);
        c->d_dirty = dalloc<uint8_t>(ncs, ow);
        {
          const size_t nib = 2 * (size_t)c->ninst * p.if_l.size();
          c->d_inbox = dalloc<uint32_t>(nib, ow);
          if (nib) k_fill<uint32_t><<<blocks_for(nib, 256), 256, 0, c->stream>>>(c->d_inbox, nib, 0x7f800000u);
          c->d_start = dalloc<uint32_t>(c->ninst, ow);
          c->h_winst.assign(c->ninst, (float)std::max(0.0, o->window));
          c->d_winst = dupload(c->h_winst, ow);
          c->d_flag = dalloc<uint32_t>(c->ninst, ow);
          HIPCHECK(hipMemset(c->d_start, 0, sizeof(uint32_t) * c->ninst));
          // per submesh: interface-copy bits of each 32 local copies and the
          // number of interface entries before that word (if_l ascends)
          c->wps = (uint32_t)((c->nn_max + 63) / 64 * 2);
          std::vector<uint2> ifm((size_t)c->nsub * c->wps, make_uint2(0u, 0u));
          for (uint32_t s = 0; s < c->nsub; ++s) {
            const SubInfo &si = p.sub[s];
            for (uint32_t j = 0; j < si.ni; ++j) {
              const uint32_t l = p.if_l[si.ioff + j];
              if (j > 0 && l <= p.if_l[si.ioff + j - 1]) throw Error(FIM_EINVAL, "interface list not ascending");
              ifm[(size_t)s * c->wps + (l >> 5)].x |= 1u << (l & 31);
            }
            uint32_t run = 0;
            for (uint32_t w = 0; w < c->wps; ++w) {
              ifm[(size_t)s * c->wps + w].y = run;
              run += (uint32_t)__builtin_popcount(ifm[(size_t)s * c->wps + w].x);
            }
          }
          c->d_ifm = dupload(ifm, ow);
        }
        c->d_act = dalloc<uint32_t>(2 * nss, ow);
        c->d_wake = dalloc<float>(nss, ow);
        c->d_wpush = dalloc<float>(2 * nss, ow);
        c->d_cnt = dalloc<uint32_t>(3 * kCntWords, ow);
        for (int k = 0; k < 3; ++k) {
          c->wl[k].bcnt = dalloc<uint32_t>(c->nsub, ow);
          c->wl[k].bins = dalloc<uint32_t>(nss, ow);
          c->wl[k].plan = dalloc<uint32_t>((size_t)c->nsub * c->maxch, ow);
          c->wl[k].cnt = c->d_cnt + kCntWords * k;
        }
        c->d_rscale = dalloc<float>(4 * (size_t)c->ninst, ow);
        c->d_tmpf = dalloc<float>(c->nn, ow);
        k_fill<float><<<blocks_for(4 * (size_t)c->ninst, 256), 256, 0, c->stream>>>(c->d_rscale, 4 * (size_t)c->ninst, 1.0f);
        c->h_rscale.assign(4 * (size_t)c->ninst, 1.0f);
        HIPCHECK(hipHostMalloc((void **)&c->h_par, 5 * (size_t)c->ninst * sizeof(float), hipHostMallocDefault));
        HIPCHECK(hipHostGetDevicePointer((void **)&c->d_par, c->h_par, 0));
        // one resident wave of workgroups: registers, LDS and wave slots.
        // Workgroups of 256 put one wave on each SIMD, so the LDS carve
        // alone caps the waves per SIMD at 160 KB / carve; the band kernel
        // variant sized for that many waves gets the registers left over.
        if (!few) {
          const uint32_t lds_cap = 160u * 1024u / std::max<uint32_t>(c->lds_conv, 1u);
          c->band_wpe = lds_cap <= 5u ? 5 : (lds_cap >= 8u ? 8 : (int)lds_cap);
          if (o->waves > 0) c->band_wpe = std::min(c->band_wpe, std::max(o->waves, 5));
        }
        auto size_grid = [&] {
          set_lds_attr(c);
          int per_cu = 0;
          HIPCHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, conv_kernel_ptr(c), c->block, c->lds_conv));
          c->grid = o->grid > 0 ? o->grid : ncu * std::max(per_cu, 1);
          c->grid = std::max(c->grid, (int)kXcd);  // every XCD eighth needs a workgroup
        };
        size_grid();
        // GATHER, where the submeshes on average, and a launch of all units, would
        // use it (its tests cost the others 1 %)
        const uint64_t per_wave = (uint64_t)c->ne / c->nsub / ((uint32_t)c->block / 64u);
        const bool fills = 2u * (uint64_t)c->nsub * c->maxch >= (uint64_t)c->grid;
        c->band_gather = c->band_pairs && !few && per_wave <= (fills ? kGatherFull : kGatherAlways);
        if (c->band_gather) size_grid();
        c->lds_compat = 0;
        c->ca = ConvArgs{c->d_sub, c->d_e2n, c->d_geo32, c->d_hgt, c->d_ereg, c->d_rscale, c->d_phi,
                         c->d_dirty, c->d_act, c->d_wake, c->d_wpush, c->d_if_l, c->d_ifm, c->d_inbox, c->d_if_fo,
                         c->d_if_os, WorkList{}, WorkList{}, c->d_stats, nullptr, c->d_start,
                         c->d_erec, c->d_adj, c->d_adj_ptr, c->d_adj_more,
                         c->nsub, c->ncopy, c->ninst, c->direct_plan ? 1u : 0u,
                         (float)(o->eps_rel > 0 ? o->eps_rel : 1e-6),
                         c->d_winst, o->local_iters, c->unit, c->maxch, (uint32_t)p.if_l.size(),
                         c->wps, lds.elcap, lds.o_phin, lds.o_flg, lds.o_tch, lds.o_dfr, lds.o_e2n, lds.o_geo,
                         lds.o_list, lds.o_vlist, lds.o_misc, lds.o_wrt, lds.o_ifc};
        c->n_if = (uint32_t)p.if_l.size();
      } else {
        const uint32_t nn = (uint32_t)c->nn_max;
        const uint32_t o_tphi = al16(8 * nn);
        const uint32_t o_st = o_tphi + al16(8 * nn);
        const uint32_t o_tst = o_st + al16(nn);
        const uint32_t o_snap = o_tst + al16(nn);
        const uint32_t o_misc = o_snap + al16(nn);
        c->lds_compat = o_misc + 16;
        if (c->lds_compat > 160 * 1024)
          throw Error(FIM_ELIMIT, "largest submesh too large for compat mode LDS");
        const uint32_t s_tmin = 2 * al16(8 * nn), s_st = s_tmin + al16(8 * nn);
        const uint32_t s_misc = s_st + al16(nn), s_blob = s_misc + al16(32 + 2 * 4 * ((uint32_t)c->block / 32));
        uint32_t chunks = 0, words = 0, gwords = 0;  // largest submesh
        uint64_t total = 0, gtotal = 0;              // all
        std::vector<CompatSub> cs(p.nsub);
        parallel_ranges((size_t)p.nsub, 512, [&](size_t b, size_t e) {
          for (size_t q = b; q < e; ++q) {
            const SubInfo &si = p.sub[q];
            uint32_t nch = 0;
            for (uint32_t l = 0; l < si.nn; ++l) nch += (p.n2e_dsp[si.coff + l + 1] - p.n2e_dsp[si.coff + l] + 3) / 4;
            const uint32_t w = (2 * (si.nn + 1) + 15) / 16 + (8 * si.ne + 15) / 16 + (8 * nch + 15) / 16;
            cs[q] = CompatSub{si.coff, si.nn, si.eoff, si.ne, si.ioff, 0u, w, nch};
          }
        });
        for (const CompatSub &q : cs) {
          chunks = std::max(chunks, q.nch);
          words = std::max(words, q.nw);
          gwords = std::max(gwords, q.nw + 3 * q.ne);
          total += q.nw;
          gtotal += q.nw + 3 * q.ne;
        }
        // k_compat_small needs a thread per copy and its data in LDS; 40 KB
        // leave a CU the four workgroups that its registers admit.  Without
        // the geometry in LDS (submeshes of 256 copies, say) it comes from L2.
        // A submesh's place in the blocks is a number of words in 32 bits.
        const uint32_t lists = 2 * al16(8 * chunks);
        constexpr uint32_t kSmallLds = 40 * 1024;
        c->compat_small = nn <= (uint32_t)c->block && (uint32_t)c->ne_max < (kNoSlot >> 2) && chunks < (1u << 16) &&
                          s_blob + 16 * words + lists <= kSmallLds && total < (1ull << 32);
        c->compat_geo = c->compat_small && s_blob + 16 * gwords + lists <= kSmallLds && gtotal < (1ull << 32);
        const uint32_t s_lp = s_blob + 16 * (c->compat_geo ? gwords : words), s_lq = s_lp + al16(8 * chunks);
        if (c->compat_small) {
          c->lds_compat = s_blob + 16 * (c->compat_geo ? gwords : words) + lists;
          total = 0;
          for (CompatSub &q : cs) {
            if (c->compat_geo) q.nw += 3 * q.ne;
            q.boff = (uint32_t)total;
            total += q.nw;
          }
          c->d_csub = dupload(cs, ow);
          c->d_blob = dalloc<uint4>(total, ow);
          const CompatBlockArgs ba{c->d_csub, c->d_e2n, dupload(p.n2e_dsp, tmp.v), dupload(p.n2e_le, tmp.v),
                                   dupload(p.n2e_pos, tmp.v),
                                   c->compat_geo ? reinterpret_cast<const uint4 *>(dupload(p.geo64, tmp.v)) : nullptr,
                                   c->d_blob, c->nsub};
          k_compat_block<<<(int)std::min<uint32_t>(c->nsub, 65536u), 256, 0, c->stream>>>(ba);
          HIPCHECK(hipGetLastError());
        }
        if (!c->compat_geo) c->d_geo64 = dupload(p.geo64, ow);
        if (!c->compat_small) {
          c->d_n2e_dsp = dupload(p.n2e_dsp, ow);
          c->d_n2e_le = dupload(p.n2e_le, ow);
          c->d_n2e_pos = dupload(p.n2e_pos, ow);
          c->d_n2n_dsp = dupload(p.n2n_dsp, ow);
          c->d_n2n_lv = dupload(p.n2n_lv, ow);
        }
        c->d_phi64 = dalloc<double>(c->ncopy, ow);
        c->d_st = dalloc<int8_t>(c->ncopy, ow);
        c->d_nexte = dalloc<double>(c->nsub, ow);
        c->d_list = dalloc<uint32_t>(2 * (size_t)c->nsub, ow);
        c->d_mark = dalloc<uint32_t>(c->nsub, ow);
        c->d_lcnt = dalloc<uint32_t>(3, ow);
        c->d_cshared = dalloc<uint32_t>(c->ncopy, ow);
        k_compat_shared<<<blocks_for(c->ncopy, 256), 256, 0, c->stream>>>(c->d_c2g, c->d_g2c_dsp, c->d_cshared, c->ncopy);
        HIPCHECK(hipGetLastError());
        c->d_vrec = dalloc<uint32_t>(p.if_l.size(), ow);
        c->d_vcnt = dalloc<uint32_t>(c->nsub, ow);
        c->d_done = dalloc<unsigned long long>(1, ow);
        HIPCHECK(hipFuncSetAttribute(compat_kernel_ptr(c), hipFuncAttributeMaxDynamicSharedMemorySize,
                                     (int)c->lds_compat));
        int ncu = 256, per_cu = 0;
        HIPCHECK(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, c->dev));
        HIPCHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, compat_kernel_ptr(c), c->block, c->lds_compat));
        c->grid = (int)std::min<uint32_t>(c->nsub, (uint32_t)(ncu * std::max(per_cu, 1)));
        c->lds_conv = 0;
        c->xa = CompatArgs{c->d_sub, c->d_e2n, c->d_geo64, c->d_n2e_dsp, c->d_n2e_le, c->d_n2e_pos,
                           c->d_n2n_dsp, c->d_n2n_lv, c->d_phi64, c->d_st,
                           c->d_nexte, nullptr, nullptr, c->d_cshared, c->d_vrec, c->d_vcnt,
                           c->d_done, c->d_pin, c->nsub,
                           o->local == FIM_LOCAL_EXACT ? 1 : 0, 0, 0, 0, 0, o->apd > 0 ? o->apd : 3e5,
                           o_tphi, c->compat_small ? s_st : o_st, o_tst, o_snap,
                           c->compat_small ? s_misc : o_misc, c->d_csub, c->d_blob, s_tmin, s_lp, s_lq, s_blob};
      }
      HIPCHECK(hipStreamSynchronize(c->stream));
      *out = c;
    } catch (...) {
      destroy_ctx(c);
      throw;
    }
    if (fim_reset(*out) != FIM_OK) {
      const std::string msg = fim_last_error();
      destroy_ctx(*out);
      *out = nullptr;
      throw Error(FIM_EDEVICE, msg);
    }
  });
}

int fim_reset(fim_ctx *c) {
  return guarded([&] {
    if (!c) throw Error(FIM_EINVAL, "null context");
    HIPCHECK(hipSetDevice(c->dev));
    FillArgs f;
    if (c->o.mode == FIM_MODE_CONVERGE) {
      const size_t ncs = (size_t)c->ninst * c->ncopy, nss = (size_t)c->ninst * c->nsub;
      settle(c);  // empties the inbox
      f.add(c->d_phi, ncs, F_INF);
      f.add(c->d_dirty, ncs, (uint8_t)0);
      f.add(c->d_act, 2 * nss, 0u);
      f.add(c->d_wake, nss, F_INF);
      f.add(c->d_wpush, 2 * nss, F_INF);
      f.add(c->d_cnt, 3 * kCntWords, 0u);
      f.add(c->d_start, c->ninst, 0u);
      c->next_iter = 0;
      for (int k = 0; k < 3; ++k) f.add(c->wl[k].bcnt, c->nsub, 0u);
    } else {
      f.add(c->d_phi64, c->ncopy, DBL_MAX);
      f.add(c->d_st, c->ncopy, (int8_t)FIM_FAR);
      f.add(c->d_nexte, c->nsub, (double)INFINITY);
      f.add(c->d_lcnt, 3, 0u);
      f.add(c->d_mark, c->nsub, 0u);
      f.add(c->d_done, 1, 0ull);
      c->stamp = 0u;
    }
    k_fill_all<<<blocks_for(f.seg[0].bytes / 16 + 1, 256), 256, 0, c->stream>>>(f);
    HIPCHECK(hipGetLastError());
    HIPCHECK(hipStreamSynchronize(c->stream));
  });
}

namespace {
// seeds (instance, copy) pairs at t0 through the context's staging buffers
// (grown, never shrunk); returns once the pinned buffer may be reused
void seed_pairs(fim_ctx *c, const std::vector<uint2> &ic, double t0) {
  if (ic.empty()) return;
  if (c->o.mode == FIM_MODE_CONVERGE && !(t0 >= 0.0)) throw Error(FIM_EINVAL, "converge mode needs t0 >= 0");
  if (ic.size() >= (1ull << 32)) throw Error(FIM_ELIMIT, "too many seed copies");
  HIPCHECK(hipSetDevice(c->dev));
  if (ic.size() > c->seed_cap) {
    HIPCHECK(hipStreamSynchronize(c->stream));
    if (c->h_seed) HIPCHECK(hipHostFree(c->h_seed));
    c->h_seed = nullptr;
    c->d_seed = nullptr;
    c->seed_cap = 0;
    const size_t cap = std::max<size_t>(ic.size(), 1024);
    HIPCHECK(hipHostMalloc((void **)&c->h_seed, cap * sizeof(uint2), hipHostMallocDefault));
    HIPCHECK(hipHostGetDevicePointer((void **)&c->d_seed, c->h_seed, 0));
    c->seed_cap = cap;
  }
  std::memcpy(c->h_seed, ic.data(), ic.size() * sizeof(uint2));
  const int g = blocks_for(ic.size(), 256);
  if (c->o.mode == FIM_MODE_CONVERGE) {
    k_conv_seed<<<g, 256, 0, c->stream>>>(c->d_seed, (uint32_t)ic.size(), (float)t0, c->d_c2s, c->d_phi,
                                          c->d_dirty, c->d_wake, list0(c), c->ncopy);
  } else {
    k_compat_seed<<<g, 256, 0, c->stream>>>(c->d_seed, (uint32_t)ic.size(), t0, c->d_c2s, c->d_phi64,
                                            c->d_st, c->d_nexte);
  }
  HIPCHECK(hipGetLastError());
  HIPCHECK(hipStreamSynchronize(c->stream));
}

void append_copies(const fim_ctx *c, int32_t inst, const int64_t *vtx, int64_t n, std::vector<uint2> &out) {
  for (uint32_t cp : copies_of(c, vtx, n)) out.push_back(make_uint2((uint32_t)inst, cp));
}
}  // namespace

int fim_seed(fim_ctx *c, int32_t inst, const int64_t *vtx, int64_t n, double t0) {
  return guarded([&] {
    if (!c || (!vtx && n > 0) || n < 0) throw Error(FIM_EINVAL, "bad seed arguments");
    check_inst(c, inst);
    std::vector<uint2> ic;
    append_copies(c, inst, vtx, n, ic);
    seed_pairs(c, ic, t0);
  });
}

int fim_seed_batch(fim_ctx *c, int32_t n_inst, const int32_t *inst, const int64_t *off,
                   const int64_t *vtx, double t0) {
  return guarded([&] {
    if (!c || n_inst < 0 || (n_inst > 0 && (!inst || !off))) throw Error(FIM_EINVAL, "bad seed arguments");
    if (n_inst == 0) return;
    if (off[0] != 0) throw Error(FIM_EINVAL, "off[0] must be 0");
    if (off[n_inst] > 0 && !vtx) throw Error(FIM_EINVAL, "bad seed arguments");
    std::vector<uint2> ic;
    for (int32_t i = 0; i < n_inst; ++i) {
      check_inst(c, inst[i]);
      if (off[i + 1] < off[i]) throw Error(FIM_EINVAL, "offsets must not decrease");
      append_copies(c, inst[i], vtx + off[i], off[i + 1] - off[i], ic);
    }
    seed_pairs(c, ic, t0);
  });
}

int fim_set_scaling(fim_ctx *c, int32_t inst, const float scale[4]) {
  return guarded([&] {
    if (!c || !scale) throw Error(FIM_EINVAL, "null argument");
    if (c->o.mode != FIM_MODE_CONVERGE) throw Error(FIM_ESTATE, "scaling needs converge mode");
    check_inst(c, inst);
    float m[4];
    for (int k = 0; k < 4; ++k) {
      if (!(scale[k] > 0.0f)) throw Error(FIM_EINVAL, "scalings must be positive");
      m[k] = 1.0f / (scale[k] * scale[k]);  // both speeds scaled: M scales by 1/s^2
    }
    std::memcpy(&c->h_rscale[4 * (size_t)inst], m, sizeof(m));
    c->params_dirty = true;
  });
}

int fim_set_window(fim_ctx *c, int32_t inst, double window) {
  return guarded([&] {
    if (!c) throw Error(FIM_EINVAL, "null context");
    if (c->o.mode != FIM_MODE_CONVERGE) throw Error(FIM_ESTATE, "time windows need converge mode");
    check_inst(c, inst);
    if (!(window >= 0.0) || !(window < 1e30)) throw Error(FIM_EINVAL, "window must be >= 0 and finite");
    c->h_winst[inst] = (float)window;
    c->params_dirty = true;
  });
}

int fim_init_field(fim_ctx *c, int32_t inst, const float *phi0) {
  return guarded([&] {
    if (!c || !phi0) throw Error(FIM_EINVAL, "null argument");
    if (c->o.mode != FIM_MODE_CONVERGE) throw Error(FIM_ESTATE, "warm start needs converge mode");
    check_inst(c, inst);
    for (uint32_t v = 0; v < c->nn; ++v)
      if (!(phi0[v] >= 0.0f)) throw Error(FIM_EINVAL, "initial field must be >= 0 (inf allowed)");
    HIPCHECK(hipSetDevice(c->dev));
    settle(c);
    HIPCHECK(hipMemcpyAsync(c->d_tmpf, phi0, c->nn * sizeof(float), hipMemcpyHostToDevice, c->stream));
    k_conv_init<<<blocks_for(c->ncopy, 256), 256, 0, c->stream>>>(c->d_tmpf, c->d_c2g, (uint32_t)inst,
                                                                   c->d_phi, c->d_dirty, c->ncopy, 1);
    k_conv_queue_all<<<blocks_for(c->nsub, 256), 256, 0, c->stream>>>((uint32_t)inst, c->d_wake, list0(c));
    HIPCHECK(hipGetLastError());
    HIPCHECK(hipStreamSynchronize(c->stream));
  });
}

int fim_step(fim_ctx *c, double phi_start, double cur_time, double dt, double front_width,
             int32_t *n_active) {
  return guarded([&] {
    if (!c) throw Error(FIM_EINVAL, "null context");
    if (c->o.mode != FIM_MODE_COMPAT) throw Error(FIM_ESTATE, "fim_step needs compat mode");
    HIPCHECK(hipSetDevice(c->dev));
    HIPCHECK(hipEventRecord(c->ev0, c->stream));
    if (++c->stamp == 0u) {  // after 2^32 - 1 windows the stamps start over
      k_fill<uint32_t><<<blocks_for(c->nsub, 256), 256, 0, c->stream>>>(c->d_mark, c->nsub, 0u);
      c->stamp = 1u;
    }
    const uint32_t turn = c->turn = (c->turn + 1u) % 6u;
    uint32_t *list = c->d_list + (turn & 1u) * (size_t)c->nsub, *last = c->d_list + ((turn & 1u) ^ 1u) * (size_t)c->nsub;
    const CompatSyncArgs sy{c->d_sub, last, c->d_lcnt + (turn + 2) % 3, c->d_vrec, c->d_vcnt, c->d_g2c_dsp, c->d_g2c,
                            c->d_c2s, c->d_phi64, c->d_st, c->d_nexte, c->nsub, cur_time, list,
                            c->d_lcnt + turn % 3, c->d_lcnt + (turn + 1) % 3, c->d_mark, c->stamp};
    // a wave for every submesh the last window can have listed, up to 8 waves per SIMD
    k_compat_sync<<<std::min<int>(blocks_for((size_t)c->nsub * 64, 256), 2048), 256, 0, c->stream>>>(sy);
    HIPCHECK(hipGetLastError());
    CompatArgs a = c->xa;
    a.list = list;
    a.nlist = c->d_lcnt + turn % 3;
    a.fw = front_width;
    a.cur = cur_time;
    a.phi_start = phi_start;
    a.dt = dt;
    launch_compat_compute(c, a);
    HIPCHECK(hipEventRecord(c->ev1, c->stream));
    HIPCHECK(hipStreamSynchronize(c->stream));
    float ms = 0;
    HIPCHECK(hipEventElapsedTime(&ms, c->ev0, c->ev1));
    c->stats.last_ms = ms;
    if (n_active) *n_active = (int32_t)c->h_pin[0];
  });
}

namespace {
// The loop of global iterations in phases -- begin, a chunk of graph_iters
// iterations with the read-back of the queued units, collect, end -- so that
// one host thread can also drive several contexts at once (fim_run_multi),
// whose streams then overlap on the device.  Device counters accumulate from
// the last begin with reset_stats.
struct RunState {
  int32_t max_iters = 0, done = 0;
  uint32_t left = 1;
  double kms = 0.0;
  int64_t klaunch = 0;
};

void run_begin(fim_ctx *c, int32_t max_iters, bool reset_stats, RunState &r) {
  HIPCHECK(hipSetDevice(c->dev));
  flush_params(c, reset_stats);
  // profile mode launches the same sequence of kernels without the graph
  // (events cannot be timed inside a graph) and times every compute launch
  if (c->o.profile && c->kev.empty()) {
    c->kev.assign(2 * c->graph_iters, nullptr);
    for (auto &e : c->kev) HIPCHECK(hipEventCreate(&e));
  }
  if (!c->o.profile && !c->direct && !c->gexec) build_graph(c);
  if (reset_stats) {
    c->stats.compute_ms = 0.0;
    c->stats.compute_launches = 0;
  }
  c->inbox_left = true;  // until the run has ended with nothing queued
  HIPCHECK(hipEventRecord(c->ev0, c->stream));
  // units of the list the seeds (or an earlier run) filled
  if (!c->direct_plan) launch_plan(c, 0, -1);
  r = RunState{};
  r.max_iters = max_iters;
}

// enqueues graph_iters iterations, the read-back of the queued units and the
// chunk's completion event
void run_chunk(fim_ctx *c, RunState &r) {
  HIPCHECK(hipSetDevice(c->dev));
  if (c->next_iter + (uint32_t)c->graph_iters > kIterEnd) renumber(c, 0u);
  c->next_iter += (uint32_t)c->graph_iters;
  if (c->o.profile || c->direct) {
    for (int i = 0; i < c->graph_iters; ++i) enqueue_iteration(c, i, c->o.profile != 0);
  } else {
    HIPCHECK(hipGraphLaunch(c->gexec, c->stream));
  }
  r.done += c->graph_iters;
  k_chunk_end<<<1, 64, 0, c->stream>>>(c->d_cnt, reinterpret_cast<const uint32_t *>(c->d_stats), c->d_pin);
  HIPCHECK(hipGetLastError());
  HIPCHECK(hipEventRecord(c->evc, c->stream));
}

// after the chunk's event has completed: launch times (profile mode) and
// queued units; true while more iterations are to run
bool run_collect(fim_ctx *c, RunState &r) {
  if (c->o.profile) {
    for (int j = 0; j < c->graph_iters; ++j) {
      float ms = 0;
      HIPCHECK(hipEventElapsedTime(&ms, c->kev[2 * j], c->kev[2 * j + 1]));
      r.kms += ms;
      ++r.klaunch;
    }
  }
  r.left = c->h_pin[0];
  return r.left != 0 && r.done < r.max_iters;
}

void run_end(fim_ctx *c, RunState &r) {
  unsigned long long st[8];  // of the last chunk, whose event has completed
  std::memcpy(st, c->h_pin + 2, sizeof(st));
  float ms = 0;
  HIPCHECK(hipSetDevice(c->dev));
  HIPCHECK(hipEventElapsedTime(&ms, c->ev0, c->evc));
  c->stats.last_ms = ms;
  c->stats.activations = (int64_t)st[0];
  c->stats.local_iters = (int64_t)st[1];
  c->stats.elem_updates = (int64_t)st[2];
  c->stats.global_iters = (int64_t)st[3];
  c->stats.alg_bytes = (int64_t)st[4];
  c->stats.vertex_updates = (int64_t)st[5];
  c->inbox_left = r.left != 0;
  c->stats.compute_ms += r.kms;
  c->stats.compute_launches += r.klaunch;
}

// Runs global iterations in graph-sized chunks until no work is queued or
// max_iters (rounded up to whole chunks) have run; returns the queued units
// left (0 = every instance converged).
uint32_t run_iterations(fim_ctx *c, int32_t max_iters, bool reset_stats) {
  RunState r;
  run_begin(c, max_iters, reset_stats, r);
  do {
    run_chunk(c, r);
    HIPCHECK(hipEventSynchronize(c->evc));
  } while (run_collect(c, r));
  run_end(c, r);
  return r.left;
}

std::vector<uint32_t> checked_instances(const fim_ctx *c, int32_t n, const int32_t *insts) {
  if (n < 0 || (n > 0 && !insts)) throw Error(FIM_EINVAL, "bad instance list");
  std::vector<uint32_t> v(n);
  for (int32_t i = 0; i < n; ++i) {
    check_inst(c, insts[i]);
    v[i] = (uint32_t)insts[i];
  }
  return v;
}
}  // namespace

int fim_run(fim_ctx *c, int32_t max_iters, int32_t *iters) {
  return guarded([&] {
    if (!c) throw Error(FIM_EINVAL, "null context");
    if (c->o.mode != FIM_MODE_CONVERGE) throw Error(FIM_ESTATE, "fim_run needs converge mode");
    if (max_iters <= 0) throw Error(FIM_EINVAL, "max_iters must be positive");
    const uint32_t left = run_iterations(c, max_iters, true);
    if (iters) *iters = (int32_t)c->stats.global_iters;
    if (left != 0) throw Error(FIM_ENOCONV, "iteration cap reached before convergence");
  });
}

int fim_advance(fim_ctx *c, int32_t iters, int32_t reset_stats, int32_t *left) {
  return guarded([&] {
    if (!c) throw Error(FIM_EINVAL, "null context");
    if (c->o.mode != FIM_MODE_CONVERGE) throw Error(FIM_ESTATE, "fim_advance needs converge mode");
    if (iters <= 0) throw Error(FIM_EINVAL, "iters must be positive");
    const uint32_t l = run_iterations(c, iters, reset_stats != 0);
    if (left) *left = (int32_t)l;
  });
}

int fim_run_multi(fim_ctx *const *cs, int32_t n, int32_t max_iters, int32_t *iters) {
  return guarded([&] {
    if (!cs || n <= 0) throw Error(FIM_EINVAL, "bad context list");
    if (max_iters <= 0) throw Error(FIM_EINVAL, "max_iters must be positive");
    for (int32_t i = 0; i < n; ++i) {
      if (!cs[i]) throw Error(FIM_EINVAL, "null context");
      if (cs[i]->o.mode != FIM_MODE_CONVERGE) throw Error(FIM_ESTATE, "fim_run_multi needs converge mode");
      for (int32_t j = 0; j < i; ++j)
        if (cs[j] == cs[i]) throw Error(FIM_EINVAL, "context listed twice");
    }
    std::vector<RunState> rs(n);
    std::vector<uint8_t> running(n, 1);
    for (int32_t i = 0; i < n; ++i) {
      run_begin(cs[i], max_iters, true, rs[i]);
      run_chunk(cs[i], rs[i]);
    }
    // the host polls the chunks' events and keeps every stream fed; the
    // streams' kernels share the device, so one context's launch tail is
    // filled by another's work
    for (int32_t active = n; active > 0;) {
      bool progress = false;
      for (int32_t i = 0; i < n; ++i) {
        if (!running[i]) continue;
        HIPCHECK(hipSetDevice(cs[i]->dev));
        const hipError_t q = hipEventQuery(cs[i]->evc);
        if (q == hipErrorNotReady) continue;
        HIPCHECK(q);
        progress = true;
        if (run_collect(cs[i], rs[i])) {
          run_chunk(cs[i], rs[i]);
        } else {
          run_end(cs[i], rs[i]);
          running[i] = 0;
          --active;
        }
      }
      if (!progress) std::this_thread::yield();
    }
    bool capped = false;
    for (int32_t i = 0; i < n; ++i) {
      if (iters) iters[i] = (int32_t)cs[i]->stats.global_iters;
      capped = capped || rs[i].left != 0;
    }
    if (capped) throw Error(FIM_ENOCONV, "iteration cap reached before convergence");
  });
}

int fim_ctx_renumber(fim_ctx *c, uint32_t n) {
  return guarded([&] {
    if (!c || (c->o.mode == FIM_MODE_CONVERGE && n >= kIterEnd)) throw Error(FIM_EINVAL, "bad renumbering");
    HIPCHECK(hipSetDevice(c->dev));
    if (c->o.mode == FIM_MODE_CONVERGE) renumber(c, n);
    else c->stamp = n - 1u;
    HIPCHECK(hipStreamSynchronize(c->stream));
  });
}

int fim_active(fim_ctx *c, int32_t *active) {
  return guarded([&] {
    if (!c || !active) throw Error(FIM_EINVAL, "null argument");
    if (c->o.mode != FIM_MODE_CONVERGE) throw Error(FIM_ESTATE, "fim_active needs converge mode");
    HIPCHECK(hipSetDevice(c->dev));
    k_inst_active<<<c->ninst, 256, 0, c->stream>>>(list0(c), c->d_flag);
    HIPCHECK(hipGetLastError());
    std::vector<uint32_t> h(c->ninst);
    HIPCHECK(hipMemcpyAsync(h.data(), c->d_flag, sizeof(uint32_t) * c->ninst, hipMemcpyDeviceToHost, c->stream));
    HIPCHECK(hipStreamSynchronize(c->stream));
    for (uint32_t i = 0; i < c->ninst; ++i) active[i] = (int32_t)h[i];
  });
}

int fim_recycle(fim_ctx *c, int32_t n, const int32_t *insts) {
  return guarded([&] {
    if (!c) throw Error(FIM_EINVAL, "null context");
    if (c->o.mode != FIM_MODE_CONVERGE) throw Error(FIM_ESTATE, "fim_recycle needs converge mode");
    const std::vector<uint32_t> v = checked_instances(c, n, insts);
    if (v.empty()) return;
    HIPCHECK(hipSetDevice(c->dev));
    // only instances with nothing queued may be recycled
    k_inst_active<<<c->ninst, 256, 0, c->stream>>>(list0(c), c->d_flag);
    HIPCHECK(hipGetLastError());
    std::vector<uint32_t> h(c->ninst);
    HIPCHECK(hipMemcpyAsync(h.data(), c->d_flag, sizeof(uint32_t) * c->ninst, hipMemcpyDeviceToHost, c->stream));
    HIPCHECK(hipStreamSynchronize(c->stream));
    std::vector<uint8_t> seen(c->ninst, 0);
    for (uint32_t i : v) {
      if (h[i]) throw Error(FIM_ESTATE, "instance " + std::to_string(i) + " still has queued work");
      if (seen[i]++) throw Error(FIM_EINVAL, "instance listed twice");
    }
    HIPCHECK(hipMemcpyAsync(c->d_flag, v.data(), sizeof(uint32_t) * v.size(), hipMemcpyHostToDevice, c->stream));
    const size_t total = ((size_t)c->ncopy + c->nsub) * v.size();
    k_inst_reset<<<blocks_for(total, 256), 256, 0, c->stream>>>(c->d_flag, (uint32_t)v.size(), c->d_phi, c->d_dirty,
                                                               c->d_wake, c->d_start, c->wl[0].cnt + kIterWord, c->ncopy,
                                                               c->nsub);
    HIPCHECK(hipGetLastError());
    HIPCHECK(hipStreamSynchronize(c->stream));
  });
}

int fim_download(fim_ctx *c, int32_t inst, double *phi, int32_t *state) {
  return guarded([&] {
    if (!c) throw Error(FIM_EINVAL, "null context");
    check_inst(c, inst);
    HIPCHECK(hipSetDevice(c->dev));
    // The gather kernel writes pinned host memory itself (no copy after it,
    // no array of the call's own to fault in), and the loops below vectorise:
    // 362,894 vertices in 166 us, 40 of them until the map is on the host,
    // against 272 and 114 with a pageable copy and one branching loop; 9,261
    // vertices in 20 against 34 us.  Four threads take 110, but the caller's
    // next pass over the map then finds it in their caches (34 us more).
    const int g = blocks_for(c->nn, 256);
    if (c->o.mode == FIM_MODE_CONVERGE) {
      k_conv_gather<<<g, 256, 0, c->stream>>>(c->d_phi, c->d_g2c_dsp, c->d_g2c, c->nn, (size_t)inst * c->ncopy,
                                              reinterpret_cast<float *>(c->d_map));
      HIPCHECK(hipGetLastError());
      HIPCHECK(hipStreamSynchronize(c->stream));
      // times are >= 0, so their bits compare as they do.  (Compared as floats,
      // the loop of the states took 21 or 37 us of a call, by where the linker
      // happened to put it.)
      const float *h = reinterpret_cast<const float *>(c->h_map);
      const int32_t *bits = reinterpret_cast<const int32_t *>(c->h_map);
      for (uint32_t v0 = 0; v0 < c->nn; v0 += 4096) {
        const uint32_t v1 = std::min(c->nn, v0 + 4096);
        if (phi)
          for (uint32_t v = v0; v < v1; ++v) phi[v] = h[v] < F_INF ? (double)h[v] : DBL_MAX;
        if (state)
          for (uint32_t v = v0; v < v1; ++v) state[v] = bits[v] < 0x7f800000 ? FIM_FROZEN : FIM_FAR;
      }
    } else {
      const size_t nb = c->nn * sizeof(double);
      k_compat_gather<<<g, 256, 0, c->stream>>>(c->d_phi64, c->d_st, c->d_g2c_dsp, c->d_g2c, c->nn,
                                                reinterpret_cast<double *>(c->d_map),
                                                reinterpret_cast<int32_t *>(c->d_map + nb));
      HIPCHECK(hipGetLastError());
      HIPCHECK(hipStreamSynchronize(c->stream));
      if (phi) std::memcpy(phi, c->h_map, nb);
      if (state) std::memcpy(state, c->h_map + nb, c->nn * sizeof(int32_t));
    }
  });
}

int fim_residual(fim_ctx *c, int32_t inst, double *res) {
  return guarded([&] {
    if (!c || !res) throw Error(FIM_EINVAL, "null argument");
    if (c->o.mode != FIM_MODE_CONVERGE) throw Error(FIM_ESTATE, "residual needs converge mode");
    check_inst(c, inst);
    HIPCHECK(hipSetDevice(c->dev));
    flush_params(c);
    settle(c);
    k_fill<uint32_t><<<1, 64, 0, c->stream>>>(c->d_tmpu, 1, 0u);
    k_conv_residual<<<(int)std::min<uint32_t>(c->nsub, 4096u), 256, 0, c->stream>>>(
        c->d_sub, c->nsub, c->d_e2n, c->d_geo32, c->d_ereg, c->d_rscale, c->d_phi,
        (size_t)inst * c->ncopy, (uint32_t)inst, c->d_tmpu);
    HIPCHECK(hipGetLastError());
    uint32_t bits = 0;
    HIPCHECK(hipMemcpyAsync(&bits, c->d_tmpu, 4, hipMemcpyDeviceToHost, c->stream));
    HIPCHECK(hipStreamSynchronize(c->stream));
    float r;
    std::memcpy(&r, &bits, 4);
    *res = r;
  });
}

int fim_support(fim_ctx *c, int32_t inst, double *worst) {
  return guarded([&] {
    if (!c || !worst) throw Error(FIM_EINVAL, "null argument");
    if (c->o.mode != FIM_MODE_CONVERGE) throw Error(FIM_ESTATE, "support check needs converge mode");
    check_inst(c, inst);
    HIPCHECK(hipSetDevice(c->dev));
    uint32_t *best = nullptr;
    HIPCHECK(hipMalloc(&best, (size_t)c->nn * sizeof(uint32_t)));
    try {
      *worst = support_into(c, inst, best);
    } catch (...) {
      (void)hipFree(best);
      throw;
    }
    HIPCHECK(hipFree(best));
  });
}

int fim_support_noalloc(fim_ctx *c, int32_t inst, double *worst) {
  return guarded([&] {
    if (!c || !worst) throw Error(FIM_EINVAL, "null argument");
    if (c->o.mode != FIM_MODE_CONVERGE) throw Error(FIM_ESTATE, "support check needs converge mode");
    check_inst(c, inst);
    if (c->nn > kNoAllocMaxVertices)
      throw Error(FIM_ELIMIT, "fim_support_noalloc: " + std::to_string(c->nn) +
                                  " vertices exceed its scratch of " + std::to_string(kNoAllocMaxVertices) +
                                  " (use fim_support)");
    HIPCHECK(hipSetDevice(c->dev));
    *worst = support_into(c, inst, noalloc_scratch(c->dev));
  });
}

int fim_stats(const fim_ctx *c, fim_stats_t *s) {
  return guarded([&] {
    if (!c || !s) throw Error(FIM_EINVAL, "null argument");
    *s = c->stats;
  });
}

void fim_destroy(fim_ctx *c) {
  if (c) (void)hipSetDevice(c->dev);
  destroy_ctx(c);
}

int fim_device_info(int32_t device, char *buf, int64_t len) {
  return guarded([&] {
    if (!buf || len <= 0) throw Error(FIM_EINVAL, "null buffer");
    int n = 0;
    HIPCHECK(hipGetDeviceCount(&n));
    if (device < 0 || device >= n) throw Error(FIM_EINVAL, "no such device");
    hipDeviceProp_t p;
    HIPCHECK(hipGetDeviceProperties(&p, device));
    std::snprintf(buf, (size_t)len,
                  "device %d: %s (%s), %d CUs, %.1f GiB, LDS/block %zu B, wavefront %d, clock %d kHz, "
                  "devices visible %d",
                  device, p.name, p.gcnArchName, p.multiProcessorCount,
                  (double)p.totalGlobalMem / (1024.0 * 1024.0 * 1024.0), (size_t)p.sharedMemPerBlock,
                  p.warpSize, p.clockRate, n);
  });
}

}  // extern "C"
