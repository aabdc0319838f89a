// grd_ops.hpp -- operator policies of the BSP traversal and their combine
// rules (shared by the push, pull and exchange kernels).
#pragma once

#include <type_traits>

#include "grd_device.hpp"
#include "grd_internal.hpp"

namespace grd {

// CC: label propagation, atomicMin (cc.cpp:65-78, DistributedGraph.hpp:103-112)
struct OpCC {
  using V = uint32_t;
  static constexpr bool kMin = true;
  __device__ static V edge(V v, uint32_t) { return v; }
};
// SSSP hop count: dist + 1 (sssp.cpp:69); the unreached value stays unreached
struct OpHop {
  using V = uint32_t;
  static constexpr bool kMin = true;
  __device__ static V edge(V v, uint32_t) { return v == 0xFFFFFFFFu ? v : v + 1u; }
};
// SSSP weighted (extension): saturating dist + w (the unreached value stays
// unreached)
struct OpWeighted {
  using V = uint32_t;
  static constexpr bool kMin = true;
  __device__ static V edge(V v, uint32_t w)
  {
    uint32_t t = v + w;
    return t < v ? 0xFFFFFFFFu : t;
  }
};
// Reference PageRank: push the vertex property, atomicAdd (pr.cpp:95-120)
struct OpPR {
  using V = float;
  static constexpr bool kMin = false;
  __device__ static V edge(V v, uint32_t) { return v; }
};

template <class Op>
__device__ __forceinline__ typename Op::V op_identity()
{
  if constexpr (Op::kMin) return 0xFFFFFFFFu;
  else return 0.0f;
}

template <class Op>
__device__ __forceinline__ typename Op::V op_combine(typename Op::V a, typename Op::V b)
{
  if constexpr (Op::kMin) return a < b ? a : b;
  else return a + b;
}

// A value that a pass only lowers, or a word in which it only sets bits, as the
// compute unit last saw it (an L1 hit serves): an old one costs an atomic that
// changes nothing, never a missed one.  With system-scope loads every look at a
// dirty word or a current value went to the L2: the heavy pass of a delta-push
// PageRank superstep over RMAT-18 157 us, now 108.
template <typename T>
__device__ __forceinline__ T peek(const T *p)
{
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

__device__ __forceinline__ void set_bit(uint64_t *bits, uint32_t i)
{
  uint64_t b = 1ull << (i & 63);
  uint64_t *wd = bits + (i >> 6);
  if (!(peek(wd) & b)) atomicOr((unsigned long long *)wd, (unsigned long long)b);
}

// minUpdate / addUpdate, marking the dirty bit (DistributedGraph.hpp:103-130).
// minUpdate marks only on improvement.  addUpdate always marks: on the
// memory side a proxy's update is zero until its first add of the iteration
// (the previous reduce cleared it), so the first add (old == 0) marks; on the
// compute side residuals below the threshold persist, so every add marks.
template <class Op, bool kAlwaysMark = false>
__device__ __forceinline__ void relax(typename Op::V *upd, uint64_t *dirty, uint32_t dst, typename Op::V cand)
{
  if constexpr (Op::kMin) {
    uint32_t cur = peek(upd + dst);
    if (cand < cur) {
      uint32_t old = atomicMin(upd + dst, cand);
      if (cand < old) set_bit(dirty, dst);
    }
  } else {
    float old = atomicAdd(upd + dst, cand);
    if (kAlwaysMark || old == 0.0f) set_bit(dirty, dst);
  }
}

// The arcs of a wave (on: the lanes that have one) that all meet at one vertex
// become one arc of its first lane.  Called by the whole wave.
//
// Atomics on one word come one after another, some 4 ns each, and while a
// compute unit keeps an old value of the word (peek) every wave on it tries.  By
// pushes on a star of 2^20 vertices, from its hub: hop SSSP 1.72 ms a solve, now
// 0.40 (1.10 when every look at a value went to the L2); ten supersteps of delta
// PageRank 53 ms, now 2.4.  Where no wave's arcs meet the test is within the
// noise (weighted SSSP over RMAT-22 18.0 / 17.7 ms).  Fewer than kMeet lanes are
// left alone.
constexpr int kMeet = 8;
template <class Op>
__device__ __forceinline__ void wave_meet(bool &on, uint32_t dst, typename Op::V &cand)
{
  using V = typename Op::V;
  const uint64_t m = __ballot(on);
  if (__popcll(m) < kMeet) return;
  const int lead = __ffsll((unsigned long long)m) - 1;
  if (__ballot(on && dst != (uint32_t)__builtin_amdgcn_readlane((int)dst, lead))) return;
  V v = on ? cand : op_identity<Op>();
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) v = op_combine<Op>(v, __shfl_xor(v, o, kWave));
  cand = v;
  on = lane_id() == (uint32_t)lead;
}

// relax for the first cnt of N destinations of one thread: the current values
// are all loaded before any is compared, and the atomics are all issued before
// any dirty mark waits for one.  Called by the whole wave.
template <class Op, int N, bool kAlwaysMark>
__device__ __forceinline__ void relax_many(typename Op::V *upd, uint64_t *dirty, const uint32_t (&dst)[N],
                                           typename Op::V (&cand)[N], uint32_t cnt)
{
  bool on[N], mark[N];
#pragma unroll
  for (int q = 0; q < N; q++) on[q] = (uint32_t)q < cnt;
  if constexpr (Op::kMin) {
    uint32_t cur[N], old[N];
#pragma unroll
    for (int q = 0; q < N; q++) cur[q] = on[q] ? peek(upd + dst[q]) : 0u;
#pragma unroll
    for (int q = 0; q < N; q++) {
      on[q] = cand[q] < cur[q];
      wave_meet<Op>(on[q], dst[q], cand[q]);
      old[q] = on[q] ? atomicMin(upd + dst[q], cand[q]) : 0u;
    }
#pragma unroll
    for (int q = 0; q < N; q++) mark[q] = on[q] && cand[q] < old[q];
  } else if constexpr (kAlwaysMark) {
#pragma unroll
    for (int q = 0; q < N; q++) {
      wave_meet<Op>(on[q], dst[q], cand[q]);
      if (on[q]) atomicAdd(upd + dst[q], cand[q]);
      mark[q] = on[q];
    }
  } else {
    float old[N];
#pragma unroll
    for (int q = 0; q < N; q++) {
      wave_meet<Op>(on[q], dst[q], cand[q]);
      old[q] = on[q] ? atomicAdd(upd + dst[q], cand[q]) : 1.0f;
    }
#pragma unroll
    for (int q = 0; q < N; q++) mark[q] = on[q] && old[q] == 0.0f;
  }
#pragma unroll
  for (int q = 0; q < N; q++)
    if (mark[q]) set_bit(dirty, dst[q]);
}

// Sets bit i for every lane with pred.  Called by the whole wave: when all
// marked bits fall into one 64-bit word (a wave over a word of own proxies
// maps onto one word of slots) they are OR-ed across the wave and written by
// one atomic instead of up to 64 atomics on the same word.
__device__ __forceinline__ void mark_wave(uint64_t *bits, uint32_t i, bool pred)
{
  const uint64_t m = __ballot(pred);
  if (m == 0) return;
  const int leader = __ffsll((unsigned long long)m) - 1;
  const uint32_t wl = __shfl(i >> 6, leader, kWave);
  const bool same = !pred || (i >> 6) == wl;
  if (__ballot(pred && i != wl * 64 + lane_id()) == 0) {  // every lane's bit is its own: the ballot is the word
    if (lane_id() == leader) atomicOr((unsigned long long *)(bits + wl), (unsigned long long)m);
  } else if (__ballot(!same) == 0) {
    uint32_t lo = 0, hi = 0;
    if (pred) {
      if ((i & 63) < 32) lo = 1u << (i & 31);
      else hi = 1u << (i & 31);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      lo |= __shfl_xor(lo, o, kWave);
      hi |= __shfl_xor(hi, o, kWave);
    }
    if (lane_id() == leader) atomicOr((unsigned long long *)(bits + wl), ((unsigned long long)hi << 32) | lo);
  } else if (pred) {
    set_bit(bits, i);
  }
}

// How the pull's row passes accumulate (the hot pass of tiers.hip, the cold
// pass of cold.hip).  Pull PageRank: FP32 Kahan per lane, lanes
// merged by TwoSum, the compensated sum of each row rounded once to FP32.  The BSP pull (CC,
// SSSP, reference PageRank): Op::edge of the source's broadcast value and the
// arc weight, combined with the operator (min, or + in a fixed order).
// The hot part of a row is a few arcs on average (2.7 at RMAT-26, M = 4), so
// its compensated sum is kept as one FP32 value (the sum rounded once): the
// per-row partial is 4 bytes written and read instead of 8.
struct HotPR {
  using V = float;
  using Part = float;
  using Acc = Kahan;
  static constexpr bool kWeighted = false;
  __device__ static Acc zero() { return Kahan{}; }
  __device__ static V value(V v, uint32_t) { return v; }
  __device__ static void add(Acc &a, V x) { a.add(x); }
  __device__ static void merge_lanes(Acc &a, int width) { kahan_wave_merge(a, width); }
  __device__ static void merge(Acc &a, const Acc &o) { a.merge(o.s, o.c); }
  __device__ static void add_part(Acc &a, Part p) { a.merge(p, 0.0f); }
  __device__ static Part part(const Acc &a) { return a.value(); }
};
template <class Op>
struct HotBsp {
  using V = typename Op::V;
  using Part = V;
  using Acc = V;
  static constexpr bool kWeighted = std::is_same<Op, OpWeighted>::value;
  __device__ static Acc zero() { return op_identity<Op>(); }
  __device__ static V value(V v, uint32_t w) { return Op::edge(v, w); }
  __device__ static void add(Acc &a, V x) { a = op_combine<Op>(a, x); }
  __device__ static void merge_lanes(Acc &a, int width)
  {
    for (int o = width / 2; o > 0; o >>= 1) a = op_combine<Op>(a, __shfl_xor(a, o, kWave));
  }
  __device__ static void merge(Acc &a, const Acc &o) { a = op_combine<Op>(a, o); }
  __device__ static void add_part(Acc &a, Part p) { a = op_combine<Op>(a, p); }
  __device__ static Part part(const Acc &a) { return a; }
};

// apply the pulled value to the proxy's running update; true = dirty
template <class Op>
__device__ __forceinline__ bool pull_apply(typename Op::V *upd, uint32_t r, typename Op::V acc)
{
  if constexpr (Op::kMin) {
    if (acc < upd[r]) {
      upd[r] = acc;
      return true;
    }
    return false;
  } else {
    // contributions of active sources are strictly positive (pr.cpp:80)
    if (acc > 0.0f) {
      upd[r] = upd[r] + acc;
      return true;
    }
    return false;
  }
}

// the smallest candidate a pull superstep can produce: the smallest value
// broadcast plus the smallest Op::edge increment, saturating
__device__ __forceinline__ uint32_t pull_bound(const Counters *cnt, uint32_t inc)
{
  const uint32_t f = cnt->fmin;
  return f + inc < f ? 0xFFFFFFFFu : f + inc;
}

// Publishing the counters (k_publish of bsp.hip, k_mlp_publish of mlp.hip): a
// workgroup of kBlock threads.
struct Shares {
  const BlockShare *u;
  uint32_t nu;
  uint32_t *r;
  uint32_t nr;
  const SkipShare *s;
  uint32_t ns;
};

Shares shares(const grd_state *s);
uint32_t loop_blocks(const grd_ctx *ctx);  // most workgroups of a pass that leaves shares

// the counters of one superstep to their start (not the pull PageRank's
// residual and dangling mass)
__device__ __forceinline__ void zero_counters(Counters *cnt, const Shares &sh)
{
  if (threadIdx.x == 0) {
    cnt->pending = 0;
    cnt->heavy = 0;
    cnt->pend_min = 0xFFFFFFFFu;
    cnt->fmin = 0xFFFFFFFFu;
    cnt->pull_done_arcs = 0;
    cnt->frontier_uncovered = 0;
  }
  for (uint32_t c = threadIdx.x; c < (uint32_t)kMaxParts; c += kBlock) cnt->fpart[c] = 0;
  for (uint32_t b = threadIdx.x; b < sh.nr; b += kBlock) sh.r[b] = 0;
}

// a workgroup's share of what a pull leaves out
__device__ __forceinline__ void add_share(SkipShare *p, SkipShare x, bool again)
{
  if (again) {
    x.arcs += p->arcs;
    x.hot_arcs += p->hot_arcs;
    x.rows += p->rows;
  }
  *p = x;
}

// the sums of the blocks' shares, in every thread
struct FrontierCounts {
  unsigned long long frontier, edges, dirty, skipped, skipped_hot, skipped_rows;
  uint32_t maxdeg;
};
__device__ __forceinline__ FrontierCounts sum_shares(const Shares &sh)
{
  __shared__ unsigned long long s_c[kWavesPerBlock][5];
  __shared__ uint32_t s_m[kWavesPerBlock];
  unsigned long long c[5] = {0, 0, 0, 0, 0};
  uint32_t m = 0;
#pragma unroll 8
  for (uint32_t b = threadIdx.x; b < sh.nu; b += kBlock) {
    c[0] += sh.u[b].front;
    m = max(m, sh.u[b].maxdeg);
  }
#pragma unroll 8
  for (uint32_t b = threadIdx.x; b < sh.nr; b += kBlock) c[1] += sh.r[b];
#pragma unroll 4
  for (uint32_t b = threadIdx.x; b < sh.ns; b += kBlock) {
    c[2] += sh.s[b].arcs;
    c[3] += sh.s[b].hot_arcs;
    c[4] += sh.s[b].rows;
  }
#pragma unroll
  for (int q = 0; q < 5; q++) c[q] = wave_sum(c[q]);
  m = wave_max(m);
  if (lane_id() == 0) {
#pragma unroll
    for (int q = 0; q < 5; q++) s_c[wave_in_block()][q] = c[q];
    s_m[wave_in_block()] = m;
  }
  __syncthreads();
  m = 0;
#pragma unroll
  for (int q = 0; q < 5; q++) c[q] = 0;
#pragma unroll
  for (int i = 0; i < kWavesPerBlock; i++) {
#pragma unroll
    for (int q = 0; q < 5; q++) c[q] += s_c[i][q];
    m = max(m, s_m[i]);
  }
  return FrontierCounts{c[0] >> 32, c[0] & 0xFFFFFFFFull, c[1], c[2], c[3], c[4], m};
}

// the counters into the host's copy, except the words [skip0, skip1): by the
// first wave, words i and i + 64 by lane i, loaded (counter_words) before the
// shares are waited for
struct CounterWords {
  uint64_t w[2];
};
__device__ __forceinline__ CounterWords counter_words(const Counters *cnt)
{
  static_assert(sizeof(Counters) % 8 == 0 && sizeof(Counters) / 8 <= 2 * kWave, "two words per lane of a wave");
  CounterWords c{{0, 0}};
#pragma unroll
  for (uint32_t q = 0; q < 2; q++) {
    const uint32_t i = threadIdx.x + q * kWave;
    if (threadIdx.x < (uint32_t)kWave && i < sizeof(Counters) / 8) c.w[q] = reinterpret_cast<const uint64_t *>(cnt)[i];
  }
  return c;
}
__device__ __forceinline__ void copy_counters(const CounterWords &c, Counters *host, const FrontierCounts &fc,
                                              uint32_t skip0 = 0, uint32_t skip1 = 0)
{
#pragma unroll
  for (uint32_t q = 0; q < 2; q++) {
    const uint32_t i = threadIdx.x + q * kWave;
    if (threadIdx.x < (uint32_t)kWave && i >= kHostOnly && i < sizeof(Counters) / 8 && (i < skip0 || i >= skip1))
      reinterpret_cast<uint64_t *>(host)[i] = c.w[q];
  }
  if (threadIdx.x == 0) {
    host->frontier = fc.frontier;
    host->frontier_edges = fc.edges;
    host->dirty = fc.dirty;
    host->frontier_maxdeg = fc.maxdeg;
    host->pull_skipped = fc.skipped;
    host->pull_skipped_hot = fc.skipped_hot;
    host->pull_skipped_rows = fc.skipped_rows;
  }
}

// Everything stored to the host's copy is there before its sequence number: the
// first wave stores both, so that one release is enough (a system fence of every
// wave before it took 0.8 us more per superstep).  The barrier keeps the other
// waves from clearing counters that the first has not read.
__device__ __forceinline__ void publish_seq(uint32_t *host_seq, uint32_t seq)
{
  if (threadIdx.x == 0) __hip_atomic_store(host_seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  __syncthreads();
}

// push launchers (push.hip): the active list's arcs into the memory side's
// updates, or (edge shipping) into the compute side's
template <class Op>
grd_status push_launch(grd_state *s);
template <class Op>
grd_status ship_launch(grd_state *s);
// pull launchers (pull.hip)
template <class Op>
grd_status bsp_pull_launch(grd_state *s, const uint32_t *cw);
template <class Op>
grd_status bsp_pull_fixup(grd_state *s);
// CC / SSSP pull measured with time_kernel: counts the cold arcs of done rows
grd_status pull_done_arcs(grd_state *s);
// the hot pass of the hot / cold split for the BSP pull (tiers.hip)
template <class Op>
grd_status bsp_pull_hot(grd_state *s);
// its cold pass (cold.hip); skip: a flag per cold block (k_row_blocks_done),
// bcnt: the superstep's bound (either may be null)
template <class Op>
grd_status bsp_pull_cold(grd_state *s, const uint8_t *skip, const Counters *bcnt);

}  // namespace grd
