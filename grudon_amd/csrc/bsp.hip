// bsp.hip -- the BSP superstep of the per-partition operator path on gfx950.
//
// One launch covers every partition: compute slots and memory proxies of all
// partitions are laid out back to back (grd_internal.hpp), so each kernel
// below is a single grid over the concatenation.  Wave64 throughout; the
// bitvector protocol works on 64-bit words, one wave per word (lane = bit).
//
// Reference loops replaced (src/GraphAlgorithm.cpp):
//   k_bcast                       compute pack + memory unpack       :199-343
//   (push.hip) / (pull.hip)       gen_updates (pr/cc/sssp.cpp)  :348-356
//   k_reduce                      memory pack + compute aggregate    :377-581
//   k_update                      update_frontier + apply_updates +
//                                 termination popcount               :643-662
//   k_popc_blocks/k_scan_blocks/k_word_rank  DynamicBitSet::getOffsets ranks
#include <algorithm>
#include <cstring>

#include "grd_device.hpp"
#include "grd_internal.hpp"
#include "grd_ops.hpp"

namespace grd {

// ------------------------------------------------------------------------
// word popcount ranks (exclusive prefix of set bits per 64-bit word)
// ------------------------------------------------------------------------

constexpr int kWordsPerScanBlock = 1024;  // 256 threads x 4 words

__global__ void __launch_bounds__(kBlock) k_popc_blocks(const uint64_t *__restrict__ w, uint32_t nw, uint32_t *blk)
{
  uint32_t base = blockIdx.x * kWordsPerScanBlock + threadIdx.x * 4;
  uint32_t c = 0;
#pragma unroll
  for (int i = 0; i < 4; i++)
    if (base + i < nw) c += __popcll(w[base + i]);
  c = block_sum(c);
  if (threadIdx.x == 0) blk[blockIdx.x] = c;
}

// single block of 1024 threads: exclusive scan of nb partials, total -> *total
__global__ void __launch_bounds__(1024) k_scan_blocks(uint32_t *blk, uint32_t nb, uint32_t *total)
{
  __shared__ uint32_t s_w[16];
  uint32_t per = (nb + 1023) / 1024;
  uint32_t b0 = threadIdx.x * per;
  uint32_t local = 0;
  for (uint32_t i = 0; i < per; i++)
    if (b0 + i < nb) local += blk[b0 + i];
  uint32_t inc = wave_incl_scan(local);
  if (lane_id() == kWave - 1) s_w[threadIdx.x / kWave] = inc;
  __syncthreads();
  uint32_t wb = 0, tot = 0;
  for (int i = 0; i < 16; i++) {
    if (i < (int)(threadIdx.x / kWave)) wb += s_w[i];
    tot += s_w[i];
  }
  uint32_t run = wb + inc - local;
  for (uint32_t i = 0; i < per; i++)
    if (b0 + i < nb) {
      uint32_t x = blk[b0 + i];
      blk[b0 + i] = run;
      run += x;
    }
  if (threadIdx.x == 0) *total = tot;
}

__global__ void __launch_bounds__(kBlock) k_word_rank(const uint64_t *__restrict__ w, uint32_t nw,
                                                      const uint32_t *__restrict__ blk, uint32_t *__restrict__ wrank)
{
  uint32_t base = blockIdx.x * kWordsPerScanBlock + threadIdx.x * 4;
  uint32_t c[4], s = 0;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    c[i] = (base + i < nw) ? (uint32_t)__popcll(w[base + i]) : 0u;
    s += c[i];
  }
  uint32_t tot;
  uint32_t ex = block_excl_scan(s, &tot) + blk[blockIdx.x];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    if (base + i < nw) wrank[base + i] = ex;
    ex += c[i];
  }
}

// Short bitmaps in one launch: a workgroup of 1024, kRankPer consecutive words
// per thread.  (Three launches of 2.5 us each for 4096 words; one of 3.)
constexpr uint32_t kRankPer = 8;
__global__ void __launch_bounds__(1024) k_word_rank_one(const uint64_t *__restrict__ w, uint32_t nw,
                                                        uint32_t *__restrict__ wrank, uint32_t *total)
{
  __shared__ uint32_t s_w[16];
  const uint32_t base = threadIdx.x * kRankPer;
  uint32_t c[kRankPer], sum = 0;
#pragma unroll
  for (uint32_t i = 0; i < kRankPer; i++) c[i] = base + i < nw ? (uint32_t)__popcll(w[base + i]) : 0u;
#pragma unroll
  for (uint32_t i = 0; i < kRankPer; i++) sum += c[i];
  const uint32_t inc = wave_incl_scan(sum);
  if (lane_id() == kWave - 1) s_w[wave_in_block()] = inc;
  __syncthreads();
  uint32_t ex = inc - sum, tot = 0;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    if (i < wave_in_block()) ex += s_w[i];
    tot += s_w[i];
  }
#pragma unroll
  for (uint32_t i = 0; i < kRankPer; i++) {
    if (base + i < nw) wrank[base + i] = ex;
    ex += c[i];
  }
  if (threadIdx.x == 0) *total = tot;
}

static grd_status word_ranks(hipStream_t st, const uint64_t *w, uint32_t nw, uint32_t *blk, uint32_t *wrank,
                             uint32_t *total)
{
  if (nw <= 1024 * kRankPer) {
    hipLaunchKernelGGL(k_word_rank_one, dim3(1), dim3(1024), 0, st, w, nw, wrank, total);
    GRD_HIP(hipGetLastError());
    return GRD_OK;
  }
  uint32_t nb = (nw + kWordsPerScanBlock - 1) / kWordsPerScanBlock;
  if (nb == 0) nb = 1;
  hipLaunchKernelGGL(k_popc_blocks, dim3(nb), dim3(kBlock), 0, st, w, nw, blk);
  hipLaunchKernelGGL(k_scan_blocks, dim3(1), dim3(1024), 0, st, blk, nb, total);
  hipLaunchKernelGGL(k_word_rank, dim3(nb), dim3(kBlock), 0, st, w, nw, blk, wrank);
  GRD_HIP(hipGetLastError());
  return GRD_OK;
}

// Grid of the grid-stride word loops (init): up to 64 workgroups per CU.
static inline uint32_t wave_grid(const grd_ctx *ctx, uint64_t nwords)
{
  uint64_t want = (nwords + kWavesPerBlock - 1) / kWavesPerBlock;
  uint64_t cap = (uint64_t)ctx->num_cus * 64;
  return (uint32_t)std::max<uint64_t>(1, std::min(want, cap));
}

// Word-group passes (exchange, update, bucket selection): each wave owns kG
// consecutive bitmap words.  Lane j < kG loads word j of the group (one
// coalesced access), the lanes finish their zero words themselves, and the wave
// then takes the nonzero words with one lane per bit.  A sparse superstep
// therefore costs one pass over the bitmap.  kG is 8, or 2 while groups of 2
// still fit the waves the chip holds: a short bitmap then spreads over four
// times the waves, each with a quarter of the words to work through in turn
// (4096 words: the reduce 10.0 -> 5.1 us, the update 7.6 -> 4.2, the broadcast
// 5.2 -> 3.8).
constexpr uint32_t kGroupWide = 8, kGroupNarrow = 2;

template <uint32_t kG>
__device__ __forceinline__ uint32_t group_base()
{
  return (blockIdx.x * kWavesPerBlock + wave_in_block()) * kG;
}

__device__ __forceinline__ uint64_t shfl_u64(uint64_t x, int src)
{
  const uint32_t lo = __shfl((uint32_t)x, src, kWave), hi = __shfl((uint32_t)(x >> 32), src, kWave);
  return ((uint64_t)hi << 32) | lo;
}

static inline uint32_t group_grid(uint64_t nwords, uint32_t kg)
{
  const uint64_t per = (uint64_t)kg * kWavesPerBlock;
  return (uint32_t)std::max<uint64_t>(1, (nwords + per - 1) / per);
}

// Passes that end in a share of the counters (update, reduce, bucket selection)
// or an atomic (the broadcast's smallest value) loop over the groups from a grid
// of at most this many workgroups per CU.
constexpr uint32_t kLoopBlocksPerCU = 8;

static inline uint32_t loop_grid(const grd_ctx *ctx, uint64_t nwords, uint32_t kg = kGroupWide)
{
  return std::min<uint32_t>(group_grid(nwords, kg), (uint32_t)ctx->num_cus * kLoopBlocksPerCU);
}

// groups of two words fit one round of the looping grid
static inline bool narrow_groups(const grd_ctx *ctx, uint64_t nwords)
{
  return nwords <= (uint64_t)ctx->num_cus * kLoopBlocksPerCU * kWavesPerBlock * kGroupNarrow;
}

// ------------------------------------------------------------------------
// init
// ------------------------------------------------------------------------

__global__ void __launch_bounds__(kBlock) k_fill_u32(uint32_t *p, uint64_t n, uint32_t v)
{
  for (uint64_t i = blockIdx.x * (uint64_t)kBlock + threadIdx.x; i < n; i += (uint64_t)gridDim.x * kBlock) p[i] = v;
}
// the arrays a state starts from
struct InitArrays {
  uint64_t *F, *Dc, *Pend, *bvB;      // [S/64]
  uint64_t *Du, *bvR;                 // [P/64]
  uint32_t *valB;                     // [S]
  uint32_t *mprop, *mupd, *valR;      // [P]
};

// compute-side init (pr.cpp:25-50, cc.cpp:24-36, sssp.cpp:22-46), and the
// bitmaps, wires and memory-side values cleared, in one launch; a wave per
// 64-vertex word
__global__ void __launch_bounds__(kBlock) k_init_state(int algo, uint32_t nw, uint32_t nwP,
                                                       const uint32_t *__restrict__ slot_gid,
                                                       const uint32_t *__restrict__ deg, void *prop_, void *upd_,
                                                       float *pr, InitArrays A, uint32_t neutral, uint32_t source_slot)
{
  const int wpb = kWavesPerBlock;
  for (uint32_t w = blockIdx.x * wpb + wave_in_block(); w < nwP; w += gridDim.x * wpb) {
    const uint32_t p = w * 64 + lane_id();
    A.mprop[p] = neutral;
    A.mupd[p] = neutral;
    A.valR[p] = neutral;
    if (lane_id() == 0) {
      A.Du[w] = 0;
      A.bvR[w] = 0;
    }
  }
  for (uint32_t w = blockIdx.x * wpb + wave_in_block(); w < nw; w += gridDim.x * wpb) {
    uint32_t s = w * 64 + lane_id();
    uint32_t gid = slot_gid[s];
    bool valid = gid != 0xFFFFFFFFu;
    bool f = false;
    if (algo == GRD_PR) {
      float *prop = (float *)prop_, *upd = (float *)upd_;
      uint32_t d = deg[s];
      if (valid && d != 0) {
        prop[s] = (float)(0.85 * (1.0 - 0.85) / (double)d);
        pr[s] = (float)(1.0 - 0.85);
        f = true;
      } else {
        prop[s] = 0.0f;
        pr[s] = 0.0f;
      }
      upd[s] = 0.0f;
    } else {
      uint32_t *prop = (uint32_t *)prop_, *upd = (uint32_t *)upd_;
      if (algo == GRD_CC) {
        prop[s] = valid ? gid : 0xFFFFFFFFu;
        upd[s] = 0xFFFFFFFFu;
        f = valid;
      } else {
        bool src = (s == source_slot);
        prop[s] = src ? 0u : 0xFFFFFFFFu;
        upd[s] = src ? 0u : 0xFFFFFFFFu;
        f = src;
      }
    }
    A.valB[s] = neutral;
    uint64_t fm = __ballot(f);
    if (lane_id() == 0) {
      A.F[w] = fm;
      A.Dc[w] = 0;
      A.Pend[w] = 0;
      A.bvB[w] = 0;
    }
  }
}

// ------------------------------------------------------------------------
// broadcast: compute -> memory (bitvector = frontier words of the pair)
// ------------------------------------------------------------------------

// Send and receive in one pass.  A wave packs its group's words into the
// pairs' bitvectors and values (the wire) and puts the same values into the
// own proxies: the slot words of a pair map one to one onto its proxy words
// (word_dst), so the receiver needs nothing that the sender does not hold.
// For a push the active proxies get their value and the active list; for a
// pull (want_list == 0) every own proxy is written, inactive ones with the
// combine identity, so that the pull gathers one value per arc and needs no
// activity test.  With fmin (a CC / SSSP pull), also the smallest value sent:
// the grid then loops over the groups (loop_grid), so that one atomic per
// workgroup carries it.  Every load of a group is issued before its first
// store.  (With k_reduce, k_update, k_init_state and the one-launch ranks: CC on a thousand
// vertices 314 -> 218 us a solve, hop SSSP by pushes on twenty thousand 727 -> 513,
// delta-push PageRank on RMAT-18 85 -> 71 us a superstep.)
template <typename V, uint32_t kG>
__global__ void __launch_bounds__(kBlock) k_bcast(uint32_t nw, const uint64_t *__restrict__ F,
                                                  const V *__restrict__ prop, const uint32_t *__restrict__ wrank,
                                                  const uint32_t *__restrict__ word_dst, int dense, int want_list,
                                                  V ident, uint64_t *__restrict__ bv, V *__restrict__ val,
                                                  V *__restrict__ mprop, uint32_t *__restrict__ AL, unsigned int *fmin)
{
  static_assert(sizeof(V) == 4, "4-byte values on the wire");
  const int l = lane_id();
  const bool ranks = !dense || want_list;
  uint32_t lo = 0xFFFFFFFFu;
  for (uint32_t base = group_base<kG>(); base < nw; base += gridDim.x * kWavesPerBlock * kG) {
    const bool ok = l < (int)kG && base + l < nw;
    const uint64_t mine = ok ? F[base + l] : 0ull;
    const uint32_t pwl = ok ? word_dst[base + l] : 0xFFFFFFFFu;
    const uint32_t rkl = ok && ranks ? wrank[base + l] : 0u;
    if (ok) bv[base + l] = mine;
    // a sparse push walks only the words that hold a frontier vertex
    if (!dense && want_list && __ballot(mine != 0) == 0) continue;
    V x[kG];
    uint64_t word[kG];
#pragma unroll
    for (int j = 0; j < (int)kG; j++) {
      word[j] = shfl_u64(mine, j);
      x[j] = ident;
      if (base + j < nw && (dense || ((word[j] >> l) & 1ull))) x[j] = prop[(base + j) * 64 + l];
    }
#pragma unroll
    for (int j = 0; j < (int)kG; j++) {
      const uint32_t w = base + j, pw = __shfl(pwl, j, kWave), rank = __shfl(rkl, j, kWave);
      if (w >= nw) break;  // uniform over the wave
      const bool on = (word[j] >> l) & 1ull;
      const uint32_t r = rank + (uint32_t)__popcll(word[j] & lanemask_lt());
      if (dense) val[w * 64 + l] = x[j];
      else if (on) val[r] = x[j];
      if (on) {
        const uint32_t u = __builtin_bit_cast(uint32_t, x[j]);
        lo = u < lo ? u : lo;
      }
      if (pw == 0xFFFFFFFFu) continue;
      if (on || !want_list) mprop[pw * 64 + l] = on ? x[j] : ident;
      if (on && want_list) AL[r] = pw * 64 + l;
    }
  }
  if (fmin) {  // uniform: a kernel argument
    lo = block_min(lo);
    // (a workgroup that cannot lower it spares the atomic)
    if (threadIdx.x == 0 && lo < __atomic_load_n(fmin, __ATOMIC_RELAXED)) atomicMin(fmin, lo);
  }
}

// Pull of CC / SSSP, compute side: bit r of Rdone is set when memory proxy r
// belongs to a vertex whose value is at or below b = the smallest value
// broadcast this superstep plus the smallest arc increment (0 for CC, 1 for
// hop counts, the smallest arc weight for weighted SSSP; saturating).  Every
// candidate of the superstep is Op::edge of a broadcast value over an arc,
// never below b, so no candidate can improve such a row and the pull may
// leave its arcs out.  A wave covers one word of rows.
__global__ void __launch_bounds__(kBlock) k_rows_done(uint32_t nwP, const uint32_t *__restrict__ proxy_slot,
                                                      const uint32_t *__restrict__ prop, const Counters *cnt,
                                                      uint32_t inc, uint64_t *__restrict__ Rdone)
{
  const uint32_t f = cnt->fmin, fmin = f + inc < f ? 0xFFFFFFFFu : f + inc;
  const uint64_t nrow = (uint64_t)nwP * 64;
  for (uint64_t r = (uint64_t)blockIdx.x * kBlock + threadIdx.x; r < nrow; r += (uint64_t)gridDim.x * kBlock) {
    const uint32_t sl = proxy_slot[r];
    const bool done = sl != kNone && prop[sl] <= fmin;
    const uint64_t m = __ballot(done);
    if (lane_id() == 0) Rdone[r >> 6] = m;
  }
}

// ------------------------------------------------------------------------
// reduce: memory -> compute (bitvector = dirty words of the pair)
// ------------------------------------------------------------------------

// Send and receive in one pass: a wave packs its group's dirty words and values
// into the pairs' messages (the wire) and aggregates the same values into the
// compute side, all loads of the group (values, slots, and for min-combines the
// current values) before the first store, all atomics before the first mark.
// A capped grid loops over the groups (one share of the counters per workgroup).
template <class Op, uint32_t kG>
__global__ void __launch_bounds__(kBlock) k_reduce(uint32_t nw, uint64_t *__restrict__ Du,
                                                   typename Op::V *__restrict__ mupd,
                                                   const uint32_t *__restrict__ wrank,
                                                   const uint32_t *__restrict__ proxy_slot, int dense,
                                                   uint64_t *__restrict__ bv, typename Op::V *__restrict__ val,
                                                   typename Op::V *upd, uint64_t *Dc, uint32_t *__restrict__ share)
{
  using V = typename Op::V;
  const int l = lane_id();
  uint32_t ndirty = 0;
  for (uint32_t base = group_base<kG>(); base < nw; base += gridDim.x * kWavesPerBlock * kG) {
    const bool ok = l < (int)kG && base + l < nw;
    const uint64_t mine = ok ? Du[base + l] : 0ull;
    const uint32_t rkl = (ok && !dense) ? wrank[base + l] : 0u;
    if (ok) {
      bv[base + l] = mine;
      if (mine) Du[base + l] = 0;
    }
    ndirty += (uint32_t)__popcll(mine);
    if (!dense && __ballot(mine != 0) == 0) continue;
    uint64_t word[kG];
    uint32_t s[kG];
    V x[kG];
#pragma unroll
    for (int j = 0; j < (int)kG; j++) {
      word[j] = shfl_u64(mine, j);
      const uint32_t p = (base + j) * 64 + l;
      const bool on = (word[j] >> l) & 1ull;
      s[j] = 0xFFFFFFFFu;
      x[j] = V{};
      if (base + j < nw && (dense || on)) x[j] = mupd[p];
      if (on) s[j] = proxy_slot[p];
    }
    V cur[kG];
    if constexpr (Op::kMin) {
#pragma unroll
      for (int j = 0; j < (int)kG; j++)
        cur[j] = s[j] != 0xFFFFFFFFu ? __atomic_load_n(upd + s[j], __ATOMIC_RELAXED) : V{};
    }
#pragma unroll
    for (int j = 0; j < (int)kG; j++) {
      const uint32_t w = base + j, p = w * 64 + l, rank = __shfl(rkl, j, kWave);
      if (w >= nw) break;  // uniform over the wave
      const bool on = (word[j] >> l) & 1ull;
      if (dense) val[p] = x[j];
      else if (on) val[rank + (uint32_t)__popcll(word[j] & lanemask_lt())] = x[j];
      // PropertyList::clear (DistributedGraph.hpp:140-166); the min-combines keep theirs
      if (!Op::kMin && on) mupd[p] = V(0);
    }
    // aggregate(): minUpdate / addUpdate, then the dirty marks of the wave
    bool mark[kG];
#pragma unroll
    for (int j = 0; j < (int)kG; j++) {
      mark[j] = false;
      if (s[j] != 0xFFFFFFFFu) {
        if constexpr (Op::kMin) {
          mark[j] = x[j] < cur[j];
          if (mark[j]) cur[j] = atomicMin(upd + s[j], x[j]);
        } else {
          atomicAdd(upd + s[j], x[j]);
          mark[j] = true;
        }
      }
    }
#pragma unroll
    for (int j = 0; j < (int)kG; j++) {
      if (word[j] == 0) continue;  // uniform over the wave
      if constexpr (Op::kMin) mark[j] = mark[j] && x[j] < cur[j];
      mark_wave(Dc, s[j], mark[j]);
    }
  }
  uint32_t t = block_sum(ndirty);
  if (threadIdx.x == 0 && t) share[blockIdx.x] += t;
}

// The dense reduce of a min-combine from the compute side: a proxy's update only
// falls and the vertex has seen every earlier one, so the smallest of a vertex's
// proxies (its own, at the same place of its pair, and its cross mirrors, which
// lie in slot order) is the new value whichever of them are dirty, and a wave
// that owns a word of slots needs no atomics.  The wire gets the same values.  Bound by
// the bytes: four arrays of the proxies and three of the slots.  CC over RMAT-24
// symmetrized, M = 4: 294 us a superstep with an atomic per dirty proxy, now 142;
// weighted SSSP over RMAT-22 102 -> 35.  (Small layouts keep k_reduce's narrow
// groups: one launch of latency either way.)
constexpr int kMinWords = 4;
template <typename V>
__global__ void __launch_bounds__(kBlock) k_reduce_min(uint32_t nwP, uint64_t *__restrict__ Du,
                                                       uint64_t *__restrict__ bv, uint32_t nwS,
                                                       const uint32_t *__restrict__ word_dst,
                                                       const uint32_t *__restrict__ xptr,
                                                       const uint32_t *__restrict__ xlist,
                                                       const V *__restrict__ mupd, V *__restrict__ val,
                                                       V *__restrict__ upd, uint64_t *__restrict__ Dc,
                                                       uint32_t *__restrict__ share)
{
  const uint32_t l = lane_id(), stride = gridDim.x * kWavesPerBlock;
  uint32_t ndirty = 0;
  for (uint32_t w = blockIdx.x * kBlock + threadIdx.x; w < nwP; w += gridDim.x * kBlock) {
    const uint64_t mine = Du[w];
    bv[w] = mine;
    if (mine) Du[w] = 0;
    ndirty += (uint32_t)__popcll(mine);
  }
  constexpr V kTop = ~V(0);
  for (uint32_t w0 = blockIdx.x * kWavesPerBlock + wave_in_block(); w0 < nwS; w0 += kMinWords * stride) {
    uint32_t pw[kMinWords], x0[kMinWords], nx[kMinWords], i[kMinWords][3];
    V cur[kMinWords], own[kMinWords], v[kMinWords][3];
#pragma unroll
    for (int j = 0; j < kMinWords; j++) {
      const uint32_t w = w0 + j * stride, s = (w < nwS ? w : w0) * 64 + l;
      pw[j] = w < nwS ? word_dst[w] : kNone;
      x0[j] = xptr[s];
      nx[j] = xptr[s + 1];
      cur[j] = upd[s];
    }
    // the own value and up to three cross mirrors' (every vertex at M <= 4) together
#pragma unroll
    for (int j = 0; j < kMinWords; j++) {
      nx[j] = w0 + j * stride < nwS ? nx[j] - x0[j] : 0u;
#pragma unroll
      for (int q = 0; q < 3; q++) i[j][q] = nx[j] > (uint32_t)q ? xlist[x0[j] + q] : 0u;
      own[j] = pw[j] != kNone ? mupd[pw[j] * 64 + l] : kTop;
    }
#pragma unroll
    for (int j = 0; j < kMinWords; j++)
#pragma unroll
      for (int q = 0; q < 3; q++) v[j][q] = nx[j] > (uint32_t)q ? mupd[i[j][q]] : kTop;
#pragma unroll
    for (int j = 0; j < kMinWords; j++) {
      const uint32_t w = w0 + j * stride;
      if (w >= nwS) break;  // uniform over the wave
      V m = own[j];
      if (pw[j] != kNone) val[pw[j] * 64 + l] = own[j];
#pragma unroll
      for (int q = 0; q < 3; q++) {
        m = min(m, v[j][q]);
        if (nx[j] > (uint32_t)q) val[i[j][q]] = v[j][q];
      }
      for (uint32_t x = x0[j] + 3; x < x0[j] + nx[j]; x++) {
        const uint32_t p = xlist[x];
        const V u = mupd[p];
        val[p] = u;
        m = min(m, u);
      }
      const bool mark = m < cur[j];
      if (mark) upd[w * 64 + l] = m;
      const uint64_t d = __ballot(mark);
      if (l == 0 && d) Dc[w] |= d;
    }
  }
  uint32_t t = block_sum(ndirty);
  if (threadIdx.x == 0 && t) share[blockIdx.x] += t;
}

// ------------------------------------------------------------------------
// update: update_frontier + apply_updates + frontier popcount
// ------------------------------------------------------------------------

// a workgroup's share of the next frontier (one barrier, no atomic: with three
// atomics per workgroup the update of 65536 words took 29 us, now 7.6)
__device__ __forceinline__ void share_frontier(uint64_t vertices, uint64_t edges, uint32_t maxdeg, BlockShare *share)
{
  __shared__ uint64_t s_c[kWavesPerBlock];
  __shared__ uint32_t s_m[kWavesPerBlock];
  uint64_t c = wave_sum((vertices << 32) + edges);
  uint32_t m = wave_max(maxdeg);
  if (lane_id() == 0) {
    s_c[wave_in_block()] = c;
    s_m[wave_in_block()] = m;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int i = 1; i < kWavesPerBlock; i++) {
      c += s_c[i];
      m = max(m, s_m[i]);
    }
    share[blockIdx.x] = BlockShare{c, m, 0};
  }
}

// A capped grid walks the word groups (the loop is wave-uniform), so that few
// blocks leave a share of the counters.  All loads of a group's
// words are issued before any is used, and lane j stores word j's bitmap words
// (word by word, a group was a chain of up to eight dependent round trips:
// 11 us on 4096 words, 36 on 65536).
template <int ALGO, uint32_t kG>  // GRD_PR, GRD_CC or GRD_SSSP
__global__ void __launch_bounds__(kBlock) k_update(uint32_t nw, uint64_t *__restrict__ Dc, void *prop_, void *upd_,
                                                   float *__restrict__ pr, const uint32_t *__restrict__ deg,
                                                   uint64_t *__restrict__ F, uint64_t *__restrict__ Pend,
                                                   unsigned long long hi, int use_delta,
                                                   BlockShare *__restrict__ share)
{
  using V = typename std::conditional<ALGO == GRD_PR, float, uint32_t>::type;
  V *__restrict__ prop = (V *)prop_;
  V *__restrict__ upd = (V *)upd_;
  const int l = lane_id();
  uint64_t f_cnt = 0, f_edges = 0;
  uint32_t f_max = 0;
  for (uint32_t base = group_base<kG>(); base < nw; base += gridDim.x * kWavesPerBlock * kG) {
    const bool ok = l < (int)kG && base + l < nw;
    const uint64_t mine = ok ? Dc[base + l] : 0ull;
    uint64_t fmine = 0, pmine = 0;
    if (use_delta && mine) pmine = Pend[base + l];
    if (__ballot(mine != 0)) {
      uint64_t d[kG];
      V u[kG], o[kG];
      uint32_t dg[kG];
#pragma unroll
      for (int j = 0; j < (int)kG; j++) {
        d[j] = shfl_u64(mine, j);
        const uint32_t s = (base + j) * 64 + l;
        u[j] = o[j] = V(0);
        dg[j] = 0;
        if ((d[j] >> l) & 1ull) {
          u[j] = upd[s];
          o[j] = ALGO == GRD_PR ? (V)pr[s] : prop[s];
          dg[j] = deg[s];
        }
      }
#pragma unroll
      for (int j = 0; j < (int)kG; j++) {
        if (d[j] == 0) continue;  // uniform over the wave
        const uint32_t s = (base + j) * 64 + l;
        bool f = false, pend = false;
        if ((d[j] >> l) & 1ull) {
          if constexpr (ALGO == GRD_PR) {
            if ((double)u[j] > 1e-6) {  // pr.cpp:133-142 and :76-83 (prev is always 0 here)
              f = true;
              pr[s] = o[j] + u[j];
              prop[s] = (float)(0.85 * (double)u[j] / (double)dg[j]);
              upd[s] = 0.0f;
            }
          } else if (o[j] > u[j]) {  // cc.cpp:100-106, sssp.cpp:102-108
            prop[s] = u[j];
            if (use_delta && (unsigned long long)u[j] >= hi) pend = true;
            else f = true;
          }
        }
        if (f) {
          f_edges += dg[j];
          f_max = max(f_max, dg[j]);
        }
        const uint64_t fm = __ballot(f);
        if (l == j) fmine = fm;
        if (use_delta) {
          const uint64_t pm = __ballot(pend);
          if (l == j) pmine = (pmine | pm) & ~fm;
        }
      }
    }
    if (ok) {
      F[base + l] = fmine;  // (nothing changed: an empty next-frontier word)
      if (mine) {
        Dc[base + l] = 0;
        if (use_delta) Pend[base + l] = pmine;
      }
      f_cnt += (uint64_t)__popcll(fmine);
    }
  }
  share_frontier(f_cnt, f_edges, f_max, share);
}

// delta-stepping: smallest pending distance and pending count
template <uint32_t kG>
__global__ void __launch_bounds__(kBlock) k_pend_min(uint32_t nw, const uint64_t *__restrict__ Pend,
                                                     const uint32_t *__restrict__ prop, Counters *cnt)
{
  const int l = lane_id();
  uint32_t mn = 0xFFFFFFFFu;
  uint64_t c = 0;
  // capped grid, wave-uniform loop over the word groups
  for (uint32_t base = group_base<kG>(); base < nw; base += gridDim.x * kWavesPerBlock * kG) {
    const bool ok = l < (int)kG && base + l < nw;
    const uint64_t mine = ok ? Pend[base + l] : 0ull;
    uint64_t todo = __ballot(mine != 0);
    while (todo) {
      const int j = __ffsll((unsigned long long)todo) - 1;
      todo &= todo - 1;
      const uint64_t pm = shfl_u64(mine, j);
      if ((pm >> l) & 1ull) {
        uint32_t v = prop[(base + j) * 64 + l];
        mn = v < mn ? v : mn;
        c++;
      }
    }
  }
  mn = block_min(mn);
  c = block_sum(c);
  if (threadIdx.x == 0 && c) {
    if (mn < __atomic_load_n(&cnt->pend_min, __ATOMIC_RELAXED)) atomicMin(&cnt->pend_min, mn);
    atomicAdd(&cnt->pending, (unsigned long long)c);
  }
}

// delta-stepping: move pending vertices below the new bucket bound into F
// (loads and stores of a group as in k_update)
template <uint32_t kG>
__global__ void __launch_bounds__(kBlock) k_select(uint32_t nw, uint64_t *__restrict__ Pend,
                                                   const uint32_t *__restrict__ prop, const uint32_t *__restrict__ deg,
                                                   unsigned long long hi, uint64_t *__restrict__ F,
                                                   BlockShare *__restrict__ share)
{
  const int l = lane_id();
  uint64_t f_cnt = 0, f_edges = 0;
  uint32_t f_max = 0;
  for (uint32_t base = group_base<kG>(); base < nw; base += gridDim.x * kWavesPerBlock * kG) {
    const bool ok = l < (int)kG && base + l < nw;
    const uint64_t mine = ok ? Pend[base + l] : 0ull;
    uint64_t fmine = 0;
    if (__ballot(mine != 0)) {
      uint64_t pm[kG];
      uint32_t v[kG], dg[kG];
#pragma unroll
      for (int j = 0; j < (int)kG; j++) {
        pm[j] = shfl_u64(mine, j);
        const uint32_t s = (base + j) * 64 + l;
        v[j] = 0xFFFFFFFFu;
        dg[j] = 0;
        if ((pm[j] >> l) & 1ull) {
          v[j] = prop[s];
          dg[j] = deg[s];
        }
      }
#pragma unroll
      for (int j = 0; j < (int)kG; j++) {
        const bool f = ((pm[j] >> l) & 1ull) && (unsigned long long)v[j] < hi;
        const uint64_t fm = __ballot(f);
        if (l == j) fmine = fm;
        if (f) {
          f_edges += dg[j];
          f_max = max(f_max, dg[j]);
        }
      }
    }
    if (ok) {
      F[base + l] = fmine;
      if (fmine) Pend[base + l] = mine & ~fmine;
      f_cnt += (uint64_t)__popcll(fmine);
    }
  }
  share_frontier(f_cnt, f_edges, f_max, share);
}

__global__ void __launch_bounds__(kBlock) k_zero_counters(Counters *cnt, Shares sh) { zero_counters(cnt, sh); }

// The counters into the state's pinned copy, and to their start for the next
// superstep.  The host waits for `seq` behind the copy (op_wait_counters): a
// copy command and a stream synchronisation took 15 us more per superstep.
__global__ void __launch_bounds__(kBlock) k_publish(Counters *cnt, Shares sh, Counters *host, uint32_t *host_seq,
                                                    uint32_t seq)
{
  const CounterWords words = counter_words(cnt);
  const FrontierCounts fc = sum_shares(sh);
  copy_counters(words, host, fc);
  publish_seq(host_seq, seq);
  zero_counters(cnt, sh);
}

// single-element aggregate() (API compatibility path)
template <class Op>
__global__ void k_aggregate_one(typename Op::V *upd, uint64_t *Dc, uint32_t slot, typename Op::V x)
{
  if (threadIdx.x == 0 && blockIdx.x == 0) relax<Op, true>(upd, Dc, slot, x);
}

// results by gid
template <typename V>
__global__ void __launch_bounds__(kBlock) k_gather_result(uint32_t S, const uint32_t *__restrict__ slot_gid,
                                                          const V *__restrict__ src, V *__restrict__ out)
{
  for (uint32_t s = blockIdx.x * kBlock + threadIdx.x; s < S; s += gridDim.x * kBlock) {
    uint32_t g = slot_gid[s];
    if (g != 0xFFFFFFFFu) out[g] = src[s];
  }
}

// Up to kSmallOut values into pinned memory: a workgroup per kOutPart of them,
// each wave reporting its end in a flag of its own.  Slots are in degree order,
// so a workgroup looks at all slots and puts the values of its vertices
// in order in LDS first (a 4-byte store across the bus costs as much as a whole
// line).
constexpr uint32_t kOutPart = 4096;
constexpr int kOutBlock = 1024;
__global__ void __launch_bounds__(kOutBlock) k_small_out(const uint32_t *__restrict__ src,
                                                         const uint32_t *__restrict__ gid, uint32_t S, uint32_t n,
                                                         uint32_t *__restrict__ host, uint32_t *flags, uint32_t seq)
{
  __shared__ uint32_t s_o[kOutPart];
  const uint32_t g0 = blockIdx.x * kOutPart, cnt = min(n - g0, kOutPart);
#pragma unroll 8
  for (uint32_t s = threadIdx.x; s < S; s += kOutBlock) {
    const uint32_t g = gid[s], v = src[s];
    if (g != kNone && g - g0 < cnt) s_o[g - g0] = v;
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < cnt; i += kOutBlock) host[g0 + i] = s_o[i];
  if (lane_id() == 0)
    __hip_atomic_store(flags + blockIdx.x * (kOutBlock / kWave) + threadIdx.x / kWave, seq, __ATOMIC_RELEASE,
                       __HIP_MEMORY_SCOPE_SYSTEM);
}

grd_status small_out(grd_ctx *ctx, const uint32_t *src, const uint32_t *gid, uint32_t S, uint32_t n, uint32_t *host,
                     uint32_t *flags, uint32_t seq, uint32_t *nflags)
{
  static_assert((kSmallOut + kOutPart - 1) / kOutPart * (kOutBlock / kWave) <= kSmallFlags, "a flag per wave");
  const uint32_t grid = (n + kOutPart - 1) / kOutPart;
  *nflags = grid * (kOutBlock / kWave);
  hipLaunchKernelGGL(k_small_out, dim3(grid), dim3(kOutBlock), 0, ctx->stream, src, gid, S, n, host, flags, seq);
  GRD_HIP(hipGetLastError());
  return GRD_OK;
}

// ------------------------------------------------------------------------
// host orchestration
// ------------------------------------------------------------------------

// most workgroups of a looping pass (the shares' arrays)
uint32_t loop_blocks(const grd_ctx *ctx) { return (uint32_t)ctx->num_cus * kLoopBlocksPerCU; }

Shares shares(const grd_state *s)
{
  return Shares{s->ushare, s->n_ushare, s->rshare, s->n_rshare, s->sshare, s->n_sshare};
}

grd_status op_zero_counters(grd_state *s)
{
  hipLaunchKernelGGL(k_zero_counters, dim3(1), dim3(kBlock), 0, s->g->ctx->stream, s->cnt, shares(s));
  GRD_HIP(hipGetLastError());
  counters_at_start(s, false);
  return GRD_OK;
}

grd_status op_wait_counters(grd_state *s)
{
  GRD_TRY(wait_pinned(s->g->ctx, host_seq(s->hcnt), s->cnt_seq));
  if (s->bound_at == grd_state::kBoundPublished) {
    s->bound_value = s->hcnt->fmin;
    s->bound_at = grd_state::kBoundOnHost;
  }
  return GRD_OK;
}

grd_status op_read_counters(grd_state *s)
{
  hipLaunchKernelGGL(k_publish, dim3(1), dim3(kBlock), 0, s->g->ctx->stream, s->cnt, shares(s), s->hcnt,
                     host_seq(s->hcnt), ++s->cnt_seq);
  GRD_HIP(hipGetLastError());
  counters_at_start(s, true);
  return op_wait_counters(s);
}

grd_status state_alloc(grd_state *s)
{
  grd_graph *g = s->g;
  const uint64_t S = g->S, P = g->P;
  const uint32_t nwS = (uint32_t)(S / 64), nwP = (uint32_t)(P / 64);
  const uint64_t V = 4;
  DevMem &m = s->mem;
  GRD_TRY(m.alloc(&s->prop, S * V));
  GRD_TRY(m.alloc(&s->upd, S * V));
  if (s->algo == GRD_PR || s->algo == GRD_PR_PULL) GRD_TRY(m.alloc_n(&s->pr, S));
  GRD_TRY(m.alloc_n(&s->F, nwS));
  GRD_TRY(m.alloc_n(&s->Dc, nwS));
  GRD_TRY(m.alloc_n(&s->Pend, nwS));
  GRD_TRY(m.alloc(&s->mprop, P * V));
  GRD_TRY(m.alloc(&s->mupd, P * V));
  GRD_TRY(m.alloc_n(&s->Du, nwP));
  if (s->algo == GRD_CC || s->algo == GRD_SSSP) GRD_TRY(m.alloc_n(&s->Rdone, std::max<uint32_t>(nwP, 1)));
  GRD_TRY(m.alloc_n(&s->bvB, nwS));
  GRD_TRY(m.alloc_n(&s->bvR, nwP));
  GRD_TRY(m.alloc(&s->valB, S * V));
  GRD_TRY(m.alloc(&s->valR, P * V));
  uint32_t nb = (std::max(nwS, nwP) + kWordsPerScanBlock - 1) / kWordsPerScanBlock + 1;
  GRD_TRY(m.alloc_n(&s->blk, nb));
  GRD_TRY(m.alloc_n(&s->wrankB, nwS));
  GRD_TRY(m.alloc_n(&s->wrankR, nwP));
  GRD_TRY(m.alloc_n(&s->totals, 64));
  GRD_TRY(m.alloc_n(&s->AL, S));
  // heavy chunks: a vertex's last chunk may be short, and at most m / kHeavyDeg
  // vertices are heavy
  if (s->algo != GRD_PR_PULL) GRD_TRY(m.alloc_n(&s->heavy, g->m / kHeavyChunk + g->m / kHeavyDeg + 64));
  GRD_TRY(m.alloc(&s->partial, (uint64_t)std::max<uint32_t>(1, g->n_pblk) * 8));
  if (s->algo == GRD_PR_PULL) {
    GRD_TRY(m.alloc_n(&s->red, 2ull * prp_grid(g)));
    if (!g->word_nvalid) {
      // a pair group's valid slots are a prefix of its padded range, so the
      // valid slots of a word are a prefix of the word
      std::vector<uint8_t> nv(std::max<uint32_t>(nwS, 1), 0);
      for (size_t k = 0; k < g->cbase.size(); k++) {
        const uint64_t b0 = g->cbase[k], b1 = b0 + g->ccnt[k];
        if (b0 % 64) return fail(GRD_ERR_STATE, "layout: a pair group does not start on a slot word");
        for (uint64_t w = b0 / 64; w * 64 < b1 && w < nwS; w++)
          nv[w] = (uint8_t)std::min<uint64_t>(64, b1 - std::max<uint64_t>(b0, w * 64));
      }
      GRD_TRY(g->mem.alloc_n(&g->word_nvalid, nv.size()));
      GRD_HIP(hipMemcpyAsync(g->word_nvalid, nv.data(), nv.size(), hipMemcpyHostToDevice, g->ctx->stream));
      GRD_HIP(hipStreamSynchronize(g->ctx->stream));
    }
  }
  if (s->tiled) {
    if (g->tier_mode == 3) {
      // hot / cold: one 4-byte partial per row and per hot segment
      GRD_TRY(m.alloc(reinterpret_cast<void **>(&s->tpart), std::max<uint64_t>(g->n_pairs, 1) * 4));
      GRD_TRY(m.alloc(reinterpret_cast<void **>(&s->tseg), (uint64_t)std::max<uint32_t>(g->n_tblk, 1) * 4));
      GRD_TRY(m.alloc_n(&s->cseg, std::max<uint32_t>(s->cold->nblk, 1)));
    } else {
      GRD_TRY(m.alloc_n(&s->tpart, std::max<uint64_t>(g->n_pairs, 1)));
      GRD_TRY(m.alloc_n(&s->tseg, std::max<uint32_t>(g->n_tblk, 1)));
    }
  }
  if (s->Rdone) {
    // one flag per row block of the pull this state runs
    const uint32_t nblk = bsp_hot_cold(s) ? s->cold->nblk : g->n_pblk;
    GRD_TRY(m.alloc_n(&s->bskip, std::max<uint32_t>(nblk, 1)));
    if (bsp_hot_cold(s)) GRD_TRY(m.alloc_n(&s->hskip, std::max<uint32_t>(g->n_tblk, 1)));
  }
  // the counters and the shares that wait for the next publishing are one
  // piece, so that a snapshot within a superstep holds both in one copy
  const uint64_t lb = loop_blocks(g->ctx);
  const uint64_t cnt_bytes = sizeof(Counters) + 2 * lb * sizeof(SkipShare) + lb * sizeof(uint32_t);
  static_assert(sizeof(Counters) % 8 == 0 && sizeof(SkipShare) % 8 == 0, "the shares are aligned");
  GRD_TRY(m.alloc(reinterpret_cast<void **>(&s->cnt), cnt_bytes));
  s->sshare = reinterpret_cast<SkipShare *>(s->cnt + 1);
  s->rshare = reinterpret_cast<uint32_t *>(s->sshare + 2 * lb);
  GRD_TRY(m.alloc_n(&s->ushare, lb));
  s->n_rshare = loop_grid(g->ctx, nwP, narrow_groups(g->ctx, nwP) ? kGroupNarrow : kGroupWide);
  GRD_TRY(host_counters_take(g->ctx, &s->hcnt));
  // snapshot list: every array whose content carries state between iterations
  s->snap = {{s->prop, nullptr}, {s->upd, nullptr}, {s->F, nullptr},     {s->Dc, nullptr},
             {s->Pend, nullptr}, {s->mprop, nullptr}, {s->mupd, nullptr},
             {s->Du, nullptr}};
  s->snap_bytes = {S * V, S * V, nwS * 8ull, nwS * 8ull, nwS * 8ull, P * V, P * V, nwP * 8ull};
  if (s->pr) {
    s->snap.push_back({s->pr, nullptr});
    s->snap_bytes.push_back(S * 4);
  }
  // the counters carry the pull PageRank's FP64 dangling mass of the next
  // update (ping-pong by iteration parity) and the last residual
  s->snap.push_back({s->cnt, nullptr});
  s->snap_bytes.push_back(cnt_bytes);
  return GRD_OK;
}

grd_status state_init(grd_state *s)
{
  grd_graph *g = s->g;
  hipStream_t st = g->ctx->stream;
  const uint32_t nwS = g->S / 64, nwP = g->P / 64;
  const uint32_t neutral = (s->algo == GRD_PR) ? 0u : 0xFFFFFFFFu;  // PR: 0.0f bit pattern
  uint32_t source_slot = 0xFFFFFFFFu;
  if (s->algo == GRD_SSSP) source_slot = g->h_gid_slot[s->prm.source];
  const InitArrays A{s->F, s->Dc, s->Pend, s->bvB, s->Du, s->bvR, (uint32_t *)s->valB,
                     (uint32_t *)s->mprop, (uint32_t *)s->mupd, (uint32_t *)s->valR};
  hipLaunchKernelGGL(k_init_state, dim3(wave_grid(g->ctx, std::max(nwS, nwP))), dim3(kBlock), 0, st, s->algo, nwS, nwP,
                     g->slot_gid, g->slot_deg, s->prop, s->upd, s->pr, A, neutral, source_slot);
  GRD_HIP(hipGetLastError());
  GRD_TRY(op_zero_counters(s));
  s->hi = (s->algo == GRD_SSSP && s->prm.delta) ? (uint64_t)s->prm.delta : ~0ull;
  // initial frontier statistics for the first schedule decision: PR starts
  // from every vertex with out-edges, CC from every vertex, SSSP from the source
  uint64_t fr = 0, fe = 0;
  uint32_t mx = 0;
  if (s->algo == GRD_PR) {
    fr = g->n - g->n_sinks;
    fe = g->m;
    mx = g->max_deg;
  } else if (s->algo == GRD_CC) {
    fr = g->n;
    fe = g->m;
    mx = g->max_deg;
  } else {
    fr = 1;
    fe = mx = g->h_deg[s->prm.source];
  }
  s->last_frontier = fr;
  s->prev_frontier = fr;
  s->last_frontier_edges = fe;
  s->last_maxdeg = mx;
  s->last_dirty = 0;
  s->iteration = 0;
  s->bytes = 0;
  s->edges = 0;
  s->bcast_option = -1;
  s->sel_queued = false;
  s->xb_dense = s->xr_dense = -1;
  if (g->C > 1) {  // per-partition frontier sizes for the first NDPEngine vote
    GRD_TRY(op_frontier_parts(s));
    GRD_TRY(op_read_counters(s));
  }
  take_frontier_parts(s);
  return GRD_OK;
}

// translation-table words of every pair (for the exchange byte count)
static uint64_t bitvector_bytes(const grd_graph *g)
{
  uint64_t b = 0;
  for (int c = 0; c < g->C; c++)
    for (int m = 0; m < g->M; m++) {
      uint64_t T = (uint64_t)g->ccnt[(size_t)c * g->M + m] + g->xcnt[(size_t)m * g->C + c];
      b += 8 * ((T + 63) / 64);
    }
  return b;
}

__global__ void __launch_bounds__(kBlock) k_min_u32(uint64_t n, const uint32_t *__restrict__ x, uint32_t *out)
{
  uint32_t lo = 0xFFFFFFFFu;
  for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (uint64_t)gridDim.x * kBlock)
    lo = x[i] < lo ? x[i] : lo;
  lo = block_min(lo);
  if (threadIdx.x == 0 && lo != 0xFFFFFFFFu) atomicMin(out, lo);
}

// the smallest arc weight of a weighted graph (once per graph; 2^32 - 1
// when it has no arcs)
static grd_status graph_min_weight(grd_graph *g, uint32_t *out)
{
  if (!g->wmin_known) {
    hipStream_t st = g->ctx->stream;
    DevMem tmp(g->ctx);
    uint32_t *d = nullptr;
    GRD_TRY(tmp.alloc_n(&d, 1));
    hipLaunchKernelGGL(k_fill_u32, dim3(1), dim3(kBlock), 0, st, d, 1, 0xFFFFFFFFu);
    if (g->m && g->cw)
      hipLaunchKernelGGL(k_min_u32, dim3(std::min<uint64_t>((g->m + kBlock - 1) / kBlock, (uint64_t)g->ctx->num_cus * 8)),
                         dim3(kBlock), 0, st, g->m, g->cw, d);
    GRD_HIP(hipGetLastError());
    GRD_HIP(hipMemcpyAsync(&g->wmin, d, 4, hipMemcpyDeviceToHost, st));
    GRD_HIP(hipStreamSynchronize(st));
    g->wmin_known = true;
  }
  *out = g->wmin;
  return GRD_OK;
}

grd_status op_broadcast(grd_state *s, int option)
{
  grd_graph *g = s->g;
  hipStream_t st = g->ctx->stream;
  const uint32_t nwS = g->S / 64;
  const bool pull = option & 1, dense = option & 2;
  const bool need_rank = !dense || !pull;
  s->cnt_clean = s->bcast_stale = false;
  if (!pull) {
    s->al_vertices = s->last_frontier;
    s->al_edges = s->last_frontier_edges;
    s->al_maxdeg = s->last_maxdeg;
  }
  s->xb_dense = dense ? 1 : 0;
  s->xr_dense = -1;
  if (need_rank) GRD_TRY(word_ranks(st, s->F, nwS, s->blk, s->wrankB, s->totals + 0));
  // a pull of CC / SSSP also sends the smallest value broadcast and the rows
  // that cannot improve (the pull leaves out what cannot change unless the
  // caller asked for every row); the rows-done bitmap not in the first
  // superstep, where every vertex still holds its initial value and at most
  // the frontier's smallest is done
  const bool bound = pull && s->algo != GRD_PR && !s->prm.pull_every_row;
  const bool rows_done = bound && s->iteration > 0;
  const uint32_t ident = (s->algo == GRD_PR) ? 0u : 0xFFFFFFFFu;  // 0.0f or the min identity
  const auto send = [&](auto kernel, uint32_t kg) {
    hipLaunchKernelGGL(kernel, dim3(bound ? loop_grid(g->ctx, nwS, kg) : group_grid(nwS, kg)), dim3(kBlock), 0, st, nwS,
                       s->F, (const uint32_t *)s->prop, s->wrankB, g->word_dst, (int)dense, (int)!pull, ident, s->bvB,
                       (uint32_t *)s->valB, (uint32_t *)s->mprop, s->AL, bound ? &s->cnt->fmin : nullptr);
  };
  if (narrow_groups(g->ctx, nwS)) send(k_bcast<uint32_t, kGroupNarrow>, kGroupNarrow);
  else send(k_bcast<uint32_t, kGroupWide>, kGroupWide);
  const uint32_t nwP = g->P / 64;
  uint32_t inc = 0;  // the smallest Op::edge increment over an arc
  if (bound && s->algo == GRD_SSSP) {
    if (!s->prm.weighted) inc = 1;
    else GRD_TRY(graph_min_weight(g, &inc));
  }
  if (rows_done && nwP)
    hipLaunchKernelGGL(k_rows_done, dim3(loop_grid(g->ctx, nwP)), dim3(kBlock), 0, st, nwP, g->proxy_slot,
                       (const uint32_t *)s->prop, s->cnt, inc, s->Rdone);
  GRD_HIP(hipGetLastError());
  s->rdone_sent = rows_done;
  s->bound_sent = bound;
  s->bound_at = grd_state::kBoundOnDevice;
  s->bound_inc = inc;
  // exchange bytes (GraphAlgorithm.cpp:251-265): bitvector of every pair +
  // packed values (sparse) or the pair's full own slice (dense), and the
  // rows-done bitmap of a CC / SSSP pull
  uint64_t vals = dense ? (uint64_t)g->n : s->last_frontier;
  s->bytes += bitvector_bytes(g) + vals * s->vbytes + (rows_done ? 8ull * nwP : 0ull);
  return GRD_OK;
}

template <class Op>
static grd_status traverse_t(grd_state *s, int option)
{
  grd_graph *g = s->g;
  hipStream_t st = g->ctx->stream;
  const uint32_t *cwt = std::is_same<Op, OpWeighted>::value ? g->cw : nullptr;
  const bool timed = s->prm.time_kernel != 0;
  if (option & 1) {
    if (timed) GRD_HIP(hipEventRecord(s->kev[0], st));
    GRD_TRY(bsp_pull_launch<Op>(s, cwt));
    if (timed) {
      GRD_HIP(hipEventRecord(s->kev[1], st));
      s->kern_pending = 1;
      // a column and a gathered value per arc, the weight as stored (one
      // byte in the hot / cold split when every weight fits), a value per
      // row, and the rows-done bitmap; the arcs and rows of the blocks left
      // out come off when the counters are read
      const uint64_t wb = !cwt ? 0 : (bsp_hot_cold(s) && g->w8_fits) ? 1 : 4;
      s->kern_pending_bytes = (8 + wb) * g->m + 8ull * g->P + (s->rdone_sent ? g->P / 8 : 0);
      s->skip_arc_bytes = 8 + wb;
    }
    GRD_TRY(bsp_pull_fixup<Op>(s));
    // exact gather count (outside the events; time_kernel 2 leaves it out)
    if (timed && s->skip_pending && s->prm.time_kernel != 2) GRD_TRY(pull_done_arcs(s));
    s->edges += g->m;  // every arc of the memory partitions, less those left out (counters)
  } else {
    if (timed) GRD_HIP(hipEventRecord(s->kev[0], st));
    GRD_TRY(push_launch<Op>(s));
    if (timed) {
      GRD_HIP(hipEventRecord(s->kev[1], st));
      s->kern_pending = 2;  // bytes from the active list's vertices and arcs
    }
  }
  GRD_HIP(hipGetLastError());
  return GRD_OK;
}

grd_status op_traverse(grd_state *s, int option)
{
  s->cnt_clean = false;
  switch (s->algo) {
  case GRD_PR: return traverse_t<OpPR>(s, option);
  case GRD_CC: return traverse_t<OpCC>(s, option);
  case GRD_SSSP: return s->prm.weighted ? traverse_t<OpWeighted>(s, option) : traverse_t<OpHop>(s, option);
  default: return fail(GRD_ERR_STATE, "traverse: algorithm has no BSP traversal");
  }
}

template <class Op>
static grd_status reduce_t(grd_state *s, int option)
{
  grd_graph *g = s->g;
  hipStream_t st = g->ctx->stream;
  using V = typename Op::V;
  const uint32_t nwP = g->P / 64;
  const bool dense = option & 2;
  s->xr_dense = dense ? 1 : 0;
  if (!dense) GRD_TRY(word_ranks(st, s->Du, nwP, s->blk, s->wrankR, s->totals + 1));
  const auto send = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(s->n_rshare), dim3(kBlock), 0, st, nwP, s->Du, (V *)s->mupd,
                       s->wrankR, g->proxy_slot, (int)dense, s->bvR, (V *)s->valR, (V *)s->upd, s->Dc, s->rshare);
  };
  if (narrow_groups(g->ctx, nwP)) send(k_reduce<Op, kGroupNarrow>);
  else if (!Op::kMin || !dense) send(k_reduce<Op, kGroupWide>);
  else
    hipLaunchKernelGGL(k_reduce_min<uint32_t>, dim3(s->n_rshare), dim3(kBlock), 0, st, nwP, s->Du, s->bvR, g->S / 64,
                       g->word_dst, g->xptr, g->xlist, (const uint32_t *)s->mupd, (uint32_t *)s->valR,
                       (uint32_t *)s->upd, s->Dc, s->rshare);
  GRD_HIP(hipGetLastError());
  return GRD_OK;
}

grd_status op_reduce(grd_state *s, int option)
{
  s->cnt_clean = false;
  switch (s->algo) {
  case GRD_PR: return reduce_t<OpPR>(s, option);
  case GRD_CC: return reduce_t<OpCC>(s, option);
  case GRD_SSSP: return reduce_t<OpHop>(s, option);  // combine = min for both SSSP forms
  default: return fail(GRD_ERR_STATE, "reduce: algorithm has no BSP exchange");
  }
}

template <int ALGO>
static void launch_update(grd_state *s, int use_delta)
{
  grd_graph *g = s->g;
  const uint32_t nwS = g->S / 64;
  const auto go = [&](auto kernel, uint32_t kg) {
    hipLaunchKernelGGL(kernel, dim3(loop_grid(g->ctx, nwS, kg)), dim3(kBlock), 0, g->ctx->stream, nwS, s->Dc, s->prop,
                       s->upd, s->pr, g->slot_deg, s->F, s->Pend, (unsigned long long)s->hi, use_delta, s->ushare);
    s->n_ushare = loop_grid(g->ctx, nwS, kg);
  };
  if (narrow_groups(g->ctx, nwS)) go(k_update<ALGO, kGroupNarrow>, kGroupNarrow);
  else go(k_update<ALGO, kGroupWide>, kGroupWide);
}

grd_status op_update(grd_state *s)
{
  grd_graph *g = s->g;
  s->cnt_clean = false;
  s->bcast_stale = true;
  switch (s->algo) {
  case GRD_PR: launch_update<GRD_PR>(s, 0); break;
  case GRD_CC: launch_update<GRD_CC>(s, 0); break;
  case GRD_SSSP: launch_update<GRD_SSSP>(s, s->prm.delta ? 1 : 0); break;
  default: return fail(GRD_ERR_STATE, "update: algorithm has no BSP update");
  }
  GRD_HIP(hipGetLastError());
  if (g->C > 1) GRD_TRY(op_frontier_parts(s));
  return GRD_OK;
}

void take_frontier_parts(grd_state *s)
{
  if (s->g->C == 1) {
    s->last_fpart[0] = s->last_frontier;
    s->last_uncovered = 0;
    return;
  }
  for (int c = 0; c < s->g->C; c++) s->last_fpart[c] = s->hcnt->fpart[c];
  s->last_uncovered = s->hcnt->frontier_uncovered;
}

// Delta-stepping bucket advance when the frontier came out empty.  Reads the
// counters (synchronizes) and launches k_select.  *any_pending = frontier
// non-empty afterwards.
grd_status op_select_bucket(grd_state *s, bool *any_pending)
{
  grd_graph *g = s->g;
  hipStream_t st = g->ctx->stream;
  const uint32_t nwS = g->S / 64;
  const uint32_t grid = loop_grid(g->ctx, nwS);
  *any_pending = false;
  hipLaunchKernelGGL(k_pend_min<kGroupWide>, dim3(grid), dim3(kBlock), 0, st, nwS, s->Pend, (const uint32_t *)s->prop, s->cnt);
  GRD_HIP(hipGetLastError());
  GRD_TRY(op_read_counters(s));
  if (s->hcnt->pending == 0) return GRD_OK;
  uint64_t mn = s->hcnt->pend_min, d = s->prm.delta;
  s->hi = (mn / d + 1) * d;
  hipLaunchKernelGGL(k_select<kGroupWide>, dim3(grid), dim3(kBlock), 0, st, nwS, s->Pend, (const uint32_t *)s->prop, g->slot_deg,
                     (unsigned long long)s->hi, s->F, s->ushare);
  s->n_ushare = grid;
  GRD_HIP(hipGetLastError());
  if (g->C > 1) GRD_TRY(op_frontier_parts(s));
  GRD_TRY(op_read_counters(s));
  *any_pending = s->hcnt->frontier != 0;
  return GRD_OK;
}

grd_status op_aggregate_one(grd_state *s, uint32_t slot, const void *value)
{
  hipStream_t st = s->g->ctx->stream;
  if (s->algo == GRD_PR) {
    float x;
    memcpy(&x, value, 4);
    hipLaunchKernelGGL(k_aggregate_one<OpPR>, dim3(1), dim3(64), 0, st, (float *)s->upd, s->Dc, slot, x);
  } else {
    uint32_t x;
    memcpy(&x, value, 4);
    hipLaunchKernelGGL(k_aggregate_one<OpCC>, dim3(1), dim3(64), 0, st, (uint32_t *)s->upd, s->Dc, slot, x);
  }
  GRD_HIP(hipGetLastError());
  return GRD_OK;
}

grd_status op_download(grd_state *s, void *out)
{
  grd_graph *g = s->g;
  hipStream_t st = g->ctx->stream;
  const uint32_t *src = (s->algo == GRD_PR || s->algo == GRD_PR_PULL) ? (const uint32_t *)s->pr : (const uint32_t *)s->prop;
  // 8-byte properties are widened on the way, the unreached 2^32 - 1 to 2^64 - 1
  // (numeric_limits<uint64_t>::max)
  if (g->n <= kSmallOut) return copy_out_slots(g->ctx, out, src, g->slot_gid, g->S, g->n, s->wide);
  DevMem tmp(g->ctx);
  uint32_t *dout = nullptr;
  GRD_TRY(tmp.alloc_n(&dout, g->n));
  hipLaunchKernelGGL(k_gather_result<uint32_t>, dim3(std::min<uint32_t>(4096, g->S / kBlock + 1)), dim3(kBlock), 0, st,
                     g->S, g->slot_gid, src, dout);
  GRD_HIP(hipGetLastError());
  return copy_out(g->ctx, out, dout, g->n, s->wide);
}

}  // namespace grd
