// cold.hip -- the cold pass of the hot / cold pull: the arcs outside each
// partition's LDS window, gathered in source order.
//
// The rows (one per memory proxy) are cut into blocks of at most N arcs
// (cold_set).  The arcs of a block are kept sorted by source, each with the
// 16-bit place its value has in the block's row order (cpos).  A workgroup
// takes one block:
//   1. stage: the threads walk the block's arcs in source order, gather the
//      values and store each at its place in LDS, so that LDS holds the
//      block's values in row order;
//   2. reduce: groups of G lanes reduce the rows from LDS, each row's hot
//      partial first.
//
// Why sorted: the pass is bound by the rate at which the L2 serves gather
// requests (about 175 G/s on random 4-byte loads, whatever the bytes), and
// neighbouring lanes that fall into one 128-byte line make one request.  Sources are numbered in
// degree order, so the sources of 16384 cold arcs repeat the same lines often
// (RMAT-25, M = 4: 0.66 lines per arc, 0.90 in blocks of 2048).  Pull PageRank
// over RMAT-25: requests to the L2 307 M -> 230 M a pass, 1.93 -> 1.67 ms; what
// is left is the L2's misses (84 M lines, 6.4 TB/s from the fabric): every XCD
// draws the partition's 33 MB of values through its own 4 MB.  Loads that go
// past the L1 measured the same, nontemporal ones 1.7 times slower.
#include <algorithm>

#include "grd_device.hpp"
#include "grd_internal.hpp"
#include "grd_ops.hpp"
#include "grd_rows.hpp"

namespace grd {

namespace {

template <int T, int N>
__global__ void __launch_bounds__(T, 8) k_prp_pull_cold(const PullBlock *__restrict__ blocks,
                                                        const uint32_t *__restrict__ rptr,
                                                        const uint32_t *__restrict__ col,
                                                        const uint16_t *__restrict__ pos,
                                                        const float *__restrict__ mprop, float *__restrict__ out,
                                                        float2 *__restrict__ partial, const float *__restrict__ pre)
{
  __shared__ float s_v[N];
  const PullBlock d = blocks[blockIdx.x];
  const uint32_t ne = d.e1 - d.e0;
  const uint32_t G = row_group<T>(d.nrows), ngroups = T / G;
  const uint32_t rounds = (d.nrows + ngroups - 1) / ngroups, r1 = d.r0 + d.nrows;
  // the first round's rows are loaded with the columns
  uint32_t r = d.r0 + threadIdx.x / G, b = 0, e = 0;
  float hot = 0.0f;
  auto row = [&]() {
    b = e = 0;
    if (r < r1) {
      b = rptr[r] - d.e0;
      e = rptr[r + 1] - d.e0;
      hot = pre[r];
    }
  };
  row();
  for (uint32_t i0 = threadIdx.x; i0 < ne; i0 += kBatch * T) {
    uint32_t c[kBatch], p[kBatch];
    float v[kBatch];
#pragma unroll
    for (int k = 0; k < kBatch; k++) {
      const uint32_t i = i0 + k * T;
      c[k] = i < ne ? col[d.e0 + i] : col[d.e0 + i0];
      p[k] = i < ne ? pos[d.e0 + i] : pos[d.e0 + i0];
    }
#pragma unroll
    for (int k = 0; k < kBatch; k++) v[k] = mprop[c[k]];
    // (a thread's arcs past the end repeat its first one)
#pragma unroll
    for (int k = 0; k < kBatch; k++) s_v[p[k]] = v[k];
  }
  __syncthreads();
  if (d.nrows == 0) {
    const Kahan t = segment_sum<HotPR, T>(s_v, ne);
    if (threadIdx.x == 0) partial[blockIdx.x] = make_float2(t.s, t.c);
    return;
  }
  for (uint32_t k = 0; k < rounds; k++) {  // the same rounds for every group: the shuffles stay in step
    const uint32_t rn = r, bn = b, en = e;
    const float hn = hot;
    r += ngroups;
    row();  // the next round's rows are in flight during this one's sums
    const Kahan acc = row_sum<HotPR>(s_v, bn, en, G);
    if (threadIdx.x % G == 0 && rn < r1) {
      Kahan t;
      t.s = hn;  // the row's hot partial comes first
      t.merge(acc.s, acc.c);
      out[rn] = t.value();
    }
  }
}

// CC / SSSP / reference PageRank.  flag (skip): 1 = the block is left out, 2 =
// some of its rows are done.  bcnt: a row whose hot partial is already at or
// below the bound takes no cold candidate below it (every cold candidate is at
// least the bound), so it gathers nothing and its result is the hot partial.
template <class Op, class W, int T, int N>
__global__ void __launch_bounds__(T, 8) k_bsp_pull_cold(const PullBlock *__restrict__ blocks,
                                                        const uint32_t *__restrict__ rptr,
                                                        const uint32_t *__restrict__ col,
                                                        const uint16_t *__restrict__ pos, const W *__restrict__ cw,
                                                        const typename Op::V *__restrict__ mprop,
                                                        typename Op::V *__restrict__ upd, uint64_t *__restrict__ dirty,
                                                        typename Op::V *__restrict__ partial,
                                                        const typename Op::V *__restrict__ pre,
                                                        const uint8_t *__restrict__ skip,
                                                        const uint64_t *__restrict__ done,
                                                        const uint64_t *__restrict__ hasarc,
                                                        const Counters *__restrict__ bcnt, uint32_t inc)
{
  using V = typename Op::V;
  using Pol = HotBsp<Op>;
  __shared__ V s_v[N];
  __shared__ unsigned long long s_dirty[kColdRows / 64 + 2];
  const PullBlock d = blocks[blockIdx.x];
  const uint32_t flag = skip ? skip[blockIdx.x] : 0u;
  if (flag == 1) return;
  const uint32_t ne = d.e1 - d.e0;
  const uint32_t bnd = bcnt ? pull_bound(bcnt, inc) : 0u;
  if (d.nrows == 0 && bcnt && pre[d.r0] <= bnd) {  // a segment of a row that gathers nothing
    if (threadIdx.x == 0) partial[blockIdx.x] = op_identity<Op>();
    return;
  }
  const uint32_t G = row_group<T>(d.nrows), ngroups = T / G, sub = threadIdx.x % G;
  const uint32_t rounds = (d.nrows + ngroups - 1) / ngroups, r1 = d.r0 + d.nrows;
  const uint32_t w0 = d.r0 >> 6;
  for (uint32_t i = threadIdx.x; i < d.nrows / 64 + 2; i += T) s_dirty[i] = 0ull;
  // a done row, or one without arcs, has nothing to apply (its hot partial may
  // not have been written)
  auto live_row = [&](uint32_t q) {
    if (!done) return true;
    const uint64_t bit = 1ull << (q & 63);
    return !(done[q >> 6] & bit) && (hasarc[q >> 6] & bit);
  };
  const bool marked = d.nrows != 0 && (flag == 2 || bcnt);  // uniform over the block
  if (marked) {
    // every place of the block is marked first: the identity where the row
    // gathers nothing, 0 where the arc's value is wanted
    for (uint32_t k = 0; k < rounds; k++) {
      const uint32_t q = d.r0 + k * ngroups + threadIdx.x / G;
      bool gat = false;
      uint32_t b = 0, e = 0;
      if (q < r1) {
        gat = live_row(q);
        if (gat && bcnt) gat = pre[q] > bnd;
        b = rptr[q] - d.e0;
        e = rptr[q + 1] - d.e0;
      }
      row_fill(s_v, b, e, G, gat ? V(0) : op_identity<Op>());
    }
    __syncthreads();
  }
  for (uint32_t i0 = threadIdx.x; i0 < ne; i0 += kBatch * T) {
    uint32_t c[kBatch], p[kBatch], w[kBatch];
    bool on[kBatch];
#pragma unroll
    for (int k = 0; k < kBatch; k++) {
      const uint32_t i = i0 + k * T;
      on[k] = i < ne;
      c[k] = on[k] ? col[d.e0 + i] : 0u;
      p[k] = on[k] ? pos[d.e0 + i] : 0u;
      w[k] = 1u;
      if constexpr (Pol::kWeighted)
        if (on[k]) w[k] = (uint32_t)cw[d.e0 + i];
    }
    if (marked) {
#pragma unroll
      for (int k = 0; k < kBatch; k++) on[k] = on[k] && s_v[p[k]] == V(0);
    }
    V v[kBatch];
#pragma unroll
    for (int k = 0; k < kBatch; k++) v[k] = on[k] ? mprop[c[k]] : V(0);
#pragma unroll
    for (int k = 0; k < kBatch; k++)
      if (on[k]) s_v[p[k]] = Op::edge(v[k], w[k]);
  }
  __syncthreads();
  if (d.nrows == 0) {
    const V t = segment_sum<Pol, T>(s_v, ne);
    if (threadIdx.x == 0) partial[blockIdx.x] = t;
    return;
  }
  uint32_t r = d.r0 + threadIdx.x / G, b = 0, e = 0;
  bool live = false;
  V hot = op_identity<Op>();
  auto row = [&]() {
    b = e = 0;
    live = r < r1 && live_row(r);
    if (live) {
      b = rptr[r] - d.e0;
      e = rptr[r + 1] - d.e0;
      hot = pre[r];
    }
  };
  row();
  for (uint32_t k = 0; k < rounds; k++) {
    const uint32_t rn = r, bn = b, en = e;
    const bool ln = live;
    const V hn = hot;
    r += ngroups;
    row();
    const V acc = op_combine<Op>(hn, row_sum<Pol>(s_v, bn, en, G));  // the row's hot partial first
    if (sub == 0 && ln && pull_apply<Op>(upd, rn, acc)) atomicOr(&s_dirty[(rn >> 6) - w0], 1ull << (rn & 63));
  }
  __syncthreads();
  const uint32_t nw = ((r1 - 1) >> 6) - w0 + 1;
  for (uint32_t i = threadIdx.x; i < nw; i += T)
    if (s_dirty[i]) atomicOr((unsigned long long *)(dirty + w0 + i), s_dirty[i]);
}

// Flags of the row blocks of a CC / SSSP pull (the cold blocks, or those of the
// whole CSC): 1 = every row with arcs is done, 2 = some are; counts the arcs and
// rows left out.  A wave per block: a block spans up to kColdRows rows, 129 words
// of each bitmap, which a thread alone would walk one after another.
__global__ void __launch_bounds__(kBlock) k_row_blocks_done(uint32_t nblk, const PullBlock *__restrict__ blocks,
                                                             const uint64_t *__restrict__ done,
                                                             const uint64_t *__restrict__ hasarc,
                                                             uint8_t *__restrict__ bskip,
                                                             SkipShare *__restrict__ share, bool again)
{
  unsigned long long arcs = 0, rows = 0;
  const uint32_t lane = lane_id();
  for (uint32_t b = blockIdx.x * kWavesPerBlock + wave_in_block(); b < nblk; b += gridDim.x * kWavesPerBlock) {
    const PullBlock d = blocks[b];
    const uint32_t r1 = d.r0 + max(d.nrows, 1u);
    bool all = true, any = false;
    for (uint32_t w = (d.r0 >> 6) + lane; w <= (r1 - 1) >> 6; w += kWave) {
      const uint32_t lo = max(d.r0, w * 64) - w * 64, hi = min(r1 - w * 64, 64u);
      const uint64_t mask = (hi - lo == 64) ? ~0ull : (((1ull << (hi - lo)) - 1ull) << lo);
      const uint64_t dn = done[w], ha = hasarc[w];
      all = all && ((dn | ~ha) & mask) == mask;
      any = any || (dn & ha & mask) != 0;
    }
    all = __ballot(!all) == 0;
    any = __ballot(any) != 0;
    if (lane == 0) {
      bskip[b] = all ? 1 : any ? 2 : 0;
      if (all) {
        arcs += d.e1 - d.e0;
        rows += d.nrows;
      }
    }
  }
  arcs = block_sum(arcs);
  rows = block_sum(rows);
  if (threadIdx.x == 0) add_share(share + blockIdx.x, SkipShare{arcs, 0, rows}, again);
}

}  // namespace

// Cold set 0 serves the sums (pull and reference PageRank), 1 the min-combines
// (CC, SSSP).  While a partition's values fit an L2 (2^20 sources, 4 MB) small
// blocks are best for both: more of them in flight.  Beyond, the sums take
// 16384 arcs, two workgroups per CU (pull PageRank over RMAT-23: 9.2 ms a solve
// against 10.2 with 2048, RMAT-24 20.7 / 23.0, RMAT-25 46.3 / 53.2, RMAT-26
// 118 / 126; 32768 arcs leave one workgroup per CU, whose two steps then do
// not overlap: 50.2).  The min-combines leave out blocks and rows that cannot
// improve, which large blocks do worse: CC over RMAT-24 symmetrized 4.98 ms
// with 4096 arcs, 5.06 with 2048, 5.38 with 16384.
uint32_t cold_set(const grd_graph *g, int algo, uint32_t *nnz)
{
  uint32_t widest = 0;
  for (int m = 0; m < g->M; m++) {
    uint64_t own = 0;
    for (int c = 0; c < g->C; c++) own += g->ocnt[(size_t)m * g->C + c];
    widest = std::max<uint32_t>(widest, (uint32_t)own);
  }
  const bool sums = algo == GRD_PR || algo == GRD_PR_PULL, large = widest > (1u << 20);
  *nnz = !large ? 2048 : sums ? 16384 : 4096;
  return large && !sums ? 1 : 0;
}

#define COLD_SHAPES(nnz, F)            \
  switch (nnz) {                       \
  case 2048: F(256, 2048); break;      \
  case 4096: F(256, 4096); break;      \
  default: F(1024, 16384);             \
  }

grd_status cold_sort(grd_graph *g, const ColdSet &c)
{
  hipStream_t st = g->ctx->stream;
  if (!c.nblk) return GRD_OK;
  int bits = 1;
  while (bits < 31 && (g->P >> bits)) bits++;
#define F(T, N)                                                                                                     \
  if (c.w8)                                                                                                         \
    hipLaunchKernelGGL((k_block_sort<PullBlock, uint8_t, T, N>), dim3(c.nblk), dim3(T), 0, st, c.blk, c.col, c.w8, c.pos, bits); \
  else                                                                                                              \
    hipLaunchKernelGGL((k_block_sort<PullBlock, uint32_t, T, N>), dim3(c.nblk), dim3(T), 0, st, c.blk, c.col, c.w, c.pos, bits)
  COLD_SHAPES(c.nnz, F)
#undef F
  GRD_HIP(hipGetLastError());
  return GRD_OK;
}

grd_status prp_pull_cold(grd_state *s, float *out, const float *pre)
{
  grd_graph *g = s->g;
  const ColdSet &c = *s->cold;
  hipStream_t st = g->ctx->stream;
  if (!c.nblk) return GRD_OK;
#define F(T, N)                                                                                           \
  hipLaunchKernelGGL((k_prp_pull_cold<T, N>), dim3(c.nblk), dim3(T), 0, st, c.blk, g->corp, c.col, c.pos, \
                     (const float *)s->mprop, out, s->cseg, pre)
  COLD_SHAPES(c.nnz, F)
#undef F
  GRD_HIP(hipGetLastError());
  return GRD_OK;
}

template <class Op>
grd_status bsp_pull_cold(grd_state *s, const uint8_t *skip, const Counters *bcnt)
{
  grd_graph *g = s->g;
  const ColdSet &c = *s->cold;
  using V = typename Op::V;
  hipStream_t st = g->ctx->stream;
  if (!c.nblk) return GRD_OK;
  const uint64_t *done = skip ? (const uint64_t *)s->Rdone : nullptr, *ha = skip ? (const uint64_t *)g->rarc : nullptr;
#define L(W, w, T, N)                                                                                             \
  hipLaunchKernelGGL((k_bsp_pull_cold<Op, W, T, N>), dim3(c.nblk), dim3(T), 0, st, c.blk, g->corp, c.col, c.pos, \
                     (const W *)w, (const V *)s->mprop, (V *)s->mupd, s->Du, (V *)s->cseg, (const V *)s->tpart,  \
                     skip, done, ha, bcnt, s->bound_inc)
  if constexpr (std::is_same<Op, OpWeighted>::value) {
    if (c.w8) {
#define F(T, N) L(uint8_t, c.w8, T, N)
      COLD_SHAPES(c.nnz, F)
#undef F
      GRD_HIP(hipGetLastError());
      return GRD_OK;
    }
  }
#define F(T, N) L(uint32_t, c.w, T, N)
  COLD_SHAPES(c.nnz, F)
#undef F
#undef L
  GRD_HIP(hipGetLastError());
  return GRD_OK;
}
template grd_status bsp_pull_cold<OpCC>(grd_state *, const uint8_t *, const Counters *);
template grd_status bsp_pull_cold<OpHop>(grd_state *, const uint8_t *, const Counters *);
template grd_status bsp_pull_cold<OpWeighted>(grd_state *, const uint8_t *, const Counters *);
template grd_status bsp_pull_cold<OpPR>(grd_state *, const uint8_t *, const Counters *);

grd_status row_blocks_done(grd_state *s, uint32_t nblk, const PullBlock *blocks, bool again)
{
  grd_graph *g = s->g;
  if (nblk) {
    const uint32_t grid = std::min<uint32_t>((nblk + kWavesPerBlock - 1) / kWavesPerBlock, loop_blocks(g->ctx));
    hipLaunchKernelGGL(k_row_blocks_done, dim3(grid), dim3(kBlock), 0, g->ctx->stream, nblk, blocks,
                       (const uint64_t *)s->Rdone, (const uint64_t *)g->rarc, s->bskip, s->sshare + s->n_sshare, again);
    s->n_sshare += grid;
  }
  GRD_HIP(hipGetLastError());
  return GRD_OK;
}

}  // namespace grd
