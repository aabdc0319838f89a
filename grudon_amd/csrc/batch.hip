// batch.hip -- many graphs of uneven size processed by one persistent
// launch per phase, with the iterations captured in a hipGraph.
//
// The graphs' CSCs are concatenated (global vertex id = graph base + local
// id) and cut into row blocks of at most `tile` arcs or a multiple of it, each
// tagged with its graph and with its arcs in source order; rows longer than a
// block become segments merged in order by a fix-up pass.  A persistent grid
// of `grid_per_cu` x CUs workgroups walks the block list; blocks of graphs that
// have already converged are skipped, so a replay of the captured iterations
// does no work for finished graphs.
//
// PageRank (per graph, normalised pull, FP32 Kahan contributions, FP64
// dangling mass and L1 residual, converged when the L1 change < tolerance)
// and CC (per graph, synchronous min-label propagation over in-edges, the
// fixed point of src/graph_algorithms/cc.cpp) share the block structure.
//
// Tunables: tile (arcs of the smallest block), grid_per_cu
// (persistent workgroups per CU) and K (iterations per captured graph);
// grd_batch_autotune times candidate settings on the batch itself.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "grd_device.hpp"
#include "grd_internal.hpp"
#include "grd_ops.hpp"
#include "grd_rows.hpp"

namespace grd {

struct BatchBlock {
  uint32_t r0, nrows, e0, e1, graph, pad0, pad1, pad2;
};
struct BatchLong {
  uint32_t row, first, nseg, graph;
};

}  // namespace grd

struct grd_batch {
  grd_ctx *ctx = nullptr;
  uint32_t count = 0;
  uint64_t N = 0, E = 0;
  std::vector<uint64_t> vbase;  // [count+1]
  std::vector<uint32_t> h_crp;  // [N+1] concatenated CSC row pointers (global arc ids)
  std::vector<uint32_t> h_deg;  // [N] out-degree
  grd::DevMem mem;
  uint32_t *crp = nullptr, *ccol = nullptr, *deg = nullptr, *gid_local = nullptr;
  uint64_t *vb = nullptr;  // [count+1]
  // tunables
  uint32_t tile = 2048, grid_per_cu = 8, K = 4;
  // blocks for the current tile
  grd::DevMem blk_mem;
  grd::BatchBlock *blocks = nullptr;
  grd::BatchLong *longs = nullptr;
  uint32_t *scol = nullptr;   // [E] columns, each block's in source order
  uint16_t *spos = nullptr;   // [E] an arc's place in its block's row order
  uint32_t *gblk = nullptr;   // [count+1] first block of each graph
  uint32_t *glong = nullptr;  // [count+1] first long row of each graph
  double *tred = nullptr;     // [2 * nblk] (residual, dangling mass) of each block
  double *lred = nullptr;     // [2 * nlong] and of each long row
  uint32_t nblk = 0, nlong = 0, nnz = 0;
  // the captured iterations, kept while what is baked into them stays the same
  struct Captured {
    hipGraphExec_t exec = nullptr;
    double damping = 0.0, tol = 0.0;
    uint32_t max_iter = 0, K = 0, grid = 0;
  } pr_graph, cc_graph;
  // per-graph state
  grd::DevMem st_mem;
  float *r = nullptr, *contrib[2] = {nullptr, nullptr};
  float2 *partial = nullptr;
  uint32_t *lab[2] = {nullptr, nullptr};
  uint32_t *active = nullptr, *iters = nullptr, *changed = nullptr, *alive = nullptr;
  double *residual = nullptr, *dcur = nullptr;
  std::vector<double> d0;       // initial dangling mass of each graph
  uint32_t *seq = nullptr;      // device: replays so far
  uint32_t *h_alive = nullptr;  // pinned: graphs still running, replays so far
  uint32_t h_seq = 0;
  int last_algo = -1;
  std::vector<uint32_t> last_iters;
};

namespace grd {

// ------------------------------------------------------------------------
// PageRank
// ------------------------------------------------------------------------

// Pull and update in one pass.  A workgroup takes a block, gathers its arcs'
// values in source order and stores each at its place in the block's row order
// in LDS; groups of G lanes sum the rows (grd_rows.hpp), and the row's first
// lane turns the sum into the vertex's new rank and its next contribution
// (other blocks still gather the present ones: the contributions alternate
// between two arrays).  The block's residual and dangling mass go to its own
// FP64 slots, so convergence does not depend on scheduling.
template <int T, int N>
__global__ void __launch_bounds__(T) k_bpr_pull(const BatchBlock *__restrict__ blocks, uint32_t nblk,
                                                const uint32_t *__restrict__ crp, const uint32_t *__restrict__ col,
                                                const uint16_t *__restrict__ pos, const float *__restrict__ cin,
                                                float *__restrict__ cout, float *__restrict__ r,
                                                const uint32_t *__restrict__ deg, const uint64_t *__restrict__ vb,
                                                const double *__restrict__ dcur, float damping,
                                                float2 *__restrict__ partial, double *__restrict__ tred,
                                                const uint32_t *__restrict__ active)
{
  __shared__ float s_v[N];
  __shared__ double s_red[T / kWave][2];
  for (uint32_t b = blockIdx.x; b < nblk; b += gridDim.x) {
    const BatchBlock d = blocks[b];
    if (!active[d.graph]) continue;  // uniform over the workgroup
    const uint32_t ne = d.e1 - d.e0;
    const uint32_t G = row_group<T>(d.nrows), ngroups = T / G;
    const uint32_t rounds = (d.nrows + ngroups - 1) / ngroups, v1 = d.r0 + d.nrows;
    uint32_t v = d.r0 + threadIdx.x / G, lo = 0, hi = 0, dg = 0;
    float old = 0.0f;
    auto row = [&]() {
      lo = hi = 0;
      if (v < v1) {
        lo = crp[v] - d.e0;
        hi = crp[v + 1] - d.e0;
        old = r[v];
        dg = deg[v];
      }
    };
    row();  // the first round's rows are loaded with the columns
    for (uint32_t i0 = threadIdx.x; i0 < ne; i0 += kBatch * T) {
      uint32_t c[kBatch], p[kBatch];
      float x[kBatch];
#pragma unroll
      for (int k = 0; k < kBatch; k++) {
        const uint32_t i = i0 + k * T;  // (a thread's arcs past the end repeat its first one)
        c[k] = i < ne ? col[d.e0 + i] : col[d.e0 + i0];
        p[k] = i < ne ? pos[d.e0 + i] : pos[d.e0 + i0];
      }
#pragma unroll
      for (int k = 0; k < kBatch; k++) x[k] = cin[c[k]];
#pragma unroll
      for (int k = 0; k < kBatch; k++) s_v[p[k]] = x[k];
    }
    __syncthreads();
    if (d.nrows == 0) {
      const Kahan t = segment_sum<HotPR, T>(s_v, ne);
      if (threadIdx.x == 0) {
        partial[b] = make_float2(t.s, t.c);
        tred[2 * b] = tred[2 * b + 1] = 0.0;
      }
      __syncthreads();
      continue;
    }
    const double n = (double)(vb[d.graph + 1] - vb[d.graph]);
    const float base = (float)((1.0 - (double)damping) / n + (double)damping * dcur[d.graph] / n);
    double res = 0.0, dang = 0.0;
    for (uint32_t k = 0; k < rounds; k++) {
      const uint32_t vn = v, ln = lo, hn = hi, dn = dg;
      const float on = old;
      v += ngroups;
      row();  // the next round's rows are in flight during this one's sums
      const Kahan a = row_sum<HotPR>(s_v, ln, hn, G);
      if (threadIdx.x % G == 0 && vn < v1) {
        const float rn = base + damping * a.value();
        res += fabs((double)rn - (double)on);
        if (dn == 0) dang += (double)rn;
        r[vn] = rn;
        cout[vn] = dn ? rn / (float)dn : 0.0f;
      }
    }
    res = wave_sum(res);
    dang = wave_sum(dang);
    if (lane_id() == 0) {
      s_red[wave_in_block()][0] = res;
      s_red[wave_in_block()][1] = dang;
    }
    __syncthreads();  // (also: the staged values have been read)
    if (threadIdx.x < 2) {
      double t = 0.0;
      for (int j = 0; j < T / kWave; j++) t += s_red[j][threadIdx.x];
      tred[2 * b + threadIdx.x] = t;
    }
  }
}

// rows longer than a block: a wave each merges the segments and updates the vertex
__global__ void __launch_bounds__(kBlock) k_bpr_fixup(const BatchLong *__restrict__ longs, uint32_t nlong,
                                                      const float2 *__restrict__ partial, float *__restrict__ cout,
                                                      float *__restrict__ r, const uint32_t *__restrict__ deg,
                                                      const uint64_t *__restrict__ vb, const double *__restrict__ dcur,
                                                      float damping, double *__restrict__ lred,
                                                      const uint32_t *__restrict__ active)
{
  const uint32_t lane = lane_id();
  for (uint32_t i = blockIdx.x * kWavesPerBlock + wave_in_block(); i < nlong; i += gridDim.x * kWavesPerBlock) {
    const BatchLong L = longs[i];
    if (!active[L.graph]) continue;
    Kahan t;
    for (uint32_t j = lane; j < L.nseg; j += kWave) {
      const float2 p = partial[L.first + j];
      t.merge(p.x, p.y);
    }
    kahan_wave_merge(t, kWave);
    if (lane == 0) {
      const double n = (double)(vb[L.graph + 1] - vb[L.graph]);
      const float base = (float)((1.0 - (double)damping) / n + (double)damping * dcur[L.graph] / n);
      const float rn = base + damping * t.value();
      const uint32_t dg = deg[L.row];
      lred[2 * i] = fabs((double)rn - (double)r[L.row]);
      lred[2 * i + 1] = dg == 0 ? (double)rn : 0.0;
      r[L.row] = rn;
      cout[L.row] = dg ? rn / (float)dg : 0.0f;
    }
  }
}

// a wave per graph: its blocks' and long rows' sums in a fixed order, the
// convergence test, the next dangling mass
__global__ void __launch_bounds__(kBlock) k_bpr_finish(uint32_t count, uint32_t *active, uint32_t *iters,
                                                       const uint32_t *__restrict__ gblk,
                                                       const uint32_t *__restrict__ glong,
                                                       const double *__restrict__ tred, const double *__restrict__ lred,
                                                       double *residual, double *dcur, double tolerance,
                                                       uint32_t max_iter, uint32_t *alive)
{
  const uint32_t lane = lane_id();
  for (uint32_t g = blockIdx.x * kWavesPerBlock + wave_in_block(); g < count; g += gridDim.x * kWavesPerBlock) {
    if (!active[g]) continue;
    double res = 0.0, dang = 0.0;
    for (uint32_t t = gblk[g] + lane; t < gblk[g + 1]; t += kWave) {
      res += tred[2 * t];
      dang += tred[2 * t + 1];
    }
    for (uint32_t t = glong[g] + lane; t < glong[g + 1]; t += kWave) {
      res += lred[2 * t];
      dang += lred[2 * t + 1];
    }
    res = wave_sum(res);
    dang = wave_sum(dang);
    if (lane == 0) {
      const uint32_t it = ++iters[g];
      residual[g] = res;
      if (res < tolerance || it >= max_iter) active[g] = 0;
      else atomicAdd(alive, 1u);
      dcur[g] = dang;
    }
  }
}

__global__ void __launch_bounds__(kBlock) k_bpr_init(uint64_t N, const uint64_t *__restrict__ vb, uint32_t count,
                                                     const uint32_t *__restrict__ gidx, const uint32_t *__restrict__ deg,
                                                     float *r, float *contrib)
{
  for (uint64_t v = blockIdx.x * (uint64_t)kBlock + threadIdx.x; v < N; v += (uint64_t)gridDim.x * kBlock) {
    uint32_t g = gidx[v];
    float r0 = (float)(1.0 / (double)(vb[g + 1] - vb[g]));
    r[v] = r0;
    contrib[v] = deg[v] ? r0 / (float)deg[v] : 0.0f;
  }
}

// ------------------------------------------------------------------------
// CC (synchronous min-label propagation over in-edges)
// ------------------------------------------------------------------------

template <int T, int N>
__global__ void __launch_bounds__(T) k_bcc_pull(const BatchBlock *__restrict__ blocks, uint32_t nblk,
                                                const uint32_t *__restrict__ crp, const uint32_t *__restrict__ col,
                                                const uint16_t *__restrict__ pos, const uint32_t *__restrict__ lin,
                                                uint32_t *__restrict__ lout, uint32_t *__restrict__ partial,
                                                const uint32_t *__restrict__ active, uint32_t *changed)
{
  using Pol = HotBsp<OpCC>;
  __shared__ uint32_t s_v[N];
  for (uint32_t b = blockIdx.x; b < nblk; b += gridDim.x) {
    const BatchBlock d = blocks[b];
    if (!active[d.graph]) continue;
    const uint32_t ne = d.e1 - d.e0;
    const uint32_t G = row_group<T>(d.nrows), ngroups = T / G;
    const uint32_t rounds = (d.nrows + ngroups - 1) / ngroups, v1 = d.r0 + d.nrows;
    uint32_t v = d.r0 + threadIdx.x / G, lo = 0, hi = 0, old = 0;
    auto row = [&]() {
      lo = hi = 0;
      if (v < v1) {
        lo = crp[v] - d.e0;
        hi = crp[v + 1] - d.e0;
        old = lin[v];
      }
    };
    row();
    for (uint32_t i0 = threadIdx.x; i0 < ne; i0 += kBatch * T) {
      uint32_t c[kBatch], p[kBatch], x[kBatch];
#pragma unroll
      for (int k = 0; k < kBatch; k++) {
        const uint32_t i = i0 + k * T;
        c[k] = i < ne ? col[d.e0 + i] : col[d.e0 + i0];
        p[k] = i < ne ? pos[d.e0 + i] : pos[d.e0 + i0];
      }
#pragma unroll
      for (int k = 0; k < kBatch; k++) x[k] = lin[c[k]];
#pragma unroll
      for (int k = 0; k < kBatch; k++) s_v[p[k]] = x[k];
    }
    __syncthreads();
    if (d.nrows == 0) {
      const uint32_t t = segment_sum<Pol, T>(s_v, ne);
      if (threadIdx.x == 0) partial[b] = t;
      __syncthreads();
      continue;
    }
    bool any = false;
    for (uint32_t k = 0; k < rounds; k++) {
      const uint32_t vn = v, ln = lo, hn = hi, on = old;
      v += ngroups;
      row();
      const uint32_t m = row_sum<Pol>(s_v, ln, hn, G);
      if (threadIdx.x % G == 0 && vn < v1) {
        lout[vn] = min(on, m);
        any = any || m < on;
      }
    }
    if (__syncthreads_or(any) && threadIdx.x == 0) changed[d.graph] = 1;
  }
}

__global__ void __launch_bounds__(kBlock) k_bcc_fixup(const BatchLong *__restrict__ longs, uint32_t nlong,
                                                      const uint32_t *__restrict__ partial,
                                                      const uint32_t *__restrict__ lin, uint32_t *__restrict__ lout,
                                                      const uint32_t *__restrict__ active, uint32_t *changed)
{
  const uint32_t lane = lane_id();
  for (uint32_t i = blockIdx.x * kWavesPerBlock + wave_in_block(); i < nlong; i += gridDim.x * kWavesPerBlock) {
    const BatchLong L = longs[i];
    if (!active[L.graph]) continue;
    uint32_t m = 0xFFFFFFFFu;
    for (uint32_t j = lane; j < L.nseg; j += kWave) m = min(m, partial[L.first + j]);
    m = wave_min(m);
    if (lane == 0) {
      const uint32_t old = lin[L.row];
      lout[L.row] = min(old, m);
      if (m < old) changed[L.graph] = 1;
    }
  }
}

__global__ void k_bcc_finish(uint32_t count, uint32_t *active, uint32_t *iters, uint32_t *changed, uint32_t max_iter,
                             uint32_t *alive)
{
  for (uint32_t g = blockIdx.x * blockDim.x + threadIdx.x; g < count; g += gridDim.x * blockDim.x) {
    if (!active[g]) continue;
    uint32_t it = ++iters[g];
    if (!changed[g] || it >= max_iter) active[g] = 0;
    else atomicAdd(alive, 1u);
    changed[g] = 0;
  }
}

__global__ void __launch_bounds__(kBlock) k_bcc_init(uint64_t N, const uint32_t *__restrict__ local, uint32_t *l0,
                                                     uint32_t *l1)
{
  for (uint64_t v = blockIdx.x * (uint64_t)kBlock + threadIdx.x; v < N; v += (uint64_t)gridDim.x * kBlock) {
    l0[v] = local[v];
    l1[v] = local[v];
  }
}

// the end of a replay: the number of graphs still running and the replay's
// number into pinned memory, and the count to its start for the next replay
__global__ void __launch_bounds__(kWave) k_balive(uint32_t *alive, uint32_t *seq, uint32_t *host)
{
  if (threadIdx.x == 0) {
    host[0] = *alive;
    *alive = 0;
    const uint32_t n = *seq + 1;
    *seq = n;
    __hip_atomic_store(host + 1, n, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

__global__ void k_bfill_u32(uint32_t *p, uint32_t n, uint32_t v)
{
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = v;
}
__global__ void k_bfill_f64(double *p, uint32_t n, double v)
{
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = v;
}

// ------------------------------------------------------------------------
// host side
// ------------------------------------------------------------------------

// shapes of the pulls by arcs per block
#define BATCH_SHAPES(nnz, F)         \
  switch (nnz) {                     \
  case 1024: F(256, 1024); break;    \
  case 2048: F(256, 2048); break;    \
  case 4096: F(256, 4096); break;    \
  case 8192: F(512, 8192); break;    \
  default: F(1024, 16384);           \
  }

static void drop_captured(grd_batch *b)
{
  for (auto *c : {&b->pr_graph, &b->cc_graph}) {
    if (c->exec) (void)hipGraphExecDestroy(c->exec);
    c->exec = nullptr;
  }
}

// Blocks of `tile` to 16384 arcs: the largest that still gives every CU two.
// The larger a block, the more of its arcs share a source's line with a
// neighbour in source order (a graph of 100 K vertices has 3 K lines).
//
// What bounds an iteration (24 RMAT graphs, 58 M arcs in all, blocks of 16384):
// the gathers' lines, then the LDS.  Of 207 us (280 G arcs/s), with the parts
// left out in turn: streaming columns and places 46 us (348 MB), the scattered
// LDS stores 33, the gathers 89, the row sums and updates 39.  The whole
// PageRank took 4.36 ms with the arcs in row order, a separate update pass and
// blocks of 1024, and takes 2.72; CC took 1.70 and takes 1.41.
static uint32_t block_arcs(const grd_batch *b, uint32_t tile)
{
  while (tile < 16384 && b->E / (2 * tile) >= 2ull * (uint64_t)b->ctx->num_cus) tile *= 2;
  return tile;
}

static grd_status cut_blocks(grd_batch *b)
{
  std::vector<BatchBlock> blks;
  std::vector<BatchLong> longs;
  std::vector<uint32_t> gblk(b->count + 1, 0), glong(b->count + 1, 0);
  const uint32_t T = block_arcs(b, b->tile);
  const uint32_t rows = std::min<uint32_t>(T, 8192);
  for (uint32_t g = 0; g < b->count; g++) {
    gblk[g] = (uint32_t)blks.size();
    glong[g] = (uint32_t)longs.size();
    const uint64_t v0 = b->vbase[g], v1 = b->vbase[g + 1];
    uint64_t r = v0;
    while (r < v1) {
      uint32_t deg = b->h_crp[r + 1] - b->h_crp[r];
      if (deg > T) {
        BatchLong L{(uint32_t)r, (uint32_t)blks.size(), 0, g};
        L.nseg = cut_long_row(b->h_crp[r], b->h_crp[r + 1], T, [&blks, r, g](uint32_t x, uint32_t y) {
          blks.push_back(BatchBlock{(uint32_t)r, 0, x, y, g, 0, 0, 0});
        });
        longs.push_back(L);
        r++;
        continue;
      }
      const uint64_t rs = r;
      const uint32_t e0 = b->h_crp[r];
      while (r < v1 && r - rs < rows && b->h_crp[r + 1] - b->h_crp[r] <= T && b->h_crp[r + 1] - e0 <= T) r++;
      blks.push_back(BatchBlock{(uint32_t)rs, (uint32_t)(r - rs), e0, b->h_crp[r], g, 0, 0, 0});
    }
  }
  gblk[b->count] = (uint32_t)blks.size();
  glong[b->count] = (uint32_t)longs.size();
  drop_captured(b);  // (they hold the old blocks' addresses)
  b->blk_mem.release();
  b->nblk = (uint32_t)blks.size();
  b->nlong = (uint32_t)longs.size();
  b->nnz = T;
  if (longs.empty()) longs.push_back(BatchLong{0, 0, 0, 0});
  hipStream_t st = b->ctx->stream;
  GRD_TRY(b->blk_mem.alloc_n(&b->blocks, std::max<size_t>(1, blks.size())));
  GRD_TRY(b->blk_mem.alloc_n(&b->longs, longs.size()));
  GRD_TRY(b->blk_mem.alloc(reinterpret_cast<void **>(&b->partial), (uint64_t)std::max<uint32_t>(1, b->nblk) * 8));
  GRD_TRY(b->blk_mem.alloc_n(&b->gblk, gblk.size()));
  GRD_TRY(b->blk_mem.alloc_n(&b->glong, glong.size()));
  GRD_TRY(b->blk_mem.alloc_n(&b->tred, 2ull * std::max<uint32_t>(1, b->nblk)));
  GRD_TRY(b->blk_mem.alloc_n(&b->lred, 2ull * longs.size()));
  GRD_TRY(b->blk_mem.alloc_n(&b->scol, std::max<uint64_t>(1, b->E)));
  GRD_TRY(b->blk_mem.alloc_n(&b->spos, std::max<uint64_t>(1, b->E)));
  GRD_TRY(copy_in(b->ctx, b->gblk, gblk.data(), gblk.size() * 4));
  GRD_TRY(copy_in(b->ctx, b->glong, glong.data(), glong.size() * 4));
  GRD_TRY(copy_in(b->ctx, b->blocks, blks.data(), blks.size() * sizeof(BatchBlock)));
  GRD_TRY(copy_in(b->ctx, b->longs, longs.data(), longs.size() * sizeof(BatchLong)));
  if (b->E) GRD_HIP(hipMemcpyAsync(b->scol, b->ccol, b->E * 4, hipMemcpyDeviceToDevice, st));
  int bits = 1;
  while (bits < 31 && (b->N >> bits)) bits++;
#define F(T, N)                                                                                                    \
  hipLaunchKernelGGL((k_block_sort<BatchBlock, uint32_t, T, N>), dim3(b->nblk), dim3(T), 0, st, b->blocks, b->scol, \
                     (uint32_t *)nullptr, b->spos, bits)
  if (b->nblk) BATCH_SHAPES(b->nnz, F)
#undef F
  GRD_HIP(hipGetLastError());
  GRD_HIP(hipStreamSynchronize(st));  // the host vectors go out of scope
  return GRD_OK;
}

// the blocks for the present tile; without memory for them the batch has none
// (nnz 0) until a later tuning or run gets them
static grd_status batch_build_blocks(grd_batch *b)
{
  grd_status st;
  try {
    st = cut_blocks(b);
  } catch (const std::bad_alloc &) {
    st = fail(GRD_ERR_OOM, "batch: host allocation failed");
  }
  if (st != GRD_OK) {
    drop_captured(b);
    b->blk_mem.release();
    b->nnz = 0;
  }
  return st;
}

static uint32_t persistent_grid(const grd_batch *b) { return (uint32_t)b->ctx->num_cus * b->grid_per_cu; }

static uint32_t fixup_waves(const grd_batch *b)
{
  return std::min<uint32_t>(4096, (b->nlong + kWavesPerBlock - 1) / kWavesPerBlock);
}

static void launch_bpr(grd_batch *b, hipStream_t st, int parity, float damping, double tol, uint32_t max_iter)
{
  const float *cin = b->contrib[parity];
  float *cout = b->contrib[parity ^ 1];
  const uint32_t grid = std::min(b->nblk, persistent_grid(b));
#define F(T, N)                                                                                                      \
  hipLaunchKernelGGL((k_bpr_pull<T, N>), dim3(grid), dim3(T), 0, st, b->blocks, b->nblk, b->crp, b->scol, b->spos, \
                     cin, cout, b->r, b->deg, b->vb, b->dcur, damping, b->partial, b->tred, b->active)
  BATCH_SHAPES(b->nnz, F)
#undef F
  if (b->nlong)
    hipLaunchKernelGGL(k_bpr_fixup, dim3(fixup_waves(b)), dim3(kBlock), 0, st, b->longs, b->nlong, b->partial, cout,
                       b->r, b->deg, b->vb, b->dcur, damping, b->lred, b->active);
  hipLaunchKernelGGL(k_bpr_finish, dim3((b->count + kWavesPerBlock - 1) / kWavesPerBlock), dim3(kBlock), 0, st,
                     b->count, b->active, b->iters, b->gblk, b->glong, b->tred, b->lred, b->residual, b->dcur, tol,
                     max_iter, b->alive);
}

static void launch_bcc(grd_batch *b, hipStream_t st, int parity, uint32_t max_iter)
{
  const uint32_t grid = std::min(b->nblk, persistent_grid(b));
  uint32_t *lin = b->lab[parity], *lout = b->lab[parity ^ 1];
  uint32_t *part = reinterpret_cast<uint32_t *>(b->partial);
#define F(T, N)                                                                                                      \
  hipLaunchKernelGGL((k_bcc_pull<T, N>), dim3(grid), dim3(T), 0, st, b->blocks, b->nblk, b->crp, b->scol, b->spos, \
                     lin, lout, part, b->active, b->changed)
  BATCH_SHAPES(b->nnz, F)
#undef F
  if (b->nlong)
    hipLaunchKernelGGL(k_bcc_fixup, dim3(fixup_waves(b)), dim3(kBlock), 0, st, b->longs, b->nlong, part, lin, lout,
                       b->active, b->changed);
  hipLaunchKernelGGL(k_bcc_finish, dim3((b->count + 255) / 256), dim3(256), 0, st, b->count, b->active, b->iters,
                     b->changed, max_iter, b->alive);
}

// iterations per replay: an even number, so that the two buffers of the labels
// and of the contributions alternate inside one replay
static uint32_t replay_iters(const grd_batch *b) { return std::max<uint32_t>(2, b->K + (b->K & 1)); }

// the iterations of one replay captured into a graph, kept for the next run
// with the same parameters (capturing and instantiating take 0.2 ms)
static grd_status capture(grd_batch *b, int algo, double damping, double tol, uint32_t max_iter, hipGraphExec_t *exec)
{
  grd_batch::Captured &c = algo == GRD_CC ? b->cc_graph : b->pr_graph;
  const uint32_t grid = persistent_grid(b);
  if (c.exec && c.damping == damping && c.tol == tol && c.max_iter == max_iter && c.K == b->K && c.grid == grid) {
    *exec = c.exec;
    return GRD_OK;
  }
  if (c.exec) (void)hipGraphExecDestroy(c.exec);
  c.exec = nullptr;
  hipStream_t st = b->ctx->stream;
  hipGraph_t graph = nullptr;
  GRD_HIP(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
  for (uint32_t i = 0; i < replay_iters(b); i++) {
    if (algo == GRD_PR_PULL) launch_bpr(b, st, (int)(i & 1), (float)damping, tol, max_iter);
    else launch_bcc(b, st, (int)(i & 1), max_iter);
  }
  hipLaunchKernelGGL(k_balive, dim3(1), dim3(kWave), 0, st, b->alive, b->seq, b->h_alive);
  hipError_t e = hipStreamEndCapture(st, &graph);
  if (e != hipSuccess) return fail(GRD_ERR_HIP, std::string("hipStreamEndCapture: ") + hipGetErrorString(e));
  e = hipGraphInstantiate(&c.exec, graph, nullptr, nullptr, 0);
  (void)hipGraphDestroy(graph);
  if (e != hipSuccess) {
    c.exec = nullptr;
    return fail(GRD_ERR_HIP, std::string("hipGraphInstantiate: ") + hipGetErrorString(e));
  }
  c.damping = damping;
  c.tol = tol;
  c.max_iter = max_iter;
  c.K = b->K;
  c.grid = grid;
  *exec = c.exec;
  return GRD_OK;
}

static grd_status batch_run(grd_batch *b, int algo, double damping, double tol, uint32_t max_iter, uint32_t *iters_out,
                            double *ms_out)
{
  if (!b->nnz) GRD_TRY(batch_build_blocks(b));
  hipStream_t st = b->ctx->stream;
  const uint32_t cnt = b->count;
  // per-graph state (fill kernels: nothing memset-like inside the graph)
  hipLaunchKernelGGL(k_bfill_u32, dim3((cnt + 255) / 256), dim3(256), 0, st, b->active, cnt, 1u);
  hipLaunchKernelGGL(k_bfill_u32, dim3((cnt + 255) / 256), dim3(256), 0, st, b->iters, cnt, 0u);
  hipLaunchKernelGGL(k_bfill_u32, dim3((cnt + 255) / 256), dim3(256), 0, st, b->changed, cnt, 0u);
  hipLaunchKernelGGL(k_bfill_f64, dim3((cnt + 255) / 256), dim3(256), 0, st, b->residual, cnt, 0.0);
  const uint32_t ig = (uint32_t)std::min<uint64_t>(4096, b->N / kBlock + 1);
  if (algo == GRD_PR_PULL) {
    hipLaunchKernelGGL(k_bpr_init, dim3(ig), dim3(kBlock), 0, st, b->N, b->vb, cnt, b->changed + cnt, b->deg, b->r,
                       b->contrib[0]);
    GRD_HIP(hipMemcpyAsync(b->dcur, b->d0.data(), cnt * sizeof(double), hipMemcpyHostToDevice, st));
  } else {
    hipLaunchKernelGGL(k_bcc_init, dim3(ig), dim3(kBlock), 0, st, b->N, b->gid_local, b->lab[0], b->lab[1]);
  }
  hipLaunchKernelGGL(k_bfill_u32, dim3(1), dim3(64), 0, st, b->alive, 1u, 0u);
  GRD_HIP(hipGetLastError());
  hipGraphExec_t exec = nullptr;
  GRD_TRY(capture(b, algo, damping, tol, max_iter, &exec));
  GRD_HIP(hipEventRecord(b->ctx->ev[0], st));
  uint32_t launched = 0;
  const uint32_t per = replay_iters(b);
  grd_status rc = GRD_OK;
  while (launched < max_iter) {
    hipError_t e = hipGraphLaunch(exec, st);
    if (e != hipSuccess) {
      rc = fail(GRD_ERR_HIP, std::string("hipGraphLaunch: ") + hipGetErrorString(e));
      break;
    }
    launched += per;
    rc = wait_pinned(b->ctx, b->h_alive + 1, ++b->h_seq);
    if (rc != GRD_OK || *b->h_alive == 0) break;
  }
  if (rc != GRD_OK) (void)hipStreamSynchronize(st);
  hipEventRecord(b->ctx->ev[1], st);
  hipEventSynchronize(b->ctx->ev[1]);
  float ms = 0.0f;
  hipEventElapsedTime(&ms, b->ctx->ev[0], b->ctx->ev[1]);
  GRD_TRY(rc);
  b->last_iters.assign(cnt, 0);
  GRD_HIP(hipMemcpy(b->last_iters.data(), b->iters, cnt * 4, hipMemcpyDeviceToHost));
  if (iters_out) memcpy(iters_out, b->last_iters.data(), cnt * 4);
  if (ms_out) *ms_out = ms;
  b->last_algo = algo;
  return GRD_OK;
}

}  // namespace grd

using namespace grd;

extern "C" {

grd_status grd_batch_create(grd_ctx *ctx, uint32_t count, const uint32_t *n, const uint64_t *m,
                            const uint32_t *const *row_ptr, const uint32_t *const *col, grd_batch **out)
{
  if (!ctx || !n || !m || !row_ptr || !col || !out || count == 0) return fail(GRD_ERR_ARG, "grd_batch_create: bad argument");
  GRD_HIP(hipSetDevice(ctx->device));
  try {
    grd_batch *b = new grd_batch();
    b->ctx = b->mem.ctx = b->blk_mem.ctx = b->st_mem.ctx = ctx;
    b->count = count;
    b->vbase.assign(count + 1, 0);
    for (uint32_t g = 0; g < count; g++) {
      if (n[g] == 0 || row_ptr[g][n[g]] != m[g]) {
        delete b;
        return fail(GRD_ERR_ARG, "grd_batch_create: graph " + std::to_string(g) + " is empty or inconsistent");
      }
      b->vbase[g + 1] = b->vbase[g] + n[g];
      b->E += m[g];
    }
    b->N = b->vbase[count];
    if (b->N >= 0xFFFFFFF0ull || b->E >= 0xFFFFFFF0ull) {
      delete b;
      return fail(GRD_ERR_ARG, "grd_batch_create: batch exceeds the u32 vertex / arc limit");
    }
    // concatenated CSC (in-edges, sources ascending), out-degrees, graph ids
    b->h_crp.assign(b->N + 1, 0);
    b->h_deg.assign(b->N, 0);
    std::vector<uint32_t> gidx(b->N), local(b->N);
    for (uint32_t g = 0; g < count; g++) {
      const uint64_t vb = b->vbase[g];
      for (uint32_t u = 0; u < n[g]; u++) {
        b->h_deg[vb + u] = row_ptr[g][u + 1] - row_ptr[g][u];
        gidx[vb + u] = g;
        local[vb + u] = u;
        for (uint32_t x = row_ptr[g][u]; x < row_ptr[g][u + 1]; x++) {
          if (col[g][x] >= n[g]) {
            delete b;
            return fail(GRD_ERR_ARG, "grd_batch_create: column out of range in graph " + std::to_string(g));
          }
          b->h_crp[vb + col[g][x] + 1]++;
        }
      }
    }
    for (uint64_t v = 0; v < b->N; v++) b->h_crp[v + 1] += b->h_crp[v];
    std::vector<uint32_t> hcol(b->E), cur(b->h_crp.begin(), b->h_crp.end() - 1);
    for (uint32_t g = 0; g < count; g++) {
      const uint64_t vb = b->vbase[g];
      for (uint32_t u = 0; u < n[g]; u++)
        for (uint32_t x = row_ptr[g][u]; x < row_ptr[g][u + 1]; x++)
          hcol[cur[vb + col[g][x]]++] = (uint32_t)(vb + u);
    }
    grd_status st = GRD_OK;
    auto up = [&](uint32_t **dst, const std::vector<uint32_t> &src) -> grd_status {
      GRD_TRY(b->mem.alloc_n(dst, std::max<size_t>(1, src.size())));
      if (!src.empty()) GRD_HIP(hipMemcpy(*dst, src.data(), src.size() * 4, hipMemcpyHostToDevice));
      return GRD_OK;
    };
    if ((st = up(&b->crp, b->h_crp)) != GRD_OK || (st = up(&b->ccol, hcol)) != GRD_OK ||
        (st = up(&b->deg, b->h_deg)) != GRD_OK || (st = up(&b->gid_local, local)) != GRD_OK) {
      delete b;
      return st;
    }
    // per-graph and per-vertex state; the graph index of each vertex rides
    // behind `changed` (changed[count + v])
    DevMem &sm = b->st_mem;
    if ((st = b->mem.alloc_n(&b->vb, count + 1)) != GRD_OK || (st = sm.alloc_n(&b->r, b->N)) != GRD_OK ||
        (st = sm.alloc_n(&b->contrib[0], b->N)) != GRD_OK || (st = sm.alloc_n(&b->contrib[1], b->N)) != GRD_OK ||
        (st = sm.alloc_n(&b->lab[0], b->N)) != GRD_OK || (st = sm.alloc_n(&b->lab[1], b->N)) != GRD_OK ||
        (st = sm.alloc_n(&b->active, count)) != GRD_OK || (st = sm.alloc_n(&b->iters, count)) != GRD_OK ||
        (st = sm.alloc_n(&b->changed, count + b->N)) != GRD_OK || (st = sm.alloc_n(&b->alive, 1)) != GRD_OK ||
        (st = sm.alloc_n(&b->residual, count)) != GRD_OK || (st = sm.alloc_n(&b->dcur, count)) != GRD_OK ||
        (st = sm.alloc_n(&b->seq, 1)) != GRD_OK) {
      delete b;
      return st;
    }
    GRD_HIP(hipMemcpy(b->vb, b->vbase.data(), (count + 1) * 8, hipMemcpyHostToDevice));
    GRD_HIP(hipMemcpy(b->changed + count, gidx.data(), b->N * 4, hipMemcpyHostToDevice));
    // D0 per graph: sinks * (1/n) in FP64
    b->d0.assign(count, 0.0);
    for (uint32_t g = 0; g < count; g++) {
      uint64_t sinks = 0;
      for (uint64_t v = b->vbase[g]; v < b->vbase[g + 1]; v++) sinks += b->h_deg[v] == 0;
      b->d0[g] = (double)sinks * (double)(float)(1.0 / (double)(b->vbase[g + 1] - b->vbase[g]));
    }
    GRD_HIP(hipHostMalloc((void **)&b->h_alive, 64, hipHostMallocDefault));
    b->h_alive[0] = b->h_alive[1] = 0;
    hipLaunchKernelGGL(k_bfill_u32, dim3(1), dim3(64), 0, ctx->stream, b->seq, 1u, 0u);
    if ((st = batch_build_blocks(b)) != GRD_OK) {
      (void)hipHostFree(b->h_alive);
      delete b;
      return st;
    }
    *out = b;
    return GRD_OK;
  } catch (const std::bad_alloc &) {
    return fail(GRD_ERR_OOM, "grd_batch_create: host allocation failed");
  }
}

grd_status grd_batch_free(grd_batch *b)
{
  if (!b) return GRD_OK;
  (void)hipStreamSynchronize(b->ctx->stream);
  drop_captured(b);
  if (b->h_alive) (void)hipHostFree(b->h_alive);
  delete b;
  return GRD_OK;
}

grd_status grd_batch_tune(grd_batch *b, uint32_t tile, uint32_t grid_per_cu, uint32_t K)
{
  if (!b) return fail(GRD_ERR_ARG, "grd_batch_tune: NULL batch");
  if (tile && tile != 1024 && tile != 2048 && tile != 4096)
    return fail(GRD_ERR_ARG, "grd_batch_tune: tile must be 1024, 2048 or 4096 arcs");
  if (grid_per_cu > 64 || K > 64) return fail(GRD_ERR_ARG, "grd_batch_tune: grid_per_cu and K must be <= 64");
  if (grid_per_cu) b->grid_per_cu = grid_per_cu;
  if (K) b->K = K;
  if (tile) b->tile = tile;
  if (block_arcs(b, b->tile) != b->nnz) GRD_TRY(batch_build_blocks(b));
  return GRD_OK;
}

grd_status grd_batch_autotune(grd_batch *b, uint32_t *chosen3)
{
  if (!b) return fail(GRD_ERR_ARG, "grd_batch_autotune: NULL batch");
  const uint32_t tiles[] = {1024, 2048, 4096}, grids[] = {4, 8, 16}, Ks[] = {2, 4, 8};
  double best = 1e30;
  uint32_t bt = b->tile, bg = b->grid_per_cu, bk = b->K, last = 0;
  for (uint32_t t : tiles) {
    // tiles that give the same blocks are one candidate (from 8192 arcs
    // per CU on all of them do)
    if (block_arcs(b, t) == last) continue;
    last = block_arcs(b, t);
    for (uint32_t gpc : grids)
      for (uint32_t k : Ks) {
        GRD_TRY(grd_batch_tune(b, t, gpc, k));
        // a fixed amount of work per candidate: 16 PageRank iterations
        double ms = 0.0;
        GRD_TRY(batch_run(b, GRD_PR_PULL, 0.85, 0.0, 16, nullptr, &ms));
        if (ms < best) {
          best = ms;
          bt = t;
          bg = gpc;
          bk = k;
        }
      }
  }
  GRD_TRY(grd_batch_tune(b, bt, bg, bk));
  if (chosen3) {
    chosen3[0] = bt;
    chosen3[1] = bg;
    chosen3[2] = bk;
  }
  return GRD_OK;
}

grd_status grd_batch_pagerank(grd_batch *b, double damping, double tolerance, uint32_t max_iter, uint32_t *iters_out,
                              double *ms_out)
{
  if (!b || max_iter == 0) return fail(GRD_ERR_ARG, "grd_batch_pagerank: bad argument");
  GRD_HIP(hipSetDevice(b->ctx->device));
  return batch_run(b, GRD_PR_PULL, damping, tolerance, max_iter, iters_out, ms_out);
}

grd_status grd_batch_cc(grd_batch *b, uint32_t max_iter, uint32_t *iters_out, double *ms_out)
{
  if (!b || max_iter == 0) return fail(GRD_ERR_ARG, "grd_batch_cc: bad argument");
  GRD_HIP(hipSetDevice(b->ctx->device));
  return batch_run(b, GRD_CC, 0.0, 0.0, max_iter, iters_out, ms_out);
}

grd_status grd_batch_download(grd_batch *b, uint32_t i, int algo, void *out)
{
  if (!b || !out || i >= b->count) return fail(GRD_ERR_ARG, "grd_batch_download: bad argument");
  if (algo != b->last_algo) return fail(GRD_ERR_STATE, "grd_batch_download: that algorithm has not run last");
  const uint64_t v0 = b->vbase[i], n = b->vbase[i + 1] - v0;
  if (algo == GRD_PR_PULL) {
    return copy_out(b->ctx, out, b->r + v0, n);
  }
  if (algo == GRD_CC) {
    // the last superstep of graph i wrote buffer iters % 2 (and changed nothing)
    return copy_out(b->ctx, out, b->lab[b->last_iters[i] & 1] + v0, n);
  }
  return fail(GRD_ERR_ARG, "grd_batch_download: algo must be GRD_PR_PULL or GRD_CC");
}

}  // extern "C"
