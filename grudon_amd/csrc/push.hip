// push.hip -- the push traversal over the active list: gen_updates on the
// memory partitions, and the edge-shipping superstep, which applies the same
// arcs straight to the compute side.
#include <algorithm>
#include <type_traits>

#include "grd_device.hpp"
#include "grd_internal.hpp"
#include "grd_ops.hpp"

namespace grd {

// ------------------------------------------------------------------------
// traversal: push over the active list (degree-binned, LDS-staged tiles)
// ------------------------------------------------------------------------

// owner of position j among a tile's 256 offsets: the last t with s_off[t] <= j
// (s_off[0] = 0; eight halvings, no branch)
__device__ __forceinline__ uint32_t push_owner(const uint32_t *s_off, uint32_t j)
{
  uint32_t t = 0;
#pragma unroll
  for (uint32_t step = kBlock / 2; step > 0; step >>= 1)
    if (s_off[t + step] <= j) t += step;
  return t;
}

// A block stages `tile` active vertices in LDS (256, or 64 where the frontier
// would not fill the chip with tiles of 256).  Vertices with out-degree below
// kHeavyDeg are processed together: the block scans their degrees and every
// thread walks the concatenated edge range (coalesced col reads), locating its
// source by binary search in the LDS prefix array, four arcs in flight per
// thread.  Vertices with degree >= kHeavyDeg are appended to the heavy list as
// chunks of kHeavyChunk arcs (one counter atomic per tile) and handled by
// k_push_heavy, a wave per chunk.
//
// The active list is in degree order, so the vertices just below the threshold
// share tiles: the threshold bounds a tile's work, and a round of 1024 arcs takes
// about 4.5 us in a full chip whatever they find.  With 4096 (and chunks of
// 4096) the first tiles held a million arcs each and ran alone: CC by pushes
// over RMAT-20 symmetrized (31 M arcs) 16.7 ms a solve; with 256 and a workgroup
// per chunk of 1024 3.3, of which 1.8 in the longest tiles; with 64 and a wave
// per chunk of 256 2.5 (32 to 96 and chunks of 128 to 512 within 2 %; two arcs in
// flight a lane in the heavy pass, four measured the same).
//
// kShip: the edge-shipping superstep (ship.hip).  The columns are the
// out-neighbours' compute slots and the updates go to the compute side, where
// every add marks (addUpdate, relax).  W: the weights' storage.  The values pushed
// are val by proxy, or by compute slot with the proxies' slots in slot.
template <class Op, bool kShip, class W>
__global__ void __launch_bounds__(kBlock) k_push(const uint32_t *__restrict__ AL, const uint32_t *__restrict__ nact,
                                                 const uint32_t *__restrict__ rp, const uint32_t *__restrict__ col,
                                                 const W *__restrict__ wt, const typename Op::V *__restrict__ val,
                                                 const uint32_t *__restrict__ slot, typename Op::V *upd,
                                                 uint64_t *dirty, uint2 *heavy, Counters *cnt, uint32_t tile)
{
  using V = typename Op::V;
  constexpr int kIlp = 4;
  __shared__ uint32_t s_off[kBlock];
  __shared__ uint32_t s_beg[kBlock];
  __shared__ V s_val[kBlock];
  __shared__ unsigned long long s_slot;
  const uint32_t k = *nact;
  for (uint32_t t0 = blockIdx.x * tile; t0 < k; t0 += gridDim.x * tile) {
    const uint32_t i = t0 + threadIdx.x;
    uint32_t deg = 0, beg = 0, p = 0, nch = 0;
    V v = op_identity<Op>();
    if (threadIdx.x < tile && i < k) {
      p = AL[i];
      beg = rp[p];
      deg = rp[p + 1] - beg;
      v = val[slot ? slot[p] : p];
      if (deg >= kHeavyDeg) nch = (deg + kHeavyChunk - 1) / kHeavyChunk;
    }
    if (__syncthreads_or(nch != 0)) {
      uint32_t hch;
      const uint32_t at = block_excl_scan(nch, &hch);
      if (threadIdx.x == 0) s_slot = atomicAdd(&cnt->heavy, (unsigned long long)hch);
      __syncthreads();
      for (uint32_t c = 0; c < nch; c++) heavy[s_slot + at + c] = make_uint2(p, c * kHeavyChunk);
      if (nch) deg = 0;
    }
    uint32_t total;
    const uint32_t ex = block_excl_scan(deg, &total);
    s_off[threadIdx.x] = ex;
    s_beg[threadIdx.x] = beg;
    s_val[threadIdx.x] = v;
    __syncthreads();
    const uint32_t l = lane_id();
    for (uint32_t j0 = threadIdx.x; j0 - l < total; j0 += kIlp * kBlock) {  // the same rounds for every lane of a wave
      uint32_t c[kIlp], w[kIlp];
      V x[kIlp];
#pragma unroll
      for (int q = 0; q < kIlp; q++) {
        const uint32_t j = j0 + q * kBlock;
        const uint32_t t = push_owner(s_off, j);
        const uint32_t e = j < total ? s_beg[t] + (j - s_off[t]) : s_beg[0];
        c[q] = 0;
        w[q] = 1u;
        if (j < total) {
          c[q] = col[e];
          if constexpr (std::is_same<Op, OpWeighted>::value) w[q] = wt[e];
        }
        x[q] = s_val[t];
      }
#pragma unroll
      for (int q = 0; q < kIlp; q++) x[q] = Op::edge(x[q], w[q]);
      relax_many<Op, kIlp, kShip>(upd, dirty, c, x, j0 < total ? (total - j0 + kBlock - 1) / kBlock : 0u);
    }
    __syncthreads();
  }
}

template <class Op, bool kShip, class W>
__global__ void __launch_bounds__(kBlock) k_push_heavy(const uint2 *__restrict__ heavy, const Counters *cnt,
                                                       const uint32_t *__restrict__ rp, const uint32_t *__restrict__ col,
                                                       const W *__restrict__ wt,
                                                       const typename Op::V *__restrict__ val,
                                                       const uint32_t *__restrict__ slot, typename Op::V *upd,
                                                       uint64_t *dirty)
{
  using V = typename Op::V;
  constexpr int kIlp = 2;
  const uint32_t nch = (uint32_t)cnt->heavy, l = lane_id();
  for (uint32_t h = blockIdx.x * kWavesPerBlock + wave_in_block(); h < nch; h += gridDim.x * kWavesPerBlock) {
    const uint2 ch = heavy[h];
    const uint32_t end = rp[ch.x + 1];
    const uint32_t b = rp[ch.x] + ch.y, ne = min(end - b, kHeavyChunk);
    const V v = val[slot ? slot[ch.x] : ch.x];
    for (uint32_t j0 = l; j0 - l < ne; j0 += kIlp * kWave) {
      uint32_t c[kIlp], w[kIlp];
      V x[kIlp];
#pragma unroll
      for (int q = 0; q < kIlp; q++) {
        const uint32_t j = j0 + q * kWave;
        c[q] = 0;
        w[q] = 1u;
        if (j < ne) {
          c[q] = col[b + j];
          if constexpr (std::is_same<Op, OpWeighted>::value) w[q] = wt[b + j];
        }
      }
#pragma unroll
      for (int q = 0; q < kIlp; q++) x[q] = Op::edge(v, w[q]);
      relax_many<Op, kIlp, kShip>(upd, dirty, c, x, j0 < ne ? (ne - j0 + kWave - 1) / kWave : 0u);
    }
  }
}

__global__ void k_heavy_restart(Counters *cnt)
{
  if (threadIdx.x == 0) cnt->heavy = 0;
}

template <class Op, bool kShip, class W>
static grd_status launch(grd_state *s, const uint32_t *col, const W *wt, typename Op::V *upd, uint64_t *dirty)
{
  grd_graph *g = s->g;
  grd_ctx *ctx = g->ctx;
  hipStream_t st = ctx->stream;
  using V = typename Op::V;
  // The memory side's proxies hold what was broadcast.  Edge shipping aggregates
  // the source's property on the compute side: the same value, until an update
  // has come between.
  const bool moved = kShip && s->bcast_stale;
  const V *val = moved ? (const V *)s->prop : (const V *)s->mprop;
  const uint32_t *slot = moved ? g->proxy_slot : nullptr;
  // tiles of 64 active vertices until those fill every workgroup slot
  const uint64_t slots = (uint64_t)ctx->num_cus * 8;
  const uint32_t tile = s->al_vertices <= 64 * slots ? 64u : (uint32_t)kBlock;
  const uint32_t grid = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>((s->al_vertices + tile - 1) / tile, slots));
  // the heavy list holds one pass over the active list: another push of the same
  // broadcast lists its chunks anew
  if (s->heavy_listed) hipLaunchKernelGGL(k_heavy_restart, dim3(1), dim3(kWave), 0, st, s->cnt);
  s->heavy_listed = true;
  hipLaunchKernelGGL((k_push<Op, kShip, W>), dim3(grid), dim3(kBlock), 0, st, s->AL, s->totals + 0, g->rp, col, wt,
                     val, slot, upd, dirty, s->heavy, s->cnt, tile);
  // a vertex's out-arcs all hang off its own proxy, so the list's largest
  // out-degree tells whether any chunk was appended
  if (s->al_maxdeg >= kHeavyDeg)
    hipLaunchKernelGGL((k_push_heavy<Op, kShip, W>), dim3((uint32_t)slots), dim3(kBlock), 0, st, s->heavy, s->cnt,
                       g->rp, col, wt, val, slot, upd, dirty);
  GRD_HIP(hipGetLastError());
  s->edges += s->al_edges;  // every out-arc of the active list
  return GRD_OK;
}

template <class Op>
grd_status push_launch(grd_state *s)
{
  using V = typename Op::V;
  return launch<Op, false, uint32_t>(s, s->g->col, s->g->w, (V *)s->mupd, s->Du);
}

template <class Op>
grd_status ship_launch(grd_state *s)
{
  using V = typename Op::V;
  grd_graph *g = s->g;
  if constexpr (std::is_same<Op, OpWeighted>::value)
    if (g->ship_wbytes == 1) return launch<Op, true, uint8_t>(s, g->scol, g->w8, (V *)s->upd, s->Dc);
  return launch<Op, true, uint32_t>(s, g->scol, g->w, (V *)s->upd, s->Dc);
}

template grd_status push_launch<OpCC>(grd_state *);
template grd_status push_launch<OpHop>(grd_state *);
template grd_status push_launch<OpWeighted>(grd_state *);
template grd_status push_launch<OpPR>(grd_state *);
template grd_status ship_launch<OpCC>(grd_state *);
template grd_status ship_launch<OpHop>(grd_state *);
template grd_status ship_launch<OpWeighted>(grd_state *);
template grd_status ship_launch<OpPR>(grd_state *);

}  // namespace grd
