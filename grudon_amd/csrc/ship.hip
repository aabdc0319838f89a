// ship.hip -- the NO_OFFLOAD edge-shipping schedule and the inputs of its
// NDPEngine vote.
//
// Reference: src/GraphAlgorithm.cpp:426-474 (memory side: for every vertex
// the broadcast updated, send [gid, gid of each out-neighbour] to its master)
// and :582-637 (compute side: receive the lists of its frontier and aggregate
// the source's property into every listed neighbour); the vote is
// include/offload_engine/NDPEngine.hpp:10-51 with the coverage vector of
// src/DistributedGraph.cpp:286-370.
//
// On one GPU the memory side's send and the compute side's receive are one
// pass: the push over the active list (push.hip, kShip), reading each
// out-neighbour by compute slot, the receiver's local id, and aggregating the
// source's property into it.  The reference applies addUpdate in its receive
// whatever the algorithm (a TODO at :624); this applies the algorithm's own
// aggregate, which is what makes the schedule give the same result as the
// offloaded one.  With the records written to a buffer and read back (record
// lengths, their scan, tile starts, a send and a receive kernel) a shipping
// superstep took five more launches and 8 to 10 bytes more per arc (CC on a
// thousand vertices 364 -> 314 us a solve, weighted SSSP on RMAT-22 5.2 -> 5.1 ms).
#include <algorithm>
#include <cstring>
#include <type_traits>

#include "grd_device.hpp"
#include "grd_internal.hpp"
#include "grd_ops.hpp"

namespace grd {

// ------------------------------------------------------------------------
// coverage: a vertex is covered when all of its out-neighbours share its
// master, so that its compute partition can apply every update of its list
// ------------------------------------------------------------------------

// One thread per compute slot; a wave covers exactly one slot word.  The own
// proxy of slot w*64+l is word_dst[w]*64+l (the own region repeats the slot
// order), and it holds all of the vertex's out-arcs.
__global__ void __launch_bounds__(kBlock) k_uncovered(uint32_t S, uint32_t C, const uint32_t *__restrict__ slot_gid,
                                                      const uint32_t *__restrict__ word_dst,
                                                      const uint32_t *__restrict__ rp, const uint32_t *__restrict__ col,
                                                      const uint32_t *__restrict__ proxy_slot,
                                                      uint64_t *__restrict__ uncov)
{
  for (uint32_t s = blockIdx.x * kBlock + threadIdx.x; s < S; s += gridDim.x * kBlock) {
    const uint32_t v = slot_gid[s];
    bool unc = false;
    if (v != kNone) {
      const uint32_t pw = word_dst[s >> 6];
      if (pw != kNone) {
        const uint32_t p = pw * 64 + (s & 63), mc = v % C;
        for (uint32_t e = rp[p]; e < rp[p + 1]; e++)
          if (slot_gid[proxy_slot[col[e]]] % C != mc) {
            unc = true;
            break;
          }
      }
    }
    const uint64_t m = __ballot(unc);
    if (lane_id() == 0) uncov[s >> 6] = m;
  }
}

// ------------------------------------------------------------------------
// per-partition frontier sizes and uncovered frontier vertices
// ------------------------------------------------------------------------

__global__ void __launch_bounds__(kBlock) k_frontier_parts(uint32_t nw, const uint64_t *__restrict__ F,
                                                           const uint8_t *__restrict__ word_c,
                                                           const uint64_t *__restrict__ uncov, uint32_t C,
                                                           Counters *cnt)
{
  __shared__ unsigned long long s_fc[kMaxParts];
  for (uint32_t i = threadIdx.x; i < (uint32_t)kMaxParts; i += kBlock) s_fc[i] = 0;
  __syncthreads();
  uint64_t unc = 0;
  for (uint32_t w = blockIdx.x * kBlock + threadIdx.x; w < nw; w += gridDim.x * kBlock) {
    const uint64_t f = F[w];
    if (f) {
      atomicAdd(&s_fc[word_c[w]], (unsigned long long)__popcll(f));
      unc += (uint64_t)__popcll(f & uncov[w]);
    }
  }
  __syncthreads();
  unc = block_sum(unc);
  if (threadIdx.x == 0 && unc) atomicAdd(&cnt->frontier_uncovered, (unsigned long long)unc);
  for (uint32_t c = threadIdx.x; c < C; c += kBlock)
    if (s_fc[c]) atomicAdd(&cnt->fpart[c], s_fc[c]);
}

// ------------------------------------------------------------------------
// shipped columns and weights
// ------------------------------------------------------------------------

// (a capped grid and one atomic per workgroup: with one per wave of a flat grid,
// 3 ms for 130 M weights, now 155 us)
__global__ void __launch_bounds__(kBlock) k_weight_max(uint64_t m, const uint32_t *__restrict__ w, uint32_t *__restrict__ out)
{
  uint32_t mx = 0;
#pragma unroll 8
  for (uint64_t e = (uint64_t)blockIdx.x * kBlock + threadIdx.x; e < m; e += (uint64_t)gridDim.x * kBlock) mx = max(mx, w[e]);
  mx = block_max(mx);
  if (threadIdx.x == 0 && mx) atomicMax(out, mx);
}

__global__ void __launch_bounds__(kBlock) k_ship_w8(uint64_t m, const uint32_t *__restrict__ w, uint8_t *__restrict__ w8)
{
  for (uint64_t e = (uint64_t)blockIdx.x * kBlock + threadIdx.x; e < m; e += (uint64_t)gridDim.x * kBlock)
    w8[e] = (uint8_t)w[e];
}

__global__ void __launch_bounds__(kBlock) k_slot_col(uint64_t m, const uint32_t *__restrict__ col,
                                                     const uint32_t *__restrict__ proxy_slot, uint32_t *__restrict__ scol)
{
  for (uint64_t e = (uint64_t)blockIdx.x * kBlock + threadIdx.x; e < m; e += (uint64_t)gridDim.x * kBlock)
    scol[e] = proxy_slot[col[e]];
}

// ------------------------------------------------------------------------
// host side
// ------------------------------------------------------------------------

static uint32_t grid_for(uint64_t n, uint32_t cap = 4096)
{
  return (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(cap, (n + kBlock - 1) / kBlock));
}

grd_status build_ship_tables(grd_graph *g)
{
  hipStream_t st = g->ctx->stream;
  const uint32_t nwS = g->S / 64;
  // compute partition of every slot word: pair (c, m) owns its own count
  // rounded up to whole words from cbase[c * M + m]
  std::vector<uint8_t> wc(std::max<uint32_t>(nwS, 1), 0);
  for (int c = 0; c < g->C; c++)
    for (int m = 0; m < g->M; m++) {
      const size_t pi = (size_t)c * g->M + m;
      const uint64_t w0 = g->cbase[pi] / 64, w1 = (g->cbase[pi] + (uint64_t)g->ccnt[pi] + 63) / 64;
      for (uint64_t w = w0; w < w1 && w < nwS; w++) wc[w] = (uint8_t)c;
    }
  GRD_TRY(g->mem.alloc_n(&g->word_c, wc.size()));
  GRD_HIP(hipMemcpyAsync(g->word_c, wc.data(), wc.size(), hipMemcpyHostToDevice, st));
  GRD_TRY(g->mem.alloc_n(&g->uncov, std::max<uint32_t>(nwS, 1)));
  g->n_uncovered = 0;
  if (g->C == 1) {
    GRD_HIP(hipMemsetAsync(g->uncov, 0, (uint64_t)std::max<uint32_t>(nwS, 1) * 8, st));
  } else {
    hipLaunchKernelGGL(k_uncovered, dim3(grid_for(g->S, 1u << 16)), dim3(kBlock), 0, st, g->S, (uint32_t)g->C,
                       g->slot_gid, g->word_dst, g->rp, g->col, g->proxy_slot, g->uncov);
    GRD_HIP(hipGetLastError());
    std::vector<uint64_t> h(nwS);
    GRD_HIP(hipMemcpyAsync(h.data(), g->uncov, (uint64_t)nwS * 8, hipMemcpyDeviceToHost, st));
    GRD_HIP(hipStreamSynchronize(st));
    for (uint64_t x : h) g->n_uncovered += (uint64_t)__builtin_popcountll(x);
  }
  GRD_HIP(hipStreamSynchronize(st));
  return GRD_OK;
}

grd_status op_frontier_parts(grd_state *s)
{
  grd_graph *g = s->g;
  const uint32_t nwS = g->S / 64;
  hipLaunchKernelGGL(k_frontier_parts, dim3(grid_for(nwS, 1024)), dim3(kBlock), 0, g->ctx->stream, nwS, s->F,
                     g->word_c, g->uncov, (uint32_t)g->C, s->cnt);
  GRD_HIP(hipGetLastError());
  return GRD_OK;
}

// the largest arc weight, once per graph
grd_status weight_max(grd_graph *g, uint32_t *out)
{
  if (!g->wmax_known) {
    hipStream_t st = g->ctx->stream;
    DevMem tmp(g->ctx);
    uint32_t *d_max = nullptr;
    GRD_TRY(tmp.alloc_n(&d_max, 1));
    GRD_HIP(hipMemsetAsync(d_max, 0, 4, st));
    hipLaunchKernelGGL(k_weight_max, dim3(grid_for(g->m, (uint32_t)g->ctx->num_cus * 8)), dim3(kBlock), 0, st, g->m,
                       g->w, d_max);
    GRD_HIP(hipGetLastError());
    GRD_HIP(hipMemcpyAsync(&g->wmax, d_max, 4, hipMemcpyDeviceToHost, st));
    GRD_HIP(hipStreamSynchronize(st));
    g->wmax_known = true;
  }
  *out = g->wmax;
  return GRD_OK;
}

template <class Op>
static grd_status ship_t(grd_state *s)
{
  grd_graph *g = s->g;
  hipStream_t st = g->ctx->stream;
  const uint64_t k = s->last_frontier, E = s->last_frontier_edges;
  if (k == 0) return GRD_OK;
  // (an update since the broadcast: what was checked for coverage and is sized
  // here is not what the list holds)
  if (s->al_vertices != k || s->al_edges != E)
    return fail(GRD_ERR_STATE, "edge shipping: the active list differs from the frontier");
  const uint64_t total = k + E;
  // the records' entries (a source each, and its out-neighbours) are counted in 32 bits
  if (total > 0xFFFFFFFFull - 1024) return fail(GRD_ERR_ARG, "edge shipping: the wire would exceed 2^32 entries");
  const bool weighted = std::is_same<Op, OpWeighted>::value;
  if (weighted && !g->ship_wbytes) {
    // the weights travel as bytes when every one of them is below 256
    uint32_t wmax = 0;
    GRD_TRY(weight_max(g, &wmax));
    if (wmax < 256) {
      GRD_TRY(g->mem.alloc_n(&g->w8, std::max<uint64_t>(g->m, 1)));
      hipLaunchKernelGGL(k_ship_w8, dim3(grid_for(g->m, 1u << 16)), dim3(kBlock), 0, st, g->m, g->w, g->w8);
      GRD_HIP(hipGetLastError());
    }
    g->ship_wbytes = wmax < 256 ? 1 : 4;
  }
  if (!g->scol) {  // the push CSR's columns as compute slots, once per graph
    GRD_TRY(g->mem.alloc_n(&g->scol, std::max<uint64_t>(g->m, 1)));
    hipLaunchKernelGGL(k_slot_col, dim3(grid_for(g->m, 1u << 16)), dim3(kBlock), 0, st, g->m, g->col, g->proxy_slot,
                       g->scol);
    GRD_HIP(hipGetLastError());
  }
  const bool timed = s->prm.time_kernel != 0;
  if (timed) GRD_HIP(hipEventRecord(s->kev[0], st));
  GRD_TRY(ship_launch<Op>(s));
  if (timed) {
    GRD_HIP(hipEventRecord(s->kev[1], st));
    s->kern_pending = 2;  // bytes from the active list's vertices and arcs
  }
  // wire bytes (MPI.hpp:44 counts count * sizeof(GNode) per send): one id
  // per record header and per arc, plus the weights of a weighted SSSP
  s->bytes += 4 * total + (weighted ? 4 * E : 0);
  return GRD_OK;
}

grd_status op_ship(grd_state *s)
{
  s->cnt_clean = false;
  switch (s->algo) {
  case GRD_PR: return ship_t<OpPR>(s);
  case GRD_CC: return ship_t<OpCC>(s);
  case GRD_SSSP: return s->prm.weighted ? ship_t<OpWeighted>(s) : ship_t<OpHop>(s);
  default: return fail(GRD_ERR_STATE, "edge shipping: algorithm has no BSP traversal");
  }
}

}  // namespace grd
