// grd_rows.hpp -- row blocks whose arcs are kept in source order: the staged
// values of a block lie in LDS in row order and are reduced row by row (the cold
// pass of the hot / cold pull, the batched pulls).
#pragma once

#include <rocprim/block/block_radix_sort.hpp>

#include "grd_device.hpp"
#include "grd_ops.hpp"

namespace grd {

// arcs in flight per thread
constexpr int kBatch = 8;

// lanes per row of a block of nrows rows: as many as one round of the
// workgroup's T threads has.  More lanes than that for longer average rows cost
// extra rounds and merges: at least one lane per 8 arcs took the 24-graph batch
// from 2.72 to 3.41 ms.
template <int T>
__device__ __forceinline__ uint32_t row_group(uint32_t nrows)
{
  uint32_t g = kWave;
  while (g > 1 && g * nrows > (uint32_t)T) g >>= 1;
  return g;
}

// The row sums of one round: groups of G lanes over [b, e) of the staged
// values; the sum is valid in the group's first lane.  A row much longer than
// its group is left to the whole wave (blocks mix rows of one arc with rows of
// thousands; a lane alone takes about 30 ns per compensated add).  Called by
// the whole wave.
//
// kWideRow: arcs per lane beyond which the wave takes the row.  Below, the lanes of a wave
// run side by side; above, the wave goes from row to row.  The 24-graph batch's
// PageRank: 3.31 ms at 24, 2.73 at 48, 2.72 at 64, 2.86 at 128, 7.5 without; the
// cold pass of a hot / cold pull is within 2 % from 24 to 128.
constexpr uint32_t kWideRow = 64;
template <class Pol>
__device__ __forceinline__ typename Pol::Acc row_sum(const typename Pol::V *s_v, uint32_t b, uint32_t e, uint32_t G)
{
  const uint32_t lane = lane_id(), sub = lane % G;
  const bool wide = G < (uint32_t)kWave && e - b > kWideRow * G;
  auto a = Pol::zero();
  if (!wide)
    for (uint32_t x = b + sub; x < e; x += G) Pol::add(a, s_v[x]);
  Pol::merge_lanes(a, (int)G);
  uint64_t m = __ballot(wide && sub == 0);
  while (m) {
    const int src = __ffsll((unsigned long long)m) - 1;
    m &= m - 1;
    const uint32_t wb = __shfl(b, src, kWave), we = __shfl(e, src, kWave);
    auto t = Pol::zero();
    for (uint32_t x = wb + lane; x < we; x += kWave) Pol::add(t, s_v[x]);
    Pol::merge_lanes(t, kWave);
    if ((int)lane == src) a = t;
  }
  return a;
}

// v into the places [b, e) of each group's row, split as in row_sum; called by
// the whole wave.  (A lane that marked a row of 2000 places alone held up the
// pull: hop SSSP over 65536 vertices in four partitions, 36 us a pull, now 13.)
template <typename V>
__device__ __forceinline__ void row_fill(V *s_v, uint32_t b, uint32_t e, uint32_t G, V v)
{
  const uint32_t lane = lane_id(), sub = lane % G;
  const bool wide = G < (uint32_t)kWave && e - b > kWideRow * G;
  if (!wide)
    for (uint32_t x = b + sub; x < e; x += G) s_v[x] = v;
  uint64_t m = __ballot(wide && sub == 0);
  while (m) {
    const int src = __ffsll((unsigned long long)m) - 1;
    m &= m - 1;
    const uint32_t wb = __shfl(b, src, kWave), we = __shfl(e, src, kWave);
    const V wv = __shfl(v, src, kWave);
    for (uint32_t x = wb + lane; x < we; x += kWave) s_v[x] = wv;
  }
}

// one segment of a long row: every thread over its staged values in order, the
// waves merged in wave order by the first thread, which gets the sum
template <class Pol, int T>
__device__ __forceinline__ typename Pol::Acc segment_sum(const typename Pol::V *s_v, uint32_t ne)
{
  using Acc = typename Pol::Acc;
  __shared__ uint64_t s_w[T / kWave];
  static_assert(sizeof(Acc) <= 8, "an accumulator fits its slot");
  auto a = Pol::zero();
  for (uint32_t x = threadIdx.x; x < ne; x += T) Pol::add(a, s_v[x]);
  Pol::merge_lanes(a, kWave);
  if (lane_id() == 0) *reinterpret_cast<Acc *>(&s_w[wave_in_block()]) = a;
  __syncthreads();
  if (threadIdx.x == 0)
    for (int j = 1; j < T / kWave; j++) Pol::merge(a, *reinterpret_cast<const Acc *>(&s_w[j]));
  return a;
}

// Sorts each block's arcs by source in place (once per graph): the columns
// come in row order, leave in source order with their row-order places in pos,
// the weights with them.  Sources below 2^bits (any below 2^32 - 1 at 31 bits);
// padding keys sort last.
template <class Block, class W, int T, int N>
__global__ void __launch_bounds__(T) k_block_sort(const Block *__restrict__ blocks, uint32_t *__restrict__ col,
                                                 W *__restrict__ cw, uint16_t *__restrict__ pos, int bits)
{
  constexpr int kPer = N / T;
  using Sort = rocprim::block_radix_sort<uint32_t, T, kPer, uint16_t>;
  __shared__ typename Sort::storage_type s_sort;
  const Block d = blocks[blockIdx.x];
  const uint32_t ne = d.e1 - d.e0, pad = bits < 31 ? 1u << bits : 0xFFFFFFFFu;
  uint32_t key[kPer];
  uint16_t at[kPer];
#pragma unroll
  for (int k = 0; k < kPer; k++) {
    const uint32_t i = threadIdx.x + k * T;
    key[k] = i < ne ? col[d.e0 + i] : pad;
    at[k] = (uint16_t)i;
  }
  Sort().sort_to_striped(key, at, s_sort, 0, bits + 1);
  W w[kPer];
  if (cw) {
#pragma unroll
    for (int k = 0; k < kPer; k++) w[k] = threadIdx.x + k * T < ne ? cw[d.e0 + at[k]] : W(0);
  }
  __syncthreads();  // every weight is read before one is written
#pragma unroll
  for (int k = 0; k < kPer; k++) {
    const uint32_t i = threadIdx.x + k * T;
    if (i < ne) {
      col[d.e0 + i] = key[k];
      pos[d.e0 + i] = at[k];
      if (cw) cw[d.e0 + i] = w[k];
    }
  }
}

}  // namespace grd
