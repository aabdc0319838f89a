// mlp.hip -- schedule selector: MLP 16 -> 64 -> 64 -> 4 (ReLU), trained and
// evaluated by these kernels on the GPU.
//
// Parameter layout (5,508 values, FP32 masters during training, BF16 for
// inference):
//   W1[64][16]  b1[64]  W2[64][64]  b2[64]  W3[4][64]  b3[4]
// Output o indexes the schedule option (bit 0 pull, bit 1 dense sync).  The
// network is trained as a classifier of the fastest option with a
// cost-weighted softmax cross-entropy: sample weight = clamp((t_max -
// t_min) / t_min, 0.1, 10), so iterations where the choice matters weigh
// more.  The forward pass of training reads BF16-rounded weights so that training and
// inference see the same network.  The selector only picks the schedule of
// an iteration: every option computes the same result.
#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstring>
#include <string>
#include <vector>

#include "grd_device.hpp"
#include "grd_internal.hpp"
#include "grd_ops.hpp"

namespace grd {

constexpr int kIn = 16, kH = 64, kOut = 4;
constexpr int oW1 = 0, oB1 = oW1 + kH * kIn, oW2 = oB1 + kH, oB2 = oW2 + kH * kH, oW3 = oB2 + kH, oB3 = oW3 + kOut * kH;
constexpr int kParams = oB3 + kOut;  // 5508

// ---- staging of the allocation-free inference (grd_selector_infer_noalloc) ----
//
// Features and logits of up to kInferMax samples, in a file-scope device
// array: every GPU the library runs on holds its own copy (320 KB) until the
// process ends.  In host code `scratch` names a host-side stand-in, not the
// device copy: its device address is taken once per device by
// mlp_scratch_init (from grd_create, with that device current) and only that
// address is used.  Calls on one GPU share the array: calls that overlap on
// one GPU race.
constexpr uint32_t kInferMax = 4096;
static __device__ __align__(256) float scratch[kInferMax * (kIn + kOut)];
constexpr int kMaxDevices = 64;
static float *g_scratch_ptr[kMaxDevices] = {};

grd_status mlp_scratch_init(int device)
{
  if (device < 0 || device >= kMaxDevices) return fail(GRD_ERR_ARG, "selector scratch: device id beyond 63");
  if (g_scratch_ptr[device]) return GRD_OK;
  float *ptr = nullptr;
  GRD_HIP(hipGetSymbolAddress((void **)&ptr, HIP_SYMBOL(scratch)));
  if (!ptr) return fail(GRD_ERR_HIP, "selector scratch: no device address");
  g_scratch_ptr[device] = ptr;
  return GRD_OK;
}

__host__ __device__ __forceinline__ float bf16_to_f32(uint16_t h)
{
  uint32_t u = (uint32_t)h << 16;
  float f;
  memcpy(&f, &u, 4);
  return f;
}
// round to nearest even
__host__ __device__ __forceinline__ uint16_t f32_to_bf16(float f)
{
  uint32_t u;
  memcpy(&u, &f, 4);
  if ((u & 0x7F800000u) == 0x7F800000u) return (uint16_t)(u >> 16);  // inf / nan
  uint32_t r = u + 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(r >> 16);
}

// forward of one sample by one wave; returns logits in lanes 0..3 (value
// broadcast to all lanes through the out array).  Weights are read through
// `wf` (FP32) or `wb` (BF16) depending on which pointer is non-null.
struct Fwd {
  float h1, h2;      // this lane's hidden units (post-ReLU)
  float logit[kOut];  // all lanes hold all logits
};

template <bool BF16>
__device__ __forceinline__ float wload(const float *wf, const uint16_t *wb, int i)
{
  if constexpr (BF16) return bf16_to_f32(wb[i]);
  else return wf[i];
}

template <bool BF16>
__device__ __forceinline__ Fwd forward_wave(const float *wf, const uint16_t *wb, const float *x, float *s_h1)
{
  const int j = lane_id();
  Fwd r;
  float a = wload<BF16>(wf, wb, oB1 + j);
#pragma unroll
  for (int i = 0; i < kIn; i++) a += wload<BF16>(wf, wb, oW1 + j * kIn + i) * x[i];
  r.h1 = a > 0.0f ? a : 0.0f;
  s_h1[j] = r.h1;
  __syncthreads();  // callers keep whole blocks in step
  float b = wload<BF16>(wf, wb, oB2 + j);
  for (int k = 0; k < kH; k++) b += wload<BF16>(wf, wb, oW2 + j * kH + k) * s_h1[k];
  r.h2 = b > 0.0f ? b : 0.0f;
#pragma unroll
  for (int o = 0; o < kOut; o++) r.logit[o] = wave_sum(wload<BF16>(wf, wb, oW3 + o * kH + j) * r.h2);
#pragma unroll
  for (int o = 0; o < kOut; o++) r.logit[o] += wload<BF16>(wf, wb, oB3 + o);
  return r;
}

// Forward + backward over samples [0, n): a wave takes samples w, w + W, ...,
// lane j owning hidden unit j.  The weights a lane needs -- its rows of W1 and
// W2 and its column of W2 and W3 -- and its gradients stay in registers for all
// of its samples; hidden values and their gradients pass between the lanes
// through a wave's own LDS row (16-byte broadcast reads).  The four waves of a
// block are summed in wave order, and each block writes one partial gradient
// and loss (kPart floats), which the caller sums in block order: no atomics,
// and the result does not depend on scheduling.  20003 samples: 398 -> 61 us
// (64 blocks, weights through the caches for each sample, 5508 atomics a wave);
// bound now by each lane's chains of 64 dependent adds, one wave per SIMD.
//
// Partial layout: W1 and W2 transposed ([input][unit]), so that lanes write
// neighbouring words; the rest as the parameters; the loss last.
constexpr int kPart = kParams + 1;
__host__ __device__ __forceinline__ int part_to_param(int p)
{
  if (p < oB1) return oW1 + (p % kH) * kIn + p / kH;
  if (p >= oW2 && p < oB2) return oW2 + ((p - oW2) % kH) * kH + (p - oW2) / kH;
  return p;
}

__device__ __forceinline__ void wave_lds_order()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

template <bool BF16>
__global__ void __launch_bounds__(kBlock, 1) k_mlp_grad(const float *__restrict__ wf, const uint16_t *__restrict__ wb,
                                                        const float *__restrict__ feat,
                                                        const uint32_t *__restrict__ label,
                                                        const float *__restrict__ sw, const uint32_t *__restrict__ idx,
                                                        uint32_t n, float *__restrict__ part)
{
  __shared__ __align__(16) float s_h1[kWavesPerBlock][kH];
  __shared__ __align__(16) float s_d2[kWavesPerBlock][kH];
  __shared__ float s_part[kPart];
  const int j = lane_id(), wv = __builtin_amdgcn_readfirstlane(wave_in_block());
  const uint32_t nwaves = gridDim.x * kWavesPerBlock;
  float w1[kIn], w2r[kH], w2c[kH], w3[kOut];
#pragma unroll
  for (int i = 0; i < kIn; i++) w1[i] = wload<BF16>(wf, wb, oW1 + j * kIn + i);
#pragma unroll
  for (int k = 0; k < kH; k++) w2r[k] = wload<BF16>(wf, wb, oW2 + j * kH + k);
#pragma unroll
  for (int k = 0; k < kH; k++) w2c[k] = wload<BF16>(wf, wb, oW2 + k * kH + j);
#pragma unroll
  for (int o = 0; o < kOut; o++) w3[o] = wload<BF16>(wf, wb, oW3 + o * kH + j);
  const float b1 = wload<BF16>(wf, wb, oB1 + j), b2 = wload<BF16>(wf, wb, oB2 + j);
  float b3[kOut];
#pragma unroll
  for (int o = 0; o < kOut; o++) b3[o] = wload<BF16>(wf, wb, oB3 + o);
  float gW2[kH], gW1[kIn], gW3[kOut];
  float gb1 = 0.0f, gb2 = 0.0f, gb3 = 0.0f, lsum = 0.0f;
#pragma unroll
  for (int k = 0; k < kH; k++) gW2[k] = 0.0f;
#pragma unroll
  for (int i = 0; i < kIn; i++) gW1[i] = 0.0f;
#pragma unroll
  for (int o = 0; o < kOut; o++) gW3[o] = 0.0f;
  for (uint32_t t = blockIdx.x * kWavesPerBlock + wv; t < n; t += nwaves) {
    const uint32_t si = idx ? (uint32_t)__builtin_amdgcn_readfirstlane(idx[t]) : t;
    const uint32_t y = label[si];
    const float wgt = sw ? sw[si] : 1.0f;
    float x[kIn];
#pragma unroll
    for (int i = 0; i < kIn; i++) x[i] = feat[(uint64_t)si * kIn + i];
    float a = b1;
#pragma unroll
    for (int i = 0; i < kIn; i++) a += w1[i] * x[i];
    const float h1 = a > 0.0f ? a : 0.0f;
    s_h1[wv][j] = h1;
    wave_lds_order();
    float h[kH];
#pragma unroll
    for (int k = 0; k < kH; k += 4) {
      const float4 v = *reinterpret_cast<const float4 *>(&s_h1[wv][k]);
      h[k] = v.x;
      h[k + 1] = v.y;
      h[k + 2] = v.z;
      h[k + 3] = v.w;
    }
    float b = b2;
#pragma unroll
    for (int k = 0; k < kH; k++) b += w2r[k] * h[k];
    const float h2 = b > 0.0f ? b : 0.0f;
    float lg[kOut];
#pragma unroll
    for (int o = 0; o < kOut; o++) lg[o] = wave_sum(w3[o] * h2) + b3[o];
    // softmax cross-entropy
    float mx = lg[0];
#pragma unroll
    for (int o = 1; o < kOut; o++) mx = lg[o] > mx ? lg[o] : mx;
    float den = 0.0f, p[kOut];
#pragma unroll
    for (int o = 0; o < kOut; o++) {
      p[o] = expf(lg[o] - mx);
      den += p[o];
    }
    float py = 0.0f, dl[kOut];
#pragma unroll
    for (int o = 0; o < kOut; o++) {
      p[o] /= den;
      if (o == (int)y) py = p[o];
      dl[o] = wgt * (p[o] - (o == (int)y ? 1.0f : 0.0f));
    }
    lsum += wgt * (-logf(fmaxf(py, 1e-30f)));
    // backward
    float d2 = 0.0f;
#pragma unroll
    for (int o = 0; o < kOut; o++) {
      gW3[o] += dl[o] * h2;  // W3[o][j]
      d2 += w3[o] * dl[o];
      if (j == o) gb3 += dl[o];
    }
    d2 = h2 > 0.0f ? d2 : 0.0f;
    gb2 += d2;
#pragma unroll
    for (int k = 0; k < kH; k++) gW2[k] += d2 * h[k];  // W2[j][k]
    s_d2[wv][j] = d2;
    wave_lds_order();
    float d1 = 0.0f;
#pragma unroll
    for (int k = 0; k < kH; k += 4) {
      const float4 v = *reinterpret_cast<const float4 *>(&s_d2[wv][k]);
      d1 += w2c[k] * v.x;
      d1 += w2c[k + 1] * v.y;
      d1 += w2c[k + 2] * v.z;
      d1 += w2c[k + 3] * v.w;
    }
    d1 = h1 > 0.0f ? d1 : 0.0f;
    gb1 += d1;
#pragma unroll
    for (int i = 0; i < kIn; i++) gW1[i] += d1 * x[i];
    wave_lds_order();  // the rows are rewritten by the next sample
  }
  for (int w = 0; w < kWavesPerBlock; w++) {
    if (wv == w) {
      auto put = [&](int p, float v) { s_part[p] = w ? s_part[p] + v : v; };
#pragma unroll
      for (int i = 0; i < kIn; i++) put(oW1 + i * kH + j, gW1[i]);
      put(oB1 + j, gb1);
#pragma unroll
      for (int k = 0; k < kH; k++) put(oW2 + k * kH + j, gW2[k]);
      put(oB2 + j, gb2);
#pragma unroll
      for (int o = 0; o < kOut; o++) put(oW3 + o * kH + j, gW3[o]);
      if (j < kOut) put(oB3 + j, gb3);
      if (j == 0) put(kParams, lsum);
    }
    __syncthreads();
  }
  for (int p = threadIdx.x; p < kPart; p += kBlock) part[(uint64_t)blockIdx.x * kPart + p] = s_part[p];
}

// blocks of k_mlp_grad for n samples: a block per CU at most, a sample per wave
// at least
static uint32_t grad_blocks(const grd_ctx *ctx, uint64_t n)
{
  return (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>((n + kWavesPerBlock - 1) / kWavesPerBlock,
                                                            (uint64_t)ctx->num_cus));
}

// sum of partial entry p over the blocks, in a fixed order (four chains, so
// that the loads overlap)
__device__ __forceinline__ float part_sum(const float *__restrict__ part, uint32_t nblk, int p)
{
  float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  uint32_t b = 0;
  for (; b + 4 <= nblk; b += 4)
#pragma unroll
    for (uint32_t q = 0; q < 4; q++) s[q] += part[(uint64_t)(b + q) * kPart + p];
  for (; b < nblk; b++) s[0] += part[(uint64_t)b * kPart + p];
  return (s[0] + s[1]) + (s[2] + s[3]);
}

// gradient and loss of a batch from its partials into pinned memory (the loss
// last), each workgroup, a wave, reporting its end in its flag (with two
// copies back and a stream synchronisation 20003 samples took 237 us, now 194)
__global__ void __launch_bounds__(kWave) k_mlp_reduce(const float *__restrict__ part, uint32_t nblk,
                                                      float *__restrict__ out, uint32_t *flags, uint32_t seq)
{
  const int p = blockIdx.x * kWave + threadIdx.x;
  if (p < kPart) {
    const float g = part_sum(part, nblk, p);
    out[p == kParams ? kParams : part_to_param(p)] = g;
  }
  if (threadIdx.x == 0)
    __hip_atomic_store(flags + blockIdx.x, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Adam step on FP32 masters from a batch's partials; refreshes the BF16 copy
// and adds the batch's loss
__global__ void __launch_bounds__(kWave) k_mlp_adam(float *__restrict__ w, float *__restrict__ m1,
                                                    float *__restrict__ m2, const float *__restrict__ part,
                                                    uint32_t nblk, uint16_t *__restrict__ wb, float *__restrict__ loss,
                                                    float scale, float lr, float b1, float b2, float c1, float c2)
{
  const int p = blockIdx.x * kWave + threadIdx.x;
  if (p >= kPart) return;
  const float g = part_sum(part, nblk, p);
  if (p == kParams) {
    *loss += g;
    return;
  }
  const int i = part_to_param(p);
  const float gi = g * scale;
  m1[i] = b1 * m1[i] + (1.0f - b1) * gi;
  m2[i] = b2 * m2[i] + (1.0f - b2) * gi * gi;
  float mh = m1[i] / c1, vh = m2[i] / c2;
  w[i] -= lr * mh / (sqrtf(vh) + 1e-8f);
  wb[i] = f32_to_bf16(w[i]);
}

// Inference with the BF16 weights, logits[n*4]: a workgroup takes 16 samples,
// wave u the hidden units 16u to 16u + 15 of both layers, as FP32 matrix
// products (16x16x4) of unit rows by sample columns.  The order of the inputs
// within a product is free as long as both operands agree on it, so lane group
// q takes the inputs 4q.. (layer 1) and 16q.. (layer 2): each lane's weights and
// values are whole 16-byte loads, and the lane that computes a unit's four
// results stores them as one.  The last layer's four outputs are summed in the
// lanes that hold the units, then over the lane groups and the waves.
//
// features and logits may lie in pinned host memory (one coalesced read and one
// coalesced write per workgroup); with flags, workgroup b then reports its end
// there.  2000 samples: a wave per sample, weights through the caches for each,
// took 6 us and each of the two copies around it as long again; a call took 43
// us.  Now 19 us a call, of which the kernel is
// about 6: a PCIe read, the tile, a PCIe write (1 sample 11 us, 4096 28 us).
typedef float Vec4 __attribute__((ext_vector_type(4)));
constexpr int kTileS = 16;

__device__ __forceinline__ Vec4 bf16x4(const uint16_t *__restrict__ p)
{
  const uint2 q = *reinterpret_cast<const uint2 *>(p);
  return Vec4{__uint_as_float(q.x << 16), __uint_as_float(q.x & 0xFFFF0000u), __uint_as_float(q.y << 16),
              __uint_as_float(q.y & 0xFFFF0000u)};
}

__global__ void __launch_bounds__(kBlock) k_mlp_infer(const uint16_t *__restrict__ wb, const float *__restrict__ feat,
                                                      uint32_t n, float *__restrict__ logits, uint32_t *flags,
                                                      uint32_t seq)
{
  static_assert(kBlock == kTileS * kIn && kWavesPerBlock * 16 == kH && kIn == 16 && kOut == 4, "tile shapes");
  static_assert(oB1 % 4 == 0 && oW2 % 4 == 0 && oB2 % 4 == 0 && oW3 % 4 == 0, "weights are loaded four at a time");
  __shared__ __align__(16) float s_x[kTileS * kIn];
  __shared__ __align__(16) float s_h[kTileS][kH + 4];  // (rows four banks apart)
  __shared__ __align__(16) float s_o[kWavesPerBlock][kTileS][kOut];
  const int l = lane_id(), i = l % 16, q = l / 16, u = wave_in_block() * 16, t = threadIdx.x;
  const Vec4 w1 = bf16x4(wb + oW1 + (u + i) * kIn + 4 * q);
  Vec4 w2[4], w3[kOut];
#pragma unroll
  for (int k = 0; k < 4; k++) w2[k] = bf16x4(wb + oW2 + (u + i) * kH + 16 * q + 4 * k);
#pragma unroll
  for (int o = 0; o < kOut; o++) w3[o] = bf16x4(wb + oW3 + o * kH + u + 4 * q);
  const Vec4 b1 = bf16x4(wb + oB1 + u + 4 * q), b2 = bf16x4(wb + oB2 + u + 4 * q);
  const float b3 = bf16_to_f32(wb[oB3 + t % kOut]);
  const uint32_t tiles = (uint32_t)(((uint64_t)n + kTileS - 1) / kTileS);
  for (uint32_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    const uint64_t x0 = (uint64_t)tile * kTileS * kIn;
    s_x[t] = x0 + t < (uint64_t)n * kIn ? feat[x0 + t] : 0.0f;
    __syncthreads();
    const Vec4 x = *reinterpret_cast<const Vec4 *>(&s_x[i * kIn + 4 * q]);
    // units u + 4q + (0..3) of sample i, in two sums (four in the second layer):
    // shorter chains, and a smaller rounding error than one chain's
    const Vec4 zero{};
    Vec4 a = __builtin_amdgcn_mfma_f32_16x16x4f32(w1[0], x[0], b1, 0, 0, 0);
    Vec4 c = __builtin_amdgcn_mfma_f32_16x16x4f32(w1[1], x[1], zero, 0, 0, 0);
    a = __builtin_amdgcn_mfma_f32_16x16x4f32(w1[2], x[2], a, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(w1[3], x[3], c, 0, 0, 0);
    a += c;
#pragma unroll
    for (int k = 0; k < 4; k++) a[k] = a[k] > 0.0f ? a[k] : 0.0f;
    *reinterpret_cast<Vec4 *>(&s_h[i][u + 4 * q]) = a;
    __syncthreads();
    Vec4 s[4] = {b2, zero, zero, zero};
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const Vec4 h = *reinterpret_cast<const Vec4 *>(&s_h[i][16 * q + 4 * j]);
#pragma unroll
      for (int k = 0; k < 4; k++) s[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(w2[j][k], h[k], s[j], 0, 0, 0);
    }
    a = (s[0] + s[1]) + (s[2] + s[3]);
    Vec4 o4;
#pragma unroll
    for (int o = 0; o < kOut; o++) {
      float v = 0.0f;
#pragma unroll
      for (int k = 0; k < 4; k++) v += w3[o][k] * (a[k] > 0.0f ? a[k] : 0.0f);
      v += __shfl_xor(v, 16, kWave);
      v += __shfl_xor(v, 32, kWave);
      o4[o] = v;
    }
    if (q == 0) *reinterpret_cast<Vec4 *>(s_o[wave_in_block()][i]) = o4;
    __syncthreads();
    if (t < kTileS * kOut) {  // (the first wave)
      float v = b3;
#pragma unroll
      for (int w = 0; w < kWavesPerBlock; w++) v += s_o[w][t / kOut][t % kOut];
      const uint64_t at = (uint64_t)tile * kTileS * kOut + t;
      if (at < (uint64_t)n * kOut) logits[at] = v;
    }
  }
  if (flags && t == 0) __hip_atomic_store(flags + blockIdx.x, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// workgroups of k_mlp_infer: one per tile up to four per CU
static uint32_t infer_blocks(const grd_ctx *ctx, uint64_t n)
{
  return (uint32_t)std::min<uint64_t>((n + kTileS - 1) / kTileS, 4ull * (uint64_t)std::max(1, ctx->num_cus));
}

// per-iteration selection: one wave; writes 4 logits + argmax to out[0..4]
__global__ void k_mlp_select(const uint16_t *__restrict__ wb, const float *__restrict__ feat, float *__restrict__ out)
{
  __shared__ float s_h1[kWavesPerBlock][kH];
  float x[kIn];
#pragma unroll
  for (int i = 0; i < kIn; i++) x[i] = feat[i];
  Fwd r = forward_wave<true>(nullptr, wb, x, s_h1[wave_in_block()]);
  if (threadIdx.x == 0) {
    int best = 0;
    for (int o = 0; o < kOut; o++) {
      out[o] = r.logit[o];
      if (r.logit[o] > r.logit[best]) best = o;
    }
    out[4] = (float)best;
  }
}

// The features of the superstep that just ended: x holds those of the graph
// and the algorithm, the others come from the counters (the same formulas as
// make_features on the host).
struct SelInputs {
  double n, m, P, avg_deg, prev_frontier;
  float x[kIn];
};

// The counters of a superstep to the host (as k_publish of bsp.hip) together
// with the next decision, 4 logits and the argmax in sel.  All
// weights are in flight before the counters are looked at, and each lane
// computes one feature, so that the doubles' divisions and logarithms run side
// by side (one thread after another, and a launch of its own, took 5 us more).
// Every wave computes the features and the first layer; of the second, wave w
// sums the inputs 16w to 16w + 15 of every unit, two 16-byte loads and a chain
// of 16 adds a lane instead of eight and 64 (with the single release of
// publish_seq: 10.1 -> 8.1 us).
__global__ void __launch_bounds__(kBlock) k_mlp_publish(const uint16_t *__restrict__ wb, Counters *cnt, Shares sh,
                                                        SelInputs in, Counters *host, uint32_t *host_seq, uint32_t seq)
{
  __shared__ float s_x[kWavesPerBlock][kIn];
  __shared__ __align__(16) float s_h1[kWavesPerBlock][kH];
  __shared__ float s_b[kWavesPerBlock][kH];
  const int j = lane_id(), wv = __builtin_amdgcn_readfirstlane(wave_in_block());
  constexpr int kPer = kH / kWavesPerBlock;  // inputs of the second layer per wave
  union Row {
    uint4 v[2];
    uint16_t h[16];
  } w1, w2;
  static_assert(kIn == 16 && kPer == 16 && (oW2 * 2) % 16 == 0, "weight rows are two 16-byte units");
  const uint4 *r1 = reinterpret_cast<const uint4 *>(wb + oW1 + j * kIn);
  const uint4 *r2 = reinterpret_cast<const uint4 *>(wb + oW2 + j * kH + wv * kPer);
#pragma unroll
  for (int i = 0; i < 2; i++) w1.v[i] = r1[i];
#pragma unroll
  for (int i = 0; i < 2; i++) w2.v[i] = r2[i];
  const float b1 = bf16_to_f32(wb[oB1 + j]), b2 = bf16_to_f32(wb[oB2 + j]);
  float w3[kOut], b3[kOut];
#pragma unroll
  for (int o = 0; o < kOut; o++) {
    w3[o] = bf16_to_f32(wb[oW3 + o * kH + j]);
    b3[o] = bf16_to_f32(wb[oB3 + o]);
  }
  // the counters' copy; sel follows below
  constexpr uint32_t kSel0 = offsetof(Counters, sel) / 8, kSel1 = kSel0 + sizeof(Counters::sel) / 8;
  static_assert(offsetof(Counters, sel) % 8 == 0 && sizeof(Counters::sel) % 8 == 0, "sel is whole words");
  const CounterWords words = counter_words(cnt);
  const FrontierCounts fc = sum_shares(sh);
  copy_counters(words, host, fc, kSel0, kSel1);
  {
    const double fr = (double)fc.frontier, fe = (double)fc.edges;
    const double m = in.m > 1.0 ? in.m : 1.0;
    double num = 0.0, den = 1.0;
    if (j == 1) num = fr, den = in.n;
    if (j == 2) num = fe, den = m;
    if (j == 4) num = (double)fc.dirty, den = in.P;
    if (j == 5) num = (double)fc.maxdeg, den = fe + 1.0;
    if (j == 6 && fr > 0) num = fe, den = fr * fmax(1e-9, in.avg_deg * 4.0);
    if (j == 12) num = in.prev_frontier > 0 ? fr : 1.0, den = in.prev_frontier > 0 ? in.prev_frontier : 1.0;
    double q = num / den;
    const double lg = log2(j == 0 ? 1.0 + fr : j == 3 ? 1.0 + fe : j == 12 ? fmax(q, 1e-9) : 1.0);
    if (j == 0) q = lg / 32.0;
    if (j == 3) q = lg / 40.0;
    if (j == 6) q = fmin(4.0, q);
    if (j == 12) q = fmax(-1.0, fmin(1.0, lg / 16.0)) * 0.5 + 0.5;
    const bool counted = j <= 6 || j == 12;
    if (j < kIn) s_x[wv][j] = counted ? (float)q : in.x[j];
  }
  wave_lds_order();
  float a = b1;
#pragma unroll
  for (int i = 0; i < kIn; i++) a += bf16_to_f32(w1.h[i]) * s_x[wv][i];
  s_h1[wv][j] = a > 0.0f ? a : 0.0f;
  wave_lds_order();
  float b = wv == 0 ? b2 : 0.0f;
#pragma unroll
  for (int k = 0; k < kPer; k++) b += bf16_to_f32(w2.h[k]) * s_h1[wv][wv * kPer + k];
  s_b[wv][j] = b;
  __syncthreads();
  if (wv == 0) {
#pragma unroll
    for (int w = 1; w < kWavesPerBlock; w++) b += s_b[w][j];
    const float h2 = b > 0.0f ? b : 0.0f;
    float lg[kOut];
#pragma unroll
    for (int o = 0; o < kOut; o++) lg[o] = wave_sum(w3[o] * h2) + b3[o];
    if (j == 0) {
      int best = 0;
#pragma unroll
      for (int o = 1; o < kOut; o++)
        if (lg[o] > lg[best]) best = o;
#pragma unroll
      for (int o = 0; o < kOut; o++) host->sel[o] = lg[o];
      host->sel[4] = (float)best;
    }
  }
  publish_seq(host_seq, seq);
  zero_counters(cnt, sh);
}

// ------------------------------------------------------------------------

static grd_status sel_buffers(grd_ctx *ctx)
{
  if (!ctx->sel_out) {
    GRD_TRY(device_malloc(ctx->device, (void **)&ctx->sel_out, 32 * sizeof(float)));
    GRD_HIP(hipHostMalloc((void **)&ctx->sel_out_host, 32 * sizeof(float), hipHostMallocDefault));
  }
  return GRD_OK;
}

// pinned: features and logits of kInferMax samples, and a flag per workgroup
// (allocated with the weights, 20 us)
static grd_status infer_stage(grd_ctx *ctx)
{
  constexpr size_t kFlags = kInferMax / kTileS;
  if (!ctx->sel_stage) {
    const size_t bytes = ((size_t)kInferMax * (kIn + kOut) + kFlags) * 4;
    GRD_HIP(hipHostMalloc((void **)&ctx->sel_stage, bytes, hipHostMallocDefault));
    memset(ctx->sel_stage, 0, bytes);
  }
  return GRD_OK;
}

static void decode_logits(const float *o, int *option, float *margin)
{
  int best = (int)o[4];
  float second = -1e30f;
  for (int k = 0; k < kOut; k++)
    if (k != best) second = std::max(second, o[k]);
  *option = best;
  *margin = o[best] - second;
}

grd_status mlp_publish(grd_state *s, uint64_t prev_frontier)
{
  grd_graph *g = s->g;
  grd_ctx *ctx = g->ctx;
  SelInputs in{(double)g->n, (double)g->m, (double)g->P, g->avg_degree, (double)prev_frontier, {}};
  make_features(s, in.x);  // (those of the counters are computed on the device)
  hipLaunchKernelGGL(k_mlp_publish, dim3(1), dim3(kBlock), 0, ctx->stream, ctx->sel_w, s->cnt, shares(s), in, s->hcnt,
                     host_seq(s->hcnt), ++s->cnt_seq);
  GRD_HIP(hipGetLastError());
  counters_at_start(s, true);
  return GRD_OK;
}

void mlp_select_read(const grd_state *s, int *option, float *margin) { decode_logits(s->hcnt->sel, option, margin); }

grd_status mlp_select(grd_ctx *ctx, const float *feat16, int *option, float *margin)
{
  GRD_TRY(sel_buffers(ctx));
  memcpy(ctx->sel_out_host + 8, feat16, 16 * sizeof(float));
  GRD_HIP(hipMemcpyAsync(ctx->sel_out + 8, ctx->sel_out_host + 8, 16 * sizeof(float), hipMemcpyHostToDevice,
                         ctx->stream));
  hipLaunchKernelGGL(k_mlp_select, dim3(1), dim3(kWave), 0, ctx->stream, ctx->sel_w, ctx->sel_out + 8, ctx->sel_out);
  GRD_HIP(hipGetLastError());
  GRD_HIP(hipMemcpyAsync(ctx->sel_out_host, ctx->sel_out, 8 * sizeof(float), hipMemcpyDeviceToHost, ctx->stream));
  GRD_HIP(hipStreamSynchronize(ctx->stream));
  decode_logits(ctx->sel_out_host, option, margin);
  return GRD_OK;
}

}  // namespace grd

using namespace grd;

extern "C" {

grd_status grd_selector_load(grd_ctx *ctx, const uint16_t *w, uint64_t count, float min_margin)
{
  if (!ctx || !w) return fail(GRD_ERR_ARG, "grd_selector_load: NULL argument");
  if (count != (uint64_t)kParams)
    return fail(GRD_ERR_ARG, "grd_selector_load: expected " + std::to_string(kParams) + " BF16 weights");
  GRD_HIP(hipSetDevice(ctx->device));
  if (!ctx->sel_w) GRD_TRY(device_malloc(ctx->device, (void **)&ctx->sel_w, kParams * sizeof(uint16_t)));
  GRD_HIP(hipMemcpy(ctx->sel_w, w, kParams * sizeof(uint16_t), hipMemcpyHostToDevice));
  GRD_TRY(infer_stage(ctx));
  ctx->sel_loaded = true;
  ctx->sel_margin = min_margin;
  return GRD_OK;
}

grd_status grd_selector_train(grd_ctx *ctx, const float *feat, const uint32_t *label, const float *cost, uint64_t n,
                              uint32_t epochs, uint32_t batch, float lr, uint64_t seed, uint16_t *out_bf16,
                              float *final_loss)
{
  if (!ctx || !feat || !label || n == 0 || n > (1ull << 31) || batch == 0)
    return fail(GRD_ERR_ARG, "grd_selector_train: bad argument");
  for (uint64_t i = 0; i < n; i++)
    if (label[i] >= (uint32_t)kOut) return fail(GRD_ERR_ARG, "grd_selector_train: label out of range");
  GRD_HIP(hipSetDevice(ctx->device));
  hipStream_t st = ctx->stream;
  // sample weights from the per-option costs
  std::vector<float> sw(n, 1.0f);
  if (cost)
    for (uint64_t i = 0; i < n; i++) {
      float mn = cost[i * 4], mx = cost[i * 4];
      for (int o = 1; o < 4; o++) {
        mn = std::min(mn, cost[i * 4 + o]);
        mx = std::max(mx, cost[i * 4 + o]);
      }
      float r = mn > 0 ? (mx - mn) / mn : 1.0f;
      sw[i] = std::min(10.0f, std::max(0.1f, r));
    }
  // He initialisation from a seeded SplitMix stream
  std::vector<float> w0(kParams, 0.0f);
  uint64_t z = seed ? seed : 0x9E3779B97F4A7C15ull;
  auto uni = [&]() {
    z += 0x9E3779B97F4A7C15ull;
    uint64_t x = z;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    x ^= x >> 31;
    return (double)(x >> 11) * (1.0 / 9007199254740992.0);
  };
  auto init = [&](int off, int cnt, int fan_in) {
    double a = std::sqrt(6.0 / fan_in);
    for (int i = 0; i < cnt; i++) w0[off + i] = (float)((uni() * 2.0 - 1.0) * a);
  };
  init(oW1, kH * kIn, kIn);
  init(oW2, kH * kH, kH);
  init(oW3, kOut * kH, kH);
  DevMem mem(ctx);
  float *dw, *dm1, *dm2, *dpart, *dfeat, *dsw, *dloss;
  uint32_t *dlab, *didx;
  uint16_t *dwb;
  GRD_TRY(mem.alloc_n(&dw, kParams));
  GRD_TRY(mem.alloc_n(&dm1, kParams));
  GRD_TRY(mem.alloc_n(&dm2, kParams));
  GRD_TRY(mem.alloc_n(&dpart, (uint64_t)grad_blocks(ctx, std::min<uint64_t>(batch, n)) * kPart));
  GRD_TRY(mem.alloc_n(&dwb, kParams));
  GRD_TRY(mem.alloc_n(&dfeat, n * kIn));
  GRD_TRY(mem.alloc_n(&dsw, n));
  GRD_TRY(mem.alloc_n(&dlab, n));
  GRD_TRY(mem.alloc_n(&didx, n));
  GRD_TRY(mem.alloc_n(&dloss, 1));
  std::vector<uint16_t> wb0(kParams);
  for (int i = 0; i < kParams; i++) wb0[i] = f32_to_bf16(w0[i]);
  GRD_HIP(hipMemcpy(dw, w0.data(), kParams * 4, hipMemcpyHostToDevice));
  GRD_HIP(hipMemcpy(dwb, wb0.data(), kParams * 2, hipMemcpyHostToDevice));
  GRD_HIP(hipMemsetAsync(dm1, 0, kParams * 4, st));
  GRD_HIP(hipMemsetAsync(dm2, 0, kParams * 4, st));
  GRD_HIP(hipMemcpy(dfeat, feat, n * kIn * 4, hipMemcpyHostToDevice));
  GRD_HIP(hipMemcpy(dsw, sw.data(), n * 4, hipMemcpyHostToDevice));
  GRD_HIP(hipMemcpy(dlab, label, n * 4, hipMemcpyHostToDevice));
  std::vector<uint32_t> perm(n);
  for (uint64_t i = 0; i < n; i++) perm[i] = (uint32_t)i;
  const float b1 = 0.9f, b2 = 0.999f;
  uint64_t step = 0;
  float last = 0.0f;
  for (uint32_t ep = 0; ep < epochs; ep++) {
    for (uint64_t i = n - 1; i > 0; i--) std::swap(perm[i], perm[(uint64_t)(uni() * (double)(i + 1)) % (i + 1)]);
    GRD_HIP(hipMemcpyAsync(didx, perm.data(), n * 4, hipMemcpyHostToDevice, st));
    GRD_HIP(hipMemsetAsync(dloss, 0, 4, st));
    for (uint64_t b0 = 0; b0 < n; b0 += batch) {
      uint32_t nb = (uint32_t)std::min<uint64_t>(batch, n - b0);
      const uint32_t grid = grad_blocks(ctx, nb);
      hipLaunchKernelGGL(k_mlp_grad<true>, dim3(grid), dim3(kBlock), 0, st, dw, dwb, dfeat, dlab, dsw, didx + b0, nb,
                         dpart);
      step++;
      float c1 = 1.0f - std::pow(b1, (float)step), c2 = 1.0f - std::pow(b2, (float)step);
      hipLaunchKernelGGL(k_mlp_adam, dim3((kPart + kWave - 1) / kWave), dim3(kWave), 0, st, dw, dm1, dm2, dpart, grid,
                         dwb, dloss, 1.0f / (float)nb, lr, b1, b2, c1, c2);
    }
    GRD_HIP(hipGetLastError());
    float ls = 0.0f;
    GRD_HIP(hipMemcpyAsync(&ls, dloss, 4, hipMemcpyDeviceToHost, st));
    GRD_HIP(hipStreamSynchronize(st));
    last = ls / (float)n;
  }
  std::vector<uint16_t> wb(kParams);
  GRD_HIP(hipMemcpyAsync(wb.data(), dwb, kParams * 2, hipMemcpyDeviceToHost, st));
  GRD_HIP(hipStreamSynchronize(st));
  if (out_bf16) memcpy(out_bf16, wb.data(), kParams * 2);
  if (final_loss) *final_loss = last;
  return grd_selector_load(ctx, wb.data(), kParams, ctx->sel_margin);
}

grd_status grd_selector_infer(grd_ctx *ctx, const float *feat, uint64_t n, float *logits)
{
  if (!ctx || !feat || !logits || n == 0) return fail(GRD_ERR_ARG, "grd_selector_infer: bad argument");
  if (!ctx->sel_loaded) return fail(GRD_ERR_STATE, "grd_selector_infer: no weights loaded");
  GRD_HIP(hipSetDevice(ctx->device));
  if (n <= kInferMax) {
    // the kernel reads the features from, and writes the logits to, pinned memory
    float *x = ctx->sel_stage;
    float *out = x + (size_t)kInferMax * kIn;
    uint32_t *flags = reinterpret_cast<uint32_t *>(out + (size_t)kInferMax * kOut);
    memcpy(x, feat, n * kIn * 4);
    const uint32_t grid = infer_blocks(ctx, n), seq = ++ctx->sel_seq;
    hipLaunchKernelGGL(k_mlp_infer, dim3(grid), dim3(kBlock), 0, ctx->stream, ctx->sel_w, x, (uint32_t)n, out, flags,
                       seq);
    GRD_HIP(hipGetLastError());
    for (uint32_t b = 0; b < grid; b++) GRD_TRY(wait_pinned(ctx, flags + b, seq));
    memcpy(logits, out, n * kOut * 4);
    return GRD_OK;
  }
  DevMem mem(ctx);
  float *df, *dl;
  GRD_TRY(mem.alloc_n(&df, n * kIn));
  GRD_TRY(mem.alloc_n(&dl, n * kOut));
  GRD_TRY(copy_in(ctx, df, feat, n * kIn * 4));
  hipLaunchKernelGGL(k_mlp_infer, dim3(infer_blocks(ctx, n)), dim3(kBlock), 0, ctx->stream, ctx->sel_w, df, (uint32_t)n,
                     dl, (uint32_t *)nullptr, 0u);
  GRD_HIP(hipGetLastError());
  return copy_out(ctx, logits, dl, n * kOut);
}

grd_status grd_selector_infer_noalloc(grd_ctx *ctx, const float *feat, uint64_t n, float *logits)
{
  if (!ctx || !feat || !logits || n == 0) return fail(GRD_ERR_ARG, "grd_selector_infer_noalloc: bad argument");
  if (n > kInferMax)
    return fail(GRD_ERR_ARG, "grd_selector_infer_noalloc: at most " + std::to_string(kInferMax) + " samples per call");
  if (!ctx->sel_loaded) return fail(GRD_ERR_STATE, "grd_selector_infer_noalloc: no weights loaded");
  if (ctx->device < 0 || ctx->device >= kMaxDevices || !g_scratch_ptr[ctx->device])
    return fail(GRD_ERR_STATE, "grd_selector_infer_noalloc: scratch not set up for this device");
  GRD_HIP(hipSetDevice(ctx->device));
  // staging in the device's scratch copy: features, then logits; every
  // element read is written first in this call
  float *df = g_scratch_ptr[ctx->device];
  float *dl = df + (size_t)kInferMax * kIn;
  GRD_HIP(hipMemcpyAsync(df, feat, n * kIn * 4, hipMemcpyHostToDevice, ctx->stream));
  hipLaunchKernelGGL(k_mlp_infer, dim3(infer_blocks(ctx, n)), dim3(kBlock), 0, ctx->stream, ctx->sel_w, df, (uint32_t)n,
                     dl, (uint32_t *)nullptr, 0u);
  GRD_HIP(hipGetLastError());
  GRD_HIP(hipMemcpyAsync(logits, dl, n * kOut * 4, hipMemcpyDeviceToHost, ctx->stream));
  GRD_HIP(hipStreamSynchronize(ctx->stream));
  return GRD_OK;
}

grd_status grd_selector_grad(grd_ctx *ctx, const float *w, const float *feat, const uint32_t *label, const float *cost,
                             uint64_t n, float *loss, float *grad)
{
  if (!ctx || !w || !feat || !label || !loss || !grad || n == 0) return fail(GRD_ERR_ARG, "grd_selector_grad: bad argument");
  for (uint64_t i = 0; i < n; i++)
    if (label[i] >= (uint32_t)kOut) return fail(GRD_ERR_ARG, "grd_selector_grad: label out of range");
  GRD_HIP(hipSetDevice(ctx->device));
  hipStream_t st = ctx->stream;
  DevMem mem(ctx);
  float *dw, *df, *dsw = nullptr, *dpart;
  uint32_t *dl;
  const uint32_t grid = grad_blocks(ctx, n);
  GRD_TRY(infer_stage(ctx));
  GRD_TRY(mem.alloc_n(&dw, kParams));
  GRD_TRY(mem.alloc_n(&df, n * kIn));
  GRD_TRY(mem.alloc_n(&dl, n));
  GRD_TRY(mem.alloc_n(&dpart, (uint64_t)grid * kPart));
  GRD_TRY(copy_in(ctx, dw, w, kParams * 4));
  GRD_TRY(copy_in(ctx, df, feat, n * kIn * 4));
  GRD_TRY(copy_in(ctx, dl, label, n * 4));
  if (cost) {
    GRD_TRY(mem.alloc_n(&dsw, n));
    GRD_TRY(copy_in(ctx, dsw, cost, n * 4));
  }
  hipLaunchKernelGGL(k_mlp_grad<false>, dim3(grid), dim3(kBlock), 0, st, dw, nullptr, df, dl, dsw, nullptr,
                     (uint32_t)n, dpart);
  constexpr uint32_t kRed = (kPart + kWave - 1) / kWave;
  static_assert(kPart <= (int)(kInferMax * (kIn + kOut)) && kRed <= kInferMax / kTileS, "the stage holds a gradient");
  float *out = ctx->sel_stage;
  uint32_t *flags = reinterpret_cast<uint32_t *>(out + (size_t)kInferMax * (kIn + kOut));
  const uint32_t seq = ++ctx->sel_seq;
  hipLaunchKernelGGL(k_mlp_reduce, dim3(kRed), dim3(kWave), 0, st, (const float *)dpart, grid, out, flags, seq);
  GRD_HIP(hipGetLastError());
  for (uint32_t b = 0; b < kRed; b++) GRD_TRY(wait_pinned(ctx, flags + b, seq));
  memcpy(grad, out, kParams * 4);
  *loss = out[kParams];
  return GRD_OK;
}

}  // extern "C"
