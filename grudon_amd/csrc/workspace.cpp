// workspace.cpp -- memory a context keeps between calls: freed device blocks,
// and pinned host buffers through which large arrays travel.
//
// A graph and its state are some seventy device allocations.  hipMalloc and
// hipFree of a block take 30 to 200 us each (the free also waits for the
// device): building, solving and releasing one graph of 700 K vertices spent 11
// of 24 ms in them.  A pageable copy to the host goes through the runtime's own
// staging on one thread, and a result array fresh from the allocator takes a
// page fault per page on that thread: 67 MB of labels took 6.5 ms, a third
// more than the solve.
#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstring>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

#include "grd_internal.hpp"

namespace grd {

// ------------------------------------------------------------------------
// device blocks
// ------------------------------------------------------------------------

// Block sizes: eighths of a power of two, so a block fits its later users
// within 25 % and few sizes occur.
static uint64_t block_size(uint64_t n)
{
  n = std::max<uint64_t>(n, 256);
  uint64_t p = 256;
  while (p * 2 <= n) p *= 2;
  const uint64_t step = std::max<uint64_t>(256, p / 8);
  return (n + step - 1) / step * step;
}

void *BlockCache::take(uint64_t want, uint64_t *got)
{
  std::lock_guard<std::mutex> lock(mu);
  auto it = blocks.lower_bound(want);
  if (it == blocks.end() || it->first > want + want / 4) return nullptr;
  void *p = it->second;
  *got = it->first;
  held -= it->first;
  blocks.erase(it);
  return p;
}

bool BlockCache::give(void *p, uint64_t size)
{
  std::lock_guard<std::mutex> lock(mu);
  if (size > kMaxBlock || held + size > kMaxHeld) return false;
  try {
    blocks.emplace(size, p);
  } catch (const std::bad_alloc &) {
    return false;  // (objects are freed without memory to note it: the block goes back)
  }
  held += size;
  return true;
}

void BlockCache::trim()
{
  std::lock_guard<std::mutex> lock(mu);
  for (auto &b : blocks) (void)hipFree(b.second);
  blocks.clear();
  held = 0;
}

// The process's contexts: what they keep goes back before an allocation on
// their device may fail (the blocks kept are idle, and a cache has its lock).
constexpr size_t kHostCountersKept = 8;
static std::mutex g_contexts_mu;
static std::vector<grd_ctx *> &contexts()
{
  static std::vector<grd_ctx *> *v = new std::vector<grd_ctx *>();  // (outlives every context)
  return *v;
}

grd_status workspace_open(grd_ctx *ctx)
{
  std::lock_guard<std::mutex> lock(g_contexts_mu);
  try {
    ctx->host_counters.reserve(kHostCountersKept);  // (giving one back never allocates)
    contexts().push_back(ctx);
  } catch (const std::bad_alloc &) {
    return fail(GRD_ERR_OOM, "grd_create: host allocation failed");
  }
  return GRD_OK;
}

grd_status device_malloc(int device, void **p, uint64_t bytes)
{
  hipError_t e = hipMalloc(p, bytes);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    {
      std::lock_guard<std::mutex> lock(g_contexts_mu);
      for (grd_ctx *c : contexts())
        if (c->device == device) c->cache.trim();
    }
    e = hipMalloc(p, bytes);
  }
  if (e != hipSuccess) {
    *p = nullptr;
    (void)hipGetLastError();
    return fail(GRD_ERR_OOM, "hipMalloc(" + std::to_string(bytes) + " bytes) failed: " + hipGetErrorString(e));
  }
  return GRD_OK;
}

grd_status DevMem::alloc(void **p, uint64_t nbytes)
{
  *p = nullptr;
  const uint64_t b = nbytes ? nbytes : 64;
  uint64_t size = block_size(b);
  try {
    ptrs.emplace_back(nullptr, 0);  // room first: a block is never left without a note of it
  } catch (const std::bad_alloc &) {
    (void)hipStreamSynchronize(ctx->stream);
    return fail(GRD_ERR_OOM, "host allocation failed");
  }
  *p = ctx->cache.take(size, &size);
  if (!*p) {
    const grd_status st = device_malloc(ctx->device, p, size);
    if (st != GRD_OK) {
      // the caller gives up: what it has queued still reads its host arrays
      (void)hipStreamSynchronize(ctx->stream);
      ptrs.pop_back();
      return st;
    }
  }
  ptrs.back() = {*p, size};
  bytes += b;
  return GRD_OK;
}

void DevMem::release()
{
  // as hipFree does, wait for what may still use the blocks
  if (!ptrs.empty()) (void)hipStreamSynchronize(ctx->stream);
  for (auto &b : ptrs)
    if (!ctx->cache.give(b.first, b.second)) (void)hipFree(b.first);
  ptrs.clear();
  bytes = 0;
}

// ------------------------------------------------------------------------
// pinned staging
// ------------------------------------------------------------------------

constexpr uint64_t kSlot = 4ull << 20;        // bytes per staging slot
constexpr uint64_t kSmall = 256ull << 10;     // transfers up to this take one small buffer
// below this the runtime's own copy is as fast (370 KB in 31 us; through the
// slots 47), from here on the slots and their helpers (16 MB 0.97 ms against
// 1.33, 67 MB 2.9 ms against 6.7)
constexpr uint64_t kRing = 4ull << 20;
constexpr uint64_t kPerThread = 512ull << 10;  // bytes that pay for a helper thread
constexpr int kMaxHelpers = 7;

static grd_status stage_small(grd_ctx *ctx)
{
  if (ctx->stage_small) return GRD_OK;
  GRD_HIP(hipHostMalloc((void **)&ctx->stage_small, kSmall + kSmallFlags * 4, hipHostMallocDefault));
  memset(ctx->stage_small + kSmall, 0, kSmallFlags * 4);
  return GRD_OK;
}

static grd_status stage_ring(grd_ctx *ctx)
{
  if (ctx->stage) return GRD_OK;
  for (auto &e : ctx->stage_ev)
    if (!e) GRD_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  GRD_HIP(hipHostMalloc((void **)&ctx->stage, kSlot * kStageSlots, hipHostMallocDefault));
  return GRD_OK;
}

void workspace_release(grd_ctx *ctx)
{
  {
    std::lock_guard<std::mutex> lock(g_contexts_mu);
    auto &v = contexts();
    v.erase(std::remove(v.begin(), v.end(), ctx), v.end());
  }
  ctx->cache.trim();
  if (ctx->stage) (void)hipHostFree(ctx->stage);
  if (ctx->stage_small) (void)hipHostFree(ctx->stage_small);
  for (auto &e : ctx->stage_ev)
    if (e) (void)hipEventDestroy(e);
  for (void *p : ctx->host_counters) (void)hipHostFree(p);
}

grd_status host_counters_take(grd_ctx *ctx, Counters **out)
{
  if (!ctx->host_counters.empty()) {
    *out = (Counters *)ctx->host_counters.back();
    ctx->host_counters.pop_back();
  } else {
    GRD_HIP(hipHostMalloc((void **)out, kHostCounters, hipHostMallocDefault));
  }
  memset((void *)*out, 0, kHostCounters);
  return GRD_OK;
}

void host_counters_give(grd_ctx *ctx, Counters *p)
{
  if (!p) return;
  if (ctx->host_counters.size() < kHostCountersKept) ctx->host_counters.push_back(p);
  else (void)hipHostFree(p);
}

// A superstep of a small graph is tens of microseconds, so the host looks at the
// pinned word for a short while before it hands the wait to the runtime.
grd_status wait_pinned(grd_ctx *ctx, const uint32_t *word, uint32_t want)
{
  const auto t0 = std::chrono::steady_clock::now();
  for (uint32_t i = 1; __atomic_load_n(word, __ATOMIC_ACQUIRE) != want; i++) {
    __builtin_ia32_pause();
    if (i % 64 == 0 && std::chrono::steady_clock::now() - t0 > std::chrono::microseconds(200)) {
      GRD_HIP(hipStreamSynchronize(ctx->stream));
      if (__atomic_load_n(word, __ATOMIC_ACQUIRE) != want)
        return fail(GRD_ERR_HIP, "a device pass did not report its end");
    }
  }
  return GRD_OK;
}

// Helper threads of one transfer: thread t of T copies part t of every chunk
// once the chunk is ready (`go` chunks are), and counts it done.  The calling
// thread is thread 0.
namespace {
struct Crew {
  int T = 1;
  std::atomic<uint64_t> go{0};
  std::atomic<uint64_t> done[kStageSlots] = {};  // parts done per slot, over the whole transfer
  std::vector<std::thread> threads;
  template <class F>
  void start(int n, uint64_t chunks, F part)
  {
    // (no helper reads T before the first chunk goes, so it may be set last: a
    // thread that the system refuses leaves a smaller crew)
    try {
      for (int t = 1; t <= n; t++)
        threads.emplace_back([this, t, chunks, part]() {
          for (uint64_t c = 0; c < chunks; c++) {
            while (go.load(std::memory_order_acquire) <= c) std::this_thread::yield();
            part(c, t, T);
            done[c % kStageSlots].fetch_add(1, std::memory_order_release);
          }
        });
    } catch (...) {
    }
    T = 1 + (int)threads.size();
  }
  // every part of chunk c, the slot's c / kStageSlots-th user, is done
  void wait(uint64_t c)
  {
    const uint64_t want = (c / kStageSlots + 1) * (uint64_t)(T - 1);
    while (done[c % kStageSlots].load(std::memory_order_acquire) < want) std::this_thread::yield();
  }
  void finish(uint64_t chunks)  // (an abandoned transfer lets its helpers run through)
  {
    go.store(chunks, std::memory_order_release);
    for (auto &t : threads) t.join();
  }
};

int helpers(const grd_ctx *ctx, uint64_t bytes)
{
  return (int)std::min<uint64_t>({(uint64_t)kMaxHelpers, (uint64_t)(host_threads(ctx) - 1), bytes / kPerThread});
}

void part_of_chunk(uint64_t n, int t, int T, uint64_t *a, uint64_t *b)
{
  const uint64_t per = ((n + T - 1) / T + 63) & ~63ull;
  *a = std::min<uint64_t>(n, per * (uint64_t)t);
  *b = std::min<uint64_t>(n, *a + per);
}

// staged 4-byte values to the caller's array, as they are or widened (the
// unreached 2^32 - 1 to 2^64 - 1)
void put(void *dst, const uint32_t *src, uint64_t first, uint64_t n, bool wide)
{
  if (!wide) {
    memcpy((uint32_t *)dst + first, src, n * 4);
    return;
  }
  uint64_t *o = (uint64_t *)dst + first;
  for (uint64_t i = 0; i < n; i++) o[i] = src[i] == 0xFFFFFFFFu ? ~0ull : (uint64_t)src[i];
}
}  // namespace

// A short result: a kernel gathers the values into pinned memory and the host
// waits for its waves' flags.  With a gather, a copy command and a stream
// synchronisation a thousand labels took 16.3 us, now 12.2; 16384 24.6, now 20.
// At 32768 it is 27.8 against 29.8, so the line lies below; contiguous values are
// copied as fast by the command.
grd_status copy_out_slots(grd_ctx *ctx, void *dst, const uint32_t *src, const uint32_t *gid, uint32_t S, uint32_t n,
                          bool wide)
{
  GRD_TRY(stage_small(ctx));
  uint32_t *host = reinterpret_cast<uint32_t *>(ctx->stage_small);
  uint32_t *flags = reinterpret_cast<uint32_t *>(ctx->stage_small + kSmall), nf = 0;
  const uint32_t seq = ++ctx->stage_seq;
  GRD_TRY(small_out(ctx, src, gid, S, n, host, flags, seq, &nf));
  for (uint32_t f = 0; f < nf; f++) GRD_TRY(wait_pinned(ctx, flags + f, seq));
  put(dst, host, 0, n, wide);
  return GRD_OK;
}

grd_status copy_out(grd_ctx *ctx, void *dst, const void *src, uint64_t n, bool wide)
{
  if (!n) return GRD_OK;
  hipStream_t st = ctx->stream;
  const uint64_t bytes = n * 4;
  if (bytes <= kSmall) {
    GRD_TRY(stage_small(ctx));
    GRD_HIP(hipMemcpyAsync(ctx->stage_small, src, bytes, hipMemcpyDeviceToHost, st));
    GRD_HIP(hipStreamSynchronize(st));
    put(dst, (const uint32_t *)ctx->stage_small, 0, n, wide);
    return GRD_OK;
  }
  if (bytes < kRing && !wide) {
    GRD_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st));
    GRD_HIP(hipStreamSynchronize(st));
    return GRD_OK;
  }
  GRD_TRY(stage_ring(ctx));
  if (bytes < kRing) {
    // widened, one slot holds it, and helpers do not pay yet: 300000 values 133 us
    // (in chunks with helpers 213, widened in place in the caller's array 180), a
    // million 360 (430, 490)
    GRD_HIP(hipMemcpyAsync(ctx->stage, src, bytes, hipMemcpyDeviceToHost, st));
    GRD_HIP(hipStreamSynchronize(st));
    put(dst, (const uint32_t *)ctx->stage, 0, n, wide);
    return GRD_OK;
  }
  // chunks small enough that copy and write-out of one transfer overlap
  const uint64_t chunk = std::min<uint64_t>(kSlot, std::max<uint64_t>(kSmall, (bytes / kStageSlots + 4095) & ~4095ull)) / 4;
  const uint64_t chunks = (n + chunk - 1) / chunk;
  char *stage = ctx->stage;
  auto part = [=](uint64_t c, int t, int T) {
    const uint64_t first = c * chunk, cn = std::min(chunk, n - first);
    uint64_t a, b;
    part_of_chunk(cn, t, T, &a, &b);
    put(dst, (const uint32_t *)(stage + (c % kStageSlots) * kSlot) + a, first + a, b - a, wide);
  };
  Crew crew;
  crew.start(helpers(ctx, bytes * (wide ? 2 : 1)), chunks, part);
  hipError_t e = hipSuccess;
  uint64_t issued = 0;
  for (uint64_t c = 0; c < chunks && e == hipSuccess; c++) {
    for (; issued < chunks && issued < c + kStageSlots && e == hipSuccess; issued++) {
      if (issued >= kStageSlots) crew.wait(issued - kStageSlots);
      const uint64_t first = issued * chunk, cn = std::min(chunk, n - first);
      const int slot = (int)(issued % kStageSlots);
      e = hipMemcpyAsync(stage + slot * kSlot, (const uint32_t *)src + first, cn * 4, hipMemcpyDeviceToHost, st);
      if (e == hipSuccess) e = hipEventRecord(ctx->stage_ev[slot], st);
    }
    if (e == hipSuccess) e = hipEventSynchronize(ctx->stage_ev[c % kStageSlots]);
    if (e != hipSuccess) break;
    crew.go.store(c + 1, std::memory_order_release);
    part(c, 0, crew.T);
  }
  if (e != hipSuccess) (void)hipStreamSynchronize(st);
  crew.finish(chunks);
  GRD_HIP(e);
  return GRD_OK;
}

grd_status copy_in(grd_ctx *ctx, void *dst, const void *src, uint64_t bytes)
{
  if (!bytes) return GRD_OK;
  hipStream_t st = ctx->stream;
  if (bytes < kRing) {
    GRD_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, st));
    return GRD_OK;
  }
  GRD_TRY(stage_ring(ctx));
  const uint64_t chunk = kSlot, chunks = (bytes + chunk - 1) / chunk;
  char *stage = ctx->stage;
  auto part = [=](uint64_t c, int t, int T) {
    const uint64_t first = c * chunk, cn = std::min(chunk, bytes - first);
    uint64_t a, b;
    part_of_chunk(cn, t, T, &a, &b);
    memcpy(stage + (c % kStageSlots) * kSlot + a, (const char *)src + first + a, b - a);
  };
  Crew crew;
  crew.start(helpers(ctx, bytes), chunks, part);
  hipError_t e = hipSuccess;
  for (uint64_t c = 0; c < chunks; c++) {
    const int slot = (int)(c % kStageSlots);
    // the slot's previous transfer (of this call or an earlier one) is over
    e = hipEventSynchronize(ctx->stage_ev[slot]);
    if (e != hipSuccess) break;
    crew.go.store(c + 1, std::memory_order_release);
    part(c, 0, crew.T);
    crew.wait(c);
    const uint64_t first = c * chunk, cn = std::min(chunk, bytes - first);
    e = hipMemcpyAsync((char *)dst + first, stage + slot * kSlot, cn, hipMemcpyHostToDevice, st);
    if (e == hipSuccess) e = hipEventRecord(ctx->stage_ev[slot], st);
    if (e != hipSuccess) break;
  }
  crew.finish(chunks);
  GRD_HIP(e);
  return GRD_OK;
}

}  // namespace grd
