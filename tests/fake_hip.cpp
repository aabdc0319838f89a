// A HIP runtime without a device, for tests of what the library's host code does
// with memory: device memory is host memory within a limit, copies are copies,
// kernels do nothing.  Loaded before the library, its functions are taken.
// It also takes operator new, which can be told to fail, and asynchronous copies
// can be told to wait for the next synchronisation, so that a host array that goes
// before its copy is noticed.
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <new>
#include <vector>

#include <malloc.h>

#include <hip/hip_runtime.h>

namespace {
template <class T>
struct Plain {  // (its own bookkeeping never fails)
  using value_type = T;
  Plain() = default;
  template <class U>
  Plain(const Plain<U> &) {}
  T *allocate(size_t n) { return static_cast<T *>(malloc(n * sizeof(T))); }
  void deallocate(T *p, size_t) { free(p); }
  template <class U>
  bool operator==(const Plain<U> &) const { return true; }
  template <class U>
  bool operator!=(const Plain<U> &) const { return false; }
};
std::map<void *, size_t, std::less<void *>, Plain<std::pair<void *const, size_t>>> blocks;
uint64_t live = 0, limit = ~0ull, launches = 0, bad_frees = 0;
bool new_fails = false;
long new_fails_in = 0;  // the how many-th from now fails, once (0: none)
uint64_t news = 0;
bool new_ok()
{
  news++;
  return !new_fails && (new_fails_in == 0 || --new_fails_in != 0);
}
uint64_t mallocs_left = ~0ull;
bool defer = false;
uint64_t lost = 0;  // host arrays that went before their copy
struct Copy {
  void *d;
  const void *s;
  size_t n;
};
std::vector<Copy, Plain<Copy>> pending;
void run_pending()
{
  for (const Copy &c : pending) memcpy(c.d, c.s, c.n);
  pending.clear();
}
void drop(void *p)
{
  if (!p) return;
  const char *a = static_cast<char *>(p), *b = a + malloc_usable_size(p);
  for (size_t i = 0; i < pending.size();) {
    const char *s = static_cast<const char *>(pending[i].s), *d = static_cast<const char *>(pending[i].d);
    if ((s >= a && s < b) || (d >= a && d < b)) {
      lost++;
      pending.erase(pending.begin() + i);
    } else {
      i++;
    }
  }
  free(p);
}
struct Call {
  dim3 grid, block;
  size_t shared;
  hipStream_t stream;
} call;
}  // namespace

void *operator new(size_t n)
{
  void *p = new_ok() ? malloc(n ? n : 1) : nullptr;
  if (!p) throw std::bad_alloc();
  return p;
}
void *operator new(size_t n, const std::nothrow_t &) noexcept { return new_ok() ? malloc(n ? n : 1) : nullptr; }
void operator delete(void *p) noexcept { drop(p); }
void operator delete(void *p, size_t) noexcept { drop(p); }

extern "C" {
uint64_t fake_live() { return live; }
uint64_t fake_launches() { return launches; }
uint64_t fake_bad_frees() { return bad_frees; }
void fake_mallocs_left(uint64_t n) { mallocs_left = n; }
void fake_defer(int on) { defer = on != 0; }
uint64_t fake_lost() { return lost; }
void fake_limit(uint64_t bytes) { limit = bytes; }
void fake_new_fails(int on) { new_fails = on != 0; }
void fake_new_fails_in(long n) { new_fails_in = n; }
uint64_t fake_news() { return news; }
long fake_new_left() { return new_fails_in; }

hipError_t hipMalloc(void **p, size_t n)
{
  *p = nullptr;
  if (mallocs_left == 0) return hipErrorOutOfMemory;
  if (n > limit || live > limit - n) return hipErrorOutOfMemory;
  mallocs_left--;
  *p = calloc(n ? n : 1, 1);
  blocks[*p] = n;
  live += n;
  return hipSuccess;
}
hipError_t hipFree(void *p)
{
  run_pending();
  if (!p) return hipSuccess;
  auto it = blocks.find(p);
  if (it == blocks.end()) {
    bad_frees++;
    return hipErrorInvalidValue;
  }
  live -= it->second;
  blocks.erase(it);
  free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned int)
{
  *p = calloc(n ? n : 1, 1);
  return hipSuccess;
}
hipError_t hipHostFree(void *p)
{
  run_pending();
  free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind)
{
  run_pending();
  if (n) memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t)
{
  if (!defer) return hipMemcpy(d, s, n, k);
  if (n) pending.push_back(Copy{d, s, n});
  return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t)
{
  run_pending();
  if (n) memset(d, v, n);
  return hipSuccess;
}
hipError_t hipGetDeviceCount(int *n)
{
  *n = 2;
  return hipSuccess;
}
static thread_local int device = 0;
hipError_t hipSetDevice(int d)
{
  device = d;
  return hipSuccess;
}
hipError_t hipGetDevice(int *d)
{
  *d = device;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int)
{
  *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : a == hipDeviceAttributeWarpSize ? 64 : 1024;
  return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int)
{
  memset(p, 0, sizeof *p);
  strcpy(p->gcnArchName, "gfx950");
  p->warpSize = 64;
  p->multiProcessorCount = 256;
  p->maxThreadsPerBlock = 1024;
  return hipSuccess;
}
static char handle[64];
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned int)
{
  *s = reinterpret_cast<hipStream_t>(handle);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t)
{
  run_pending();
  return hipSuccess;
}
int hipGetStreamDeviceId(hipStream_t) { return 0; }
hipError_t hipEventCreate(hipEvent_t *e)
{
  *e = reinterpret_cast<hipEvent_t>(handle);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipStreamSynchronize(nullptr); }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t)
{
  *ms = 0.0f;
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "fake"; }
static float symbol[1 << 17];
hipError_t hipGetSymbolAddress(void **p, const void *)
{
  *p = symbol;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t)
{
  launches++;
  return hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t s, hipStream_t st)
{
  call = Call{g, b, s, st};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *s, hipStream_t *st)
{
  *g = call.grid;
  *b = call.block;
  *s = call.shared;
  *st = call.stream;
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g)
{
  *g = reinterpret_cast<hipGraph_t>(handle);
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t)
{
  *e = reinterpret_cast<hipGraphExec_t>(handle);
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
}
