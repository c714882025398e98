// A HIP runtime without a device, for the tests in tests/test_hip_host.py:
// every HIP function that libacc_cn.so calls, over host memory.  Loaded with
// its symbols global before libacc_cn.so, it takes the runtime's place in that
// process.  Device memory is zeroed host memory under a limit that the test
// sets, copies happen at once, and kernels do nothing; what the library asked
// for is kept as a log, one line per call:
//
//   alloc P BYTES | free P | copy STREAM | fill STREAM | launch STREAM KERNEL
//   record EVENT STREAM | wait STREAM EVENT | sync STREAM | sync all
//
// The library's graphs then hold no counts, so the tests use graphs whose host
// side needs none (vertices without edges).
#include <hip/hip_runtime_api.h>

#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <string>

namespace {
std::mutex mu;
std::string text;
std::map<void *, size_t> blocks;
std::map<const void *, std::string> kernels;
size_t held = 0, limit = SIZE_MAX;
long next_id = 1;
thread_local long news_left = -1;  // operator new of this thread fails once this many have been taken

void line(const char *format, ...) {
  char b[512];
  va_list a;
  va_start(a, format);
  std::vsnprintf(b, sizeof(b), format, a);
  va_end(a);
  const long keep = news_left;
  news_left = -1;  // the stand-in's own memory does not fail
  text += b;
  text += '\n';
  news_left = keep;
}

struct Config {
  dim3 grid, block;
  size_t shared;
  hipStream_t stream;
};
thread_local Config config;
}  // namespace

void *operator new(size_t n) {
  if (news_left == 0) throw std::bad_alloc();
  if (news_left > 0) news_left--;
  if (void *p = std::malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

extern "C" {

// ---- the test's side
const char *fake_log() { return text.c_str(); }
void fake_clear() { text.clear(); }
void fake_limit(size_t bytes) { limit = bytes; }
size_t fake_held() { return held; }
void fake_fail_new(long after) { news_left = after; }

// ---- code objects
void **__hipRegisterFatBinary(const void *) {
  static void *none = nullptr;
  return &none;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *,
                           void *, int *) {
  kernels[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream) {
  config = Config{grid, block, shared, stream};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shared, hipStream_t *stream) {
  *grid = config.grid;
  *block = config.block;
  *shared = config.shared;
  *stream = config.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *host, dim3, dim3, void **, size_t, hipStream_t stream) {
  std::lock_guard<std::mutex> lk(mu);
  line("launch %p %s", static_cast<void *>(stream), kernels[host].c_str());
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *) {
  static long long scratch[4096];
  *p = scratch;
  return hipSuccess;
}

// ---- the device
hipError_t hipGetDeviceCount(int *n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipGetDevice(int *d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
  std::memset(static_cast<void *>(p), 0, sizeof(*p));
  std::strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  p->sharedMemPerBlock = 160 << 10;
  p->warpSize = 64;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) {
  *v = 256;
  return hipSuccess;
}
hipError_t hipDeviceSynchronize() {
  std::lock_guard<std::mutex> lk(mu);
  line("sync all");
  return hipSuccess;
}
const char *hipGetErrorString(hipError_t) { return "fake HIP error"; }
hipError_t hipGetLastError() { return hipSuccess; }

// ---- memory
hipError_t hipMalloc(void **p, size_t bytes) {
  std::lock_guard<std::mutex> lk(mu);
  *p = nullptr;
  if (bytes > limit || held > limit - bytes) return hipErrorOutOfMemory;
  const long keep = news_left;
  news_left = -1;
  *p = std::calloc(1, bytes ? bytes : 1);
  blocks[*p] = bytes;
  held += bytes;
  line("alloc %p %zu", *p, bytes);
  news_left = keep;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  std::lock_guard<std::mutex> lk(mu);
  const long keep = news_left;
  news_left = -1;
  const auto it = blocks.find(p);
  if (it == blocks.end()) std::abort();
  held -= it->second;
  blocks.erase(it);
  line("free %p", p);
  std::free(p);
  news_left = keep;
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) {
  *p = std::calloc(1, bytes ? bytes : 1);
  return hipSuccess;
}
hipError_t hipHostFree(void *p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned) {
  *d = h;
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *, const void *) { return hipErrorInvalidValue; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t stream) {
  std::lock_guard<std::mutex> lk(mu);
  std::memcpy(d, s, n);
  line("copy %p", static_cast<void *>(stream));
  return hipSuccess;
}
hipError_t hipMemcpyWithStream(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t stream) {
  return hipMemcpyAsync(d, s, n, k, stream);
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t stream) {
  std::lock_guard<std::mutex> lk(mu);
  std::memset(d, v, n);
  line("fill %p", static_cast<void *>(stream));
  return hipSuccess;
}

// ---- streams, events, graphs
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  std::lock_guard<std::mutex> lk(mu);
  *s = reinterpret_cast<hipStream_t>(0x1000 * next_id++);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) {
  std::lock_guard<std::mutex> lk(mu);
  line("sync %p", static_cast<void *>(s));
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  std::lock_guard<std::mutex> lk(mu);
  line("wait %p %p", static_cast<void *>(s), static_cast<void *>(e));
  return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *st) {
  *st = hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *) { return hipSuccess; }
int hipGetStreamDeviceId(hipStream_t) { return 0; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  std::lock_guard<std::mutex> lk(mu);
  *e = reinterpret_cast<hipEvent_t>(0x1000 * next_id++);
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  std::lock_guard<std::mutex> lk(mu);
  line("record %p %p", static_cast<void *>(e), static_cast<void *>(s));
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
  *ms = 0;
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorNotSupported; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *) { return hipErrorNotSupported; }
hipError_t hipGraphInstantiate(hipGraphExec_t *, hipGraph_t, hipGraphNode_t *, char *, size_t) {
  return hipErrorNotSupported;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorNotSupported; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }

}  // extern "C"
