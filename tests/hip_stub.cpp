// A HIP runtime without a device, for tests of the host code's call order: device
// memory is host memory, kernels do not run, and the calls that order work are
// recorded as lines of text.  Loaded ahead of the real runtime.
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <string>

namespace {
std::mutex mu;
std::string log_text;
std::map<const void *, std::string> names;
std::map<void *, size_t> sizes;
size_t live_bytes = 0, limit_bytes = SIZE_MAX;
hipStream_t capturing = nullptr;
hipError_t last = hipSuccess;
uintptr_t next_stream = 0x1000;
thread_local hipStreamCaptureMode mode = hipStreamCaptureModeGlobal;
struct Config {
  dim3 grid, block;
  size_t shared;
  hipStream_t stream;
};
thread_local Config config;

void note(const std::string &line) {
  const std::lock_guard<std::mutex> l(mu);
  log_text += line + "\n";
}
std::string id(hipStream_t s) { return std::to_string(reinterpret_cast<uintptr_t>(s)); }
hipError_t fail(hipError_t e) { return last = e; }
// Calls that end a capture on this thread (global or thread-local mode).
bool unsafe(const char *what) {
  if (!capturing || mode == hipStreamCaptureModeRelaxed) return false;
  note(std::string("unsafe ") + what);
  (void)fail(hipErrorStreamCaptureUnsupported);
  return true;
}
}  // namespace

// Host allocations of at least this many bytes fail.
static size_t host_limit = SIZE_MAX;
void *operator new(size_t n) {
  if (n >= host_limit) throw std::bad_alloc();
  if (void *p = std::malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

extern "C" {
void stub_host_limit(size_t bytes) { host_limit = bytes; }
const char *stub_log() { return log_text.c_str(); }
void stub_clear() { log_text.clear(); }
void stub_limit(size_t bytes) { limit_bytes = bytes; }
size_t stub_live() { return live_bytes; }
void stub_capture(void *s) { capturing = static_cast<hipStream_t>(s); }

void **__hipRegisterFatBinary(const void *) {
  static void *handle;
  return &handle;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *,
                           void *, void *, int *) {
  names[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t s) {
  config = {grid, block, shared, s};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shared, hipStream_t *s) {
  *grid = config.grid;
  *block = config.block;
  *shared = config.shared;
  *s = config.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3, void **, size_t, hipStream_t s) {
  note("launch " + names[f] + " " + id(s) + " " + std::to_string(grid.x));
  return hipSuccess;
}
hipError_t hipGetDeviceCount(int *n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipGetDevice(int *d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) {
  *v = 256;
  return hipSuccess;
}
hipError_t hipGetLastError() {
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
const char *hipGetErrorString(hipError_t) { return "stub error"; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *) {
  a->type = hipMemoryTypeDevice;
  return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) {
  *n = 4;
  return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n) {
  if (unsafe("hipMalloc")) return hipErrorStreamCaptureUnsupported;
  const std::lock_guard<std::mutex> l(mu);
  if (live_bytes + n > limit_bytes) {
    log_text += "nomem\n";
    return fail(hipErrorOutOfMemory);
  }
  *p = std::calloc(1, n);
  sizes[*p] = n;
  live_bytes += n;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  const std::lock_guard<std::mutex> l(mu);
  live_bytes -= sizes[p];
  sizes.erase(p);
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
  if (unsafe("hipMemcpy")) return hipErrorStreamCaptureUnsupported;
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t st) {
  note("copy " + id(st));
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemset(void *d, int v, size_t n) {
  std::memset(d, v, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) {
  std::memset(d, v, n);
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  *s = reinterpret_cast<hipStream_t>(next_stream++);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) {
  if (capturing && s == capturing) {
    note("unsafe hipStreamSynchronize");
    return fail(hipErrorStreamCaptureUnsupported);
  }
  note("sync " + id(s));
  return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *st) {
  *st = capturing && s == capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) {
  *g = nullptr;
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) {
  *e = nullptr;
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *m) {
  std::swap(*m, mode);
  return hipSuccess;
}
}
