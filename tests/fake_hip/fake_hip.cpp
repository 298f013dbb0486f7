// The part of the HIP runtime that libaerofx calls, on host memory: kernels do
// not run, every call is logged, and a chosen call (or host allocation) can be
// made to fail.  Linked with the library's objects in place of the HIP runtime,
// it lets a test without a GPU drive the set-up code through its error paths.
#define __HIP_PLATFORM_AMD__ 1
#include <cxxabi.h>
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <string>
#include <vector>

namespace {
std::recursive_mutex mu;
std::string &log_text() {
  static std::string s;
  return s;
}
std::map<const void *, std::string> &kernels() {
  static std::map<const void *, std::string> m;
  return m;
}
std::string armed;        // the call that fails ("" = any that can)
long countdown = 0;       // 0: nothing armed
long new_countdown = 0;   // the host allocation that throws
hipError_t launch_error = hipSuccess;
thread_local int inside = 0;  // this file's own allocations do not count
struct Inside {
  Inside() { ++inside; }
  ~Inside() { --inside; }
};

// logs the call; true when it is the one to fail
bool fails(const char *name) {
  Inside in;
  std::lock_guard<std::recursive_mutex> l(mu);
  bool f = false;
  if (countdown > 0 && (armed.empty() || armed == name)) f = --countdown == 0;
  log_text() += std::string(name) + (f ? "!\n" : "\n");
  return f;
}
}  // namespace

extern "C" {
// the n-th call from now on named `name` ("" = any) fails
void fake_arm(const char *name, long n) {
  Inside in;
  armed = name;
  countdown = n;
}
// the n-th operator new from now on throws (0: none)
void fake_arm_new(long n) { new_countdown = n; }
// 1 while the armed failure has not happened
int fake_pending() { return countdown > 0 || new_countdown > 0; }
void fake_clear() { log_text().clear(); }
const char *fake_log() { return log_text().c_str(); }

hipError_t hipMalloc(void **p, size_t n) {
  if (fails("hipMalloc")) return hipErrorOutOfMemory;
  *p = std::calloc(1, n);
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  if (fails("hipHostMalloc")) return hipErrorOutOfMemory;
  *p = std::calloc(1, n);
  return hipSuccess;
}
hipError_t hipHostFree(void *p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
  if (fails("hipMemcpy")) return hipErrorUnknown;
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
  if (fails("hipMemcpyAsync")) return hipErrorUnknown;
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemset(void *d, int v, size_t n) {
  if (fails("hipMemset")) return hipErrorUnknown;
  std::memset(d, v, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) {
  if (fails("hipMemsetAsync")) return hipErrorUnknown;
  std::memset(d, v, n);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
  return fails("hipStreamSynchronize") ? hipErrorUnknown : hipSuccess;
}
// a failed launch is reported by the hipGetLastError after it
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **, size_t, hipStream_t) {
  std::lock_guard<std::recursive_mutex> l(mu);
  Inside in;
  const bool bad = fails("hipLaunchKernel");
  log_text() += "kernel " + kernels()[f] + "\n";
  if (bad) launch_error = hipErrorLaunchFailure;
  return bad ? hipErrorLaunchFailure : hipSuccess;
}
hipError_t hipGetLastError() {
  const hipError_t e = launch_error;
  launch_error = hipSuccess;
  return e;
}
const char *hipGetErrorString(hipError_t) { return "simulated failure"; }
hipError_t hipGetDevice(int *d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *) {
  static char store[256];
  *p = store;
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  *s = reinterpret_cast<hipStream_t>(std::malloc(1));
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  std::free(s);
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) {
  *e = reinterpret_cast<hipEvent_t>(std::malloc(1));
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) {
  std::free(e);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
  *ms = 0.f;
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

// what the compiler's host code of a <<<>>> launch and of the modules calls
struct CallConf {
  dim3 g, b;
  size_t shared;
  hipStream_t s;
};
static thread_local std::vector<CallConf> conf;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t shared, hipStream_t s) {
  Inside in;
  conf.push_back({g, b, shared, s});
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *shared, hipStream_t *s) {
  *g = conf.back().g;
  *b = conf.back().b;
  *shared = conf.back().shared;
  *s = conf.back().s;
  conf.pop_back();
  return hipSuccess;
}
void **__hipRegisterFatBinary(const void *) {
  static void *module = nullptr;
  return &module;
}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, dim3 *,
                           dim3 *, int *) {
  int status = 0;
  char *d = abi::__cxa_demangle(name, nullptr, nullptr, &status);
  std::string k = d ? d : name;  // [void] aerofx::[(anonymous namespace)::]k_name[<...>](...)
  std::free(d);
  const size_t b = k.find("k_");
  if (b != std::string::npos) k = k.substr(b, k.find_first_of("<(", b) - b);
  kernels()[host] = k;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void **) {}
}

void *operator new(size_t n) {
  if (!inside && new_countdown > 0 && --new_countdown == 0) throw std::bad_alloc();
  void *p = std::malloc(n ? n : 1);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }
