// A stand-in for the HIP runtime that runs no kernel: loaded with RTLD_GLOBAL
// ahead of libmcm.so, it takes the library's runtime calls, so that the CPU
// tests see what the host code allocates, launches and waits for, and can limit
// the device's memory or let a call fail.  Device memory is host memory (zeros);
// every event is a line of a log.
#include <dlfcn.h>
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <string>
#include <thread>

namespace {
std::mutex g_lock;
std::string g_log;
std::map<void*, size_t> g_device;
std::map<const void*, std::string> g_kernels;
size_t g_used = 0, g_peak = 0, g_limit = ~(size_t)0;
int g_failThreads = 0, g_failDownloads = 0;
dim3 g_grid, g_block;
size_t g_shared;
hipStream_t g_stream;

void note(const std::string& s) {
  std::lock_guard<std::mutex> l(g_lock);
  g_log += s + "\n";
}
hipError_t handle(void** h) {
  *h = (void*)0x10;
  return hipSuccess;
}
}  // namespace

extern "C" {
void fake_set_limit(size_t bytes) { g_limit = bytes; }
size_t fake_peak(int reset) {
  std::lock_guard<std::mutex> l(g_lock);
  const size_t p = g_peak;
  if (reset) g_peak = g_used;
  return p;
}
void fake_fail_threads(int on) { g_failThreads = on; }
void fake_fail_downloads(int n) { g_failDownloads = n; }  // the n-th from now on
const char* fake_log(int clear) {
  static std::string out;
  std::lock_guard<std::mutex> l(g_lock);
  out = g_log;
  if (clear) g_log.clear();
  return out.c_str();
}

hipError_t hipMalloc(void** p, size_t n) {
  std::lock_guard<std::mutex> l(g_lock);
  if (n > g_limit || g_used > g_limit - n) {
    g_log += "refused " + std::to_string(n) + "\n";
    return hipErrorOutOfMemory;
  }
  *p = calloc(1, n);
  g_device[*p] = n;
  g_used += n;
  if (g_used > g_peak) g_peak = g_used;
  g_log += "malloc " + std::to_string(n) + "\n";
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  std::lock_guard<std::mutex> l(g_lock);
  if (auto it = g_device.find(p); it != g_device.end()) {
    g_used -= it->second;
    g_device.erase(it);
    free(p);
  }
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  note("pinned " + std::to_string(n));
  *p = calloc(1, n);
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  note("memcpy " + std::to_string(n));
  memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) {
  if (k == hipMemcpyDeviceToHost) {
    std::lock_guard<std::mutex> l(g_lock);
    g_log += "download " + std::to_string(n) + "\n";
    if (g_failDownloads > 0 && --g_failDownloads == 0) return hipErrorUnknown;
  }
  memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
  note("memset " + std::to_string(n));
  if (v) memset(d, v, n);  // (what is allocated is zero already and no kernel writes)
  return hipSuccess;
}
hipError_t hipDeviceSynchronize() {
  note("sync device");
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
  note("sync stream");
  return hipSuccess;
}
hipError_t hipGetDeviceCount(int* n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  memset(p, 0, sizeof *p);
  strcpy(p->gcnArchName, "gfx950");
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
  *v = 256;
  return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
  *n = 4;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "unknown"; }
hipError_t hipStreamCreate(hipStream_t* s) { return handle((void**)s); }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return handle((void**)s); }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return handle((void**)e); }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return handle((void**)e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = 1.f;
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { return handle((void**)g); }
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) { return handle((void**)e); }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) {
  note("graph");
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) { return hipErrorUnknown; }
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3, void**, size_t, hipStream_t s) {
  note("launch " + g_kernels[f] + " " + std::to_string(g.x) + (s ? "" : " default"));
  return hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t m, hipStream_t s) {
  g_grid = g, g_block = b, g_shared = m, g_stream = s;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* m, hipStream_t* s) {
  *g = g_grid, *b = g_block, *m = g_shared, *s = g_stream;
  return hipSuccess;
}
void** __hipRegisterFatBinary(const void*) { return (void**)&g_log; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) { g_kernels[f] = name; }
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
}  // extern "C"

// std::thread's start as libmcm.so calls it: fails with bad_alloc on request.
void std::thread::_M_start_thread(_State_ptr state, void (*depend)()) {
  if (g_failThreads) throw std::bad_alloc();
  using Start = void (std::thread::*)(_State_ptr, void (*)());
  Start real;
  void* sym = dlsym(RTLD_NEXT, "_ZNSt6thread15_M_start_threadESt10unique_ptrINS_6_StateESt14default_deleteIS1_EEPFvvE");
  void* words[2] = {sym, nullptr};
  static_assert(sizeof real == sizeof words, "pointer to a non-virtual member: address and adjustment");
  memcpy(&real, words, sizeof real);
  (this->*real)(std::move(state), depend);
}
