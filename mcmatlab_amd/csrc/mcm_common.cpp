// Library-wide entry points of libmcm (errors, version, devices).
#include "mcm_common.h"

#include <algorithm>
#include <thread>

#include <cstdlib>
#include <cstring>

namespace mcm {

static thread_local char g_error[1024];

void set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_error, sizeof g_error, fmt, ap);
  va_end(ap);
}

int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_error, sizeof g_error, fmt, ap);
  va_end(ap);
  return code;
}

int use_device(int device) {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess || n == 0) return fail(MCM_ERR_NO_DEVICE, "no HIP device visible");
  if (device < 0 || device >= n) return fail(MCM_ERR_INVALID_ARGUMENT, "GPUdevice %d out of range (0..%d)", device, n - 1);
  MCM_HIP(hipSetDevice(device));
  hipDeviceProp_t prop;
  MCM_HIP(hipGetDeviceProperties(&prop, device));
  if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0)
    return fail(MCM_ERR_NO_DEVICE, "device %d is %s; this build targets gfx950", device, prop.gcnArchName);
  return MCM_OK;
}

int cu_count(int device) {
  int cus = 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess) return 256;
  return cus;
}

HostStage::~HostStage() {
  for (auto& t : done_)
    for (hipEvent_t e : t)
      if (e) (void)hipEventDestroy(e);
  if (pinned_) (void)hipHostFree(pinned_);
}

hipError_t HostStage::stripe(char* dst, const char* src, size_t bytes, int device, hipStream_t s, int t) {
  hipError_t e = hipSetDevice(device);
  char* const block = pinned_ + (size_t)t * kBlocks * kBlock;
  const int64_t n = (int64_t)((bytes + kBlock - 1) / kBlock);
  auto size = [&](int64_t k) { return std::min(kBlock, bytes - (size_t)k * kBlock); };
  auto fill = [&](int64_t k) {
    if (e != hipSuccess || k >= n) return;
    const int b = (int)(k % kBlocks);
    e = hipMemcpyAsync(block + b * kBlock, src + (size_t)k * kBlock, size(k), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipEventRecord(done_[t][b], s);
  };
  for (int64_t k = 0; k < kBlocks; ++k) fill(k);
  for (int64_t k = 0; k < n && e == hipSuccess; ++k) {
    const int b = (int)(k % kBlocks);
    e = hipEventSynchronize(done_[t][b]);
    if (e != hipSuccess) break;
    std::memcpy(dst + (size_t)k * kBlock, block + b * kBlock, size(k));
    fill(k + kBlocks);
  }
  return e;
}

int HostStage::download(void* dst, const void* src, size_t bytes, int device, hipStream_t s) {
  bool staged = bytes >= (pinned_ ? kMedium : kLarge);
  if (staged && !pinned_) {
    staged = hipHostMalloc((void**)&pinned_, kThreads * kBlocks * kBlock, hipHostMallocDefault) == hipSuccess;
    for (auto& t : done_)
      for (hipEvent_t& ev : t)
        if (staged && !ev) staged = hipEventCreateWithFlags(&ev, hipEventDisableTiming) == hipSuccess;
    if (!staged) {
      // no pinned memory to be had: the runtime's copy
      (void)hipGetLastError();
      if (pinned_) (void)hipHostFree(pinned_);
      pinned_ = nullptr;
    }
  }
  if (!staged) {
    MCM_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s));
    MCM_HIP(hipStreamSynchronize(s));
    return MCM_OK;
  }
  const size_t part = ((bytes + kThreads - 1) / kThreads + 4095) & ~(size_t)4095;
  hipError_t err[kThreads] = {};
  std::thread th[kThreads];
  auto run = [&](int t) {
    const size_t lo = std::min(bytes, t * part), hi = std::min(bytes, lo + part);
    if (hi > lo) err[t] = stripe((char*)dst + lo, (const char*)src + lo, hi - lo, device, s, t);
  };
  for (int t = 1; t < kThreads; ++t) {
    try {
      th[t] = std::thread(run, t);
    } catch (...) {  // no thread to be had (or no memory to start one): its stripe here
      run(t);
    }
  }
  run(0);
  for (auto& t : th)
    if (t.joinable()) t.join();
  for (hipError_t e : err)
    if (e != hipSuccess) {
      // copies of the other stripes, or this one's other block, may be under way
      (void)hipStreamSynchronize(s);
      MCM_HIP(e);
    }
  return MCM_OK;
}

}  // namespace mcm

extern "C" {

const char* mcm_last_error(void) { return mcm::g_error; }

int mcm_version(void) { return MCM_ABI_VERSION; }

int mcm_device_count(void) {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess) return 0;
  int good = 0;
  for (int d = 0; d < n; ++d) {
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, d) == hipSuccess && std::strncmp(prop.gcnArchName, "gfx950", 6) == 0) ++good;
  }
  return good;
}

void mcm_free(void* p) { std::free(p); }

}  // extern "C"
