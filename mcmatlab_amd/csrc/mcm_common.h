// Shared host utilities of libmcm: thread-local error text, HIP call checks,
// device selection.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdio>
#include <string>

#include "mcm_abi.h"

namespace mcm {

void set_error(const char* fmt, ...);
int fail(int code, const char* fmt, ...);

// Evaluate a HIP call; on failure record the error and return MCM_ERR_DEVICE
// (or MCM_ERR_OUT_OF_MEMORY) from the enclosing function.
#define MCM_HIP(call)                                                                               \
  do {                                                                                              \
    hipError_t e_ = (call);                                                                         \
    if (e_ != hipSuccess) {                                                                         \
      return ::mcm::fail(e_ == hipErrorOutOfMemory ? MCM_ERR_OUT_OF_MEMORY : MCM_ERR_DEVICE,        \
                         "%s failed: %s (%s:%d)", #call, hipGetErrorString(e_), __FILE__, __LINE__); \
    }                                                                                               \
  } while (0)

// Select `device` and check it is a gfx950 part.
int use_device(int device);
int cu_count(int device);

#ifdef __HIP__
// Between stores to LDS by some lanes of a wavefront and loads of them by others,
// and back.  A wavefront's LDS operations execute in their order, so no
// instruction is needed; it keeps the compiler from moving them.
__device__ inline void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
}
#endif

// Downloads of large arrays through pinned memory that a plan keeps (16 MB,
// allocated by its first large download and freed with it).  The runtime's own
// copy into pageable memory pins and faults in the pages from one thread:
// 10 GB/s into fresh ones.  Here a few threads each copy a stripe of the array
// out of two pinned blocks of their own that the stream fills in turn.
// 64 MB: 6.6 ms by the runtime, 3.8 into pages that are there, 2.2 so.  A first
// download below 8 MB would not pay for the pinned memory (a call with 4 MB of
// results 3.5 ms for 3.4).
class HostStage {
 public:
  HostStage() = default;
  HostStage(const HostStage&) = delete;
  HostStage& operator=(const HostStage&) = delete;
  ~HostStage();
  // dst[0 .. bytes) = src on the device, after the work on `s` so far; complete
  // when it returns.
  int download(void* dst, const void* src, size_t bytes, int device, hipStream_t s);

 private:
  static constexpr int kThreads = 4, kBlocks = 2;
  static constexpr size_t kBlock = 2 << 20;
  // smaller arrays: the runtime's copy (without the pinned memory / with it)
  static constexpr size_t kLarge = 8 << 20, kMedium = 2 << 20;
  hipError_t stripe(char* dst, const char* src, size_t bytes, int device, hipStream_t s, int t);
  char* pinned_ = nullptr;
  hipEvent_t done_[kThreads][kBlocks] = {};
};

}  // namespace mcm
