// The device-resident Monte Carlo plan shared by the transport
// (mc_kernel.hip) and the gradient (mc_grad.hip) translation units: device
// buffers of the model, tallies, counters and launch parameters.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "mc_photon.h"
#include "mc_setup.h"
#include "mcm_common.h"

namespace mcm {

struct McCounters {
  unsigned long long nextPacket;  // reset before every launch
  unsigned long long launched;
  unsigned long long collected;
  unsigned long long substeps;
  unsigned long long scatters;
  unsigned long long interfaces;
  unsigned int aborted;
  unsigned int runaway;
};

struct McLaunch {
  uint64_t firstPacket;
  uint64_t nPackets;
  uint32_t key0, key1, stream;
  float moveFrac;
  McCounters* ctr;
};

}  // namespace mcm

struct DevBuf {
  void* p = nullptr;
  ~DevBuf() {
    if (p) (void)hipFree(p);
  }
  template <typename T>
  T* as() const { return (T*)p; }
};

struct mcm_mc_plan {
  int device = 0;
  hipStream_t stream = nullptr;
  mcm::McTables T;
  mcm::McParams prm;
  int blocks = 0, blocksForced = 0, threads = 256;
  // share of the live lanes whose wish to move keeps a wavefront at it: 10^4
  // packets take 0.98 ms with 0.5, 0.89 with 0.3, 0.92 with 0.1; a run without
  // fluence (4 10^6, 200^3) 21.8, 20.9 and 26.5
  float moveFrac = 0.3f;
  DevBuf M, Mlin, normals, media, cdfIdx, cdfs, fpid1, aid1, fpid2, aid2, S, muaNorm;
  DevBuf nfrLin;   // linear copy of the fluence tally for mcm_mc_plan_tallies
  DevBuf NFR, image, FF, NI[6], counters, nfrOut;
  DevBuf launchRec, escapeRec;  // per-launch packet records (of escapes: without deposition criteria)
  DevBuf gradMap, gradLin, gradOut, gradSmall;  // gradient runs: mua map, its linear form, dJ/dmua, sums/flags/counter
  int gradCopies = 1;
  DevBuf gradRec;  // launch records of a gradient run
  uint64_t recCap = 0, escapeCap = 0, gradRecCap = 0;
  std::vector<double> Shost;   // cumulative 3D source table of the current wavelength
  const float* sourceDistribution = nullptr;
  double power = 0;            // current wavelength's source power
  int curL = -1;
  uint64_t lastLaunched = 0, lastCollected = 0;
  mcm::McCounters stats{};
  mcm::HostStage stage;
  ~mcm_mc_plan() {
    if (stream) (void)hipStreamDestroy(stream);
  }
};

namespace mcm {

template <typename T>
inline int upload(DevBuf& b, const T* src, size_t n, hipStream_t s) {
  if (b.p) {
    MCM_HIP(hipFree(b.p));
    b.p = nullptr;
  }
  MCM_HIP(hipMalloc(&b.p, std::max<size_t>(n, 1) * sizeof(T)));
  if (src && n) MCM_HIP(hipMemcpyAsync(b.p, src, n * sizeof(T), hipMemcpyHostToDevice, s));
  return MCM_OK;
}

inline int zeros(DevBuf& b, size_t bytes, hipStream_t s) {
  if (b.p) {
    MCM_HIP(hipFree(b.p));
    b.p = nullptr;
  }
  MCM_HIP(hipMalloc(&b.p, std::max<size_t>(bytes, 8)));
  MCM_HIP(hipMemsetAsync(b.p, 0, std::max<size_t>(bytes, 8), s));
  return MCM_OK;
}

inline void free_buf(DevBuf& b) {
  if (b.p) (void)hipFree(b.p);
  b.p = nullptr;
}

// A run is cut into launches whose packet records there is memory for, of at
// least this many packets.
constexpr uint64_t kFewestLaunchPackets = 1ull << 12;

// Voxel order of a plan for kernels that walk the grid in its linear (x
// fastest) order.
struct VoxelMap {
  int nx, ny, nbx, nbxy;
  __host__ __device__ int64_t operator()(int64_t j) const {
    if (!nbx) return j;
    const int x = (int)(j % nx), y = (int)(j / nx % ny), z = (int)(j / nx / ny);
    return brick_index(x, y, z, nbx, nbxy);
  }
};
inline VoxelMap voxel_map(const mcm_mc_plan* pl) { return {pl->T.nx, pl->T.ny, pl->prm.nbx, pl->prm.nbxy}; }

// out[map(j)] = in[j] (to the plan's voxel order)
template <typename T>
__global__ void mc_to_bricks(T* out, const T* in, VoxelMap map, int64_t L) {
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j < L) out[map(j)] = in[j];
}

// The accelerator complex die (XCD) the wavefront runs on; each XCD has its own
// L2, so XCD-private copies of a tally keep hot voxels from being contended
// across XCDs.
__device__ inline int xcd() {
  unsigned r;
  asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(r));
  return (int)(r & 7u);
}

// Copies of a tally of LB voxels that a plan starts with: as many as stay in
// the memory-side cache together.  A beam narrower than a voxel is bound by the
// adds to the voxels on its axis (10^6 packets, 100^3: 21.7 ms with one copy,
// 13 with two, 9.4 with eight), and broad ones do not mind (4 10^6 packets,
// 200^3: 36.1 and 35.7 ms with one and two).
constexpr int64_t kCopiesBytes = 256 << 20;
inline int start_copies(int64_t LB) {
  int n = 1;
  while (n < 8 && 2 * n * LB * (int64_t)sizeof(double) <= kCopiesBytes) n *= 2;
  return n;
}

// A cleared tally of `copies` times `stride` voxels; one copy when there is no
// memory for more.
inline int zero_copies(DevBuf& b, int& copies, int64_t stride, hipStream_t s) {
  int rc = zeros(b, (size_t)copies * stride * sizeof(double), s);
  if (rc && copies > 1) {
    (void)hipGetLastError();
    copies = 1;
    rc = zeros(b, (size_t)stride * sizeof(double), s);
  }
  return rc;
}

// Workgroups of a launch of n packets: as many as the packets fill, but at
// least one per CU, over whose wavefronts the packets are then spread, and at
// most `blocks`, which are resident together.  A wavefront runs one state per
// iteration, so a packet waits for the others of its wavefront, and a launch
// lasts as long as its longest-lived packets: 10^4 packets in 157 full
// wavefronts take 1.39 ms, over 1024 wavefronts 0.97 ms.  With more than a
// wavefront per SIMD those share the issue slots instead (10^5 packets over
// 4096 wavefronts are slower than over 1563 full ones).
inline int launch_blocks(const mcm_mc_plan* pl, int blocks, uint64_t n) {
  if (pl->blocksForced) return blocks;
  const uint64_t filled = (n + pl->threads - 1) / pl->threads, cus = (uint64_t)cu_count(pl->device);
  return (int)std::min<uint64_t>((uint64_t)blocks, std::max(filled, cus));
}

// Select medium table, source table and refractive indices of wavelength iL
// (mc_kernel.hip).
int select_wavelength(mcm_mc_plan* pl, int64_t iL);

}  // namespace mcm
