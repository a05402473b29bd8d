// Differentiable absorbed power (no reference counterpart; the photon
// physics is the transport kernel's, mc_photon.h).
//
// J = absorbed power inside a box of voxels, per watt of source power, with
// the per-voxel absorption coefficients mua_v (an optional map overriding the
// media table) and the scattering coefficients of every medium scaled by s:
//   dJ/dmua_v   pathwise: mua only changes packet weights, never paths.  A
//               sub-step k of length s_k in voxel v_k (weight w_k before,
//               w_k+1 after, deposit d_k) contributes
//                 -s_k * (box deposits of the packet after sub-step k)
//                 + [v_k in box] * w_k+1 * s_k
//               to dJ/dmua_(v_k).  Russian roulette keeps the expectation for
//               every weight, so the estimator stays unbiased.
//   dJ/dlog s   likelihood ratio: every flight ends in an interaction with
//               density mus exp(-tau) or is cut off with probability
//               exp(-tau), so d log p(path)/d log s = K - tau_total (K
//               interactions, tau_total the optical depth traversed); the
//               estimator is J_packet * (K - tau_total).
// Each packet runs twice with the same Philox stream: pass 1 finds the
// packet's box deposit D, pass 2 replays the path and adds the dJ/dmua terms
// with FP64 atomics (only packets with D > 0 are replayed).  Both passes run
// the same instructions (the pass is a runtime flag), so pass 2 retraces
// pass 1's path exactly; the file is built without FMA contraction.
//
// Lanes are persistent and each packet is a small state machine like the
// transport's: FETCH (take the next packet number, one atomic per wavefront,
// or the lane's own packet again for pass 2), MOVE (one voxel sub-step, with
// an interface crossed), SCATTER (roulette + deflection).  Each iteration the wavefront runs one state for the lanes in
// it (MOVE while 30 % of the live lanes want to move, otherwise the
// state with more waiting lanes), so a wavefront never waits for its
// longest-lived packet before starting others.
//
// 10^6 packets on 128^3 (pass 1 alone 5.7 ms): 16.6 ms with one
// term per lane added when a packet leaves a voxel, 11.0 ms with the terms
// parked (GradTerms) and a copy of the gradient per XCD (10^7: 0.185 and 0.107 to 0.160 s).
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <vector>

#include "mc_engine.h"
#include "mc_plan.h"

namespace mcm {

struct GradArgs {
  const float* muaMap;  // per voxel in the plan's order, or null
  int box[6];           // x0, x1, y0, y1, z0, z1
  uint64_t firstPacket, nPackets;  // of the launch
  uint32_t key0, key1, stream;
  double* grad;         // per voxel in the plan's order: sum over packets of dJ_packet/dmua
  int copies;           // of grad, one per group of XCDs
  int64_t LB;           // voxels of a copy
  double* sums;         // [4] sum D, sum D^2, sum D*S, sum (D*S)^2
  unsigned* aborted;
  unsigned long long* next;  // next packet number to hand out
  int replay;                // run pass 2 (dJ/dmua requested)
};

// The packets' launches, one record each (both passes of a packet start from
// it).  Kept out of mc_grad: launchPhoton inlined there twice took 139 registers
// a lane, three wavefronts a SIMD.
__global__ void __launch_bounds__(256) mc_grad_launch(McParams p, GradArgs g, LaunchRecord* __restrict__ rec) {
  PacketRng R;
  R.key0 = g.key0;
  R.key1 = g.key1;
  R.stream = g.stream;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; k < g.nPackets; k += stride) {
    if (__hip_atomic_load(g.aborted, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) break;
    R.start(g.firstPacket + k);
    Photon P;
    const bool ok = launch(P, p, p.media, R);
    LaunchRecord L;
    pack_launch(P, R, ok, L);
    rec[k] = L;
    if (!ok) atomicOr(g.aborted, 1u);
  }
}

__device__ inline unsigned long long grad_bcast64(unsigned long long v, int src) {
  const unsigned lo = __shfl((unsigned)v, src), hi = __shfl((unsigned)(v >> 32), src);
  return ((unsigned long long)hi << 32) | lo;
}

// Lanes in MOVE that keep the wavefront there, as a share of the live ones
// (mcm_mc_plan::moveFrac).
constexpr float kStay = 0.3f;

// Gradient terms that a lane parks in LDS and the wavefront then adds with 8
// lanes a packet (the transport's DeferSink has the reason); odd pitch against
// bank conflicts.
constexpr int kTerms = 8, kTermPitch = 9;
struct GradTerms {
  double v[256 * kTermPitch];
  int j[256 * kTermPitch];
};

__device__ inline void add_terms(double* grad, const GradTerms& t, int& n) {
  using GlobalDouble = __attribute__((address_space(1))) double;
  const int lane = __lane_id(), base = threadIdx.x & ~63;
  wave_lds_fence();
#pragma unroll 2
  for (int r = 0; r < kTerms; ++r) {
    const int src = r * (64 / kTerms) + lane / kTerms, slot = lane % kTerms;
    if (slot < __shfl(n, src, 64)) {
      const int k = (base + src) * kTermPitch + slot;
      (void)__builtin_amdgcn_global_atomic_fadd_f64((GlobalDouble*)(grad + t.j[k]), t.v[k]);
    }
  }
  wave_lds_fence();
  n = 0;
}

template <bool FRESNEL>
__global__ void __launch_bounds__(256, 4) mc_grad(McParams p, GradArgs g, const LaunchRecord* __restrict__ launches) {
  __shared__ Medium sMed[256];
  __shared__ uint8_t sCdf[256];
  __shared__ double sSum[4][256];
  __shared__ GradTerms sTerms;
  for (int k = threadIdx.x; k < p.nM; k += blockDim.x) {
    sMed[k] = p.media[k];
    sCdf[k] = p.cdfIdx[k];
  }
  const int t = threadIdx.x;
  for (int q = 0; q < 4; ++q) sSum[q][t] = 0.0;
  __syncthreads();
  constexpr int G_FETCH = 0, G_MOVE = 1, G_SCATTER = 2, G_DONE = 3;
  const int lane = __lane_id();
  PacketRng R;
  R.key0 = g.key0;
  R.key1 = g.key1;
  R.stream = g.stream;
  Photon P;
  int st = G_FETCH;
  bool pass2 = false, again = false;  // again: the lane fetches its own packet for pass 2
  uint64_t k = 0;
  double D = 0.0, tau = 0.0;  // pass 1: box deposit, optical depth; pass 2: box deposits still to come
  uint32_t K = 0;
  int nTerms = 0, parked = 0;  // terms parked by the lane, by any lane at most
  bool boxed = false;  // the packet's voxel is in the box (and the packet in the volume)
  double* const grad = g.grad + (size_t)(xcd() % g.copies) * g.LB;
  // spread few packets over the wavefronts (launch_blocks)
  {
    const unsigned long long waves = (unsigned long long)gridDim.x * (blockDim.x / 64);
    if ((unsigned long long)lane * waves >= g.nPackets) st = G_DONE;
  }
  auto in_box = [&]() {
    const int ix = clamp_axis(P.i[0], p.n[0]), iy = clamp_axis(P.i[1], p.n[1]), iz = clamp_axis(P.i[2], p.n[2]);
    return P.insideVolume & (ix >= g.box[0]) & (ix < g.box[1]) & (iy >= g.box[2]) & (iy < g.box[3]) & (iz >= g.box[4]) & (iz < g.box[5]);
  };
  auto set_voxel = [&](int j, int m, float mua) {
    P.j = j;
    const Medium md = sMed[m];
    P.mua = g.muaMap ? mua : md.mua;
    P.mus = md.mus;
    P.g = md.g;
    P.cdf = sCdf[m];
    boxed = in_box();
  };
  // checkEscape + getNewVoxelProperties after a boundary was crossed
  auto enter = [&](int j, int m, float mua) {
    const float x = P.i[0], y = P.i[1];
    check_escape(P, p);
    if (!P.alive) return;
    if (p.boundaryType == 3 && (P.i[0] != x || P.i[1] != y)) {  // wrapped to the other side
      j = voxel_of(p, P.i);
      m = p.M[j];
      if (g.muaMap) mua = g.muaMap[j];
    }
    set_voxel(j, m, mua);
  };
  // the packet goes on with its next state, or its pass ended
  auto settle = [&]() {
    st = P.stepLeft > 0.f ? G_MOVE : G_SCATTER;
    if (!P.alive) {
      st = G_FETCH;
      if (!pass2) {
        const double S = (double)K - tau;
        sSum[0][t] += D;
        sSum[1][t] += D * D;
        sSum[2][t] += D * S;
        sSum[3][t] += (D * S) * (D * S);
        again = D > 0.0 && g.replay;
      }
    }
  };
  for (;;) {
    const unsigned long long bFetch = __ballot(st == G_FETCH);
    const unsigned long long bMove = __ballot(st == G_MOVE);
    const unsigned long long bScat = __ballot(st == G_SCATTER);
    const int cF = __popcll(bFetch), cM = __popcll(bMove), cS = __popcll(bScat);
    const int active = cF + cM + cS;
    if (active == 0) break;
    int phase = G_MOVE;
    const int stay = max(1, (int)ceilf(kStay * (float)active));
    if (cM < stay) {
      int best = cM;
      if (cS > best) { best = cS; phase = G_SCATTER; }
      if (cF > best) phase = G_FETCH;
    }
    if (phase == G_MOVE) do {
      if (st == G_MOVE) {
        if (P.substeps >= kMaxSubsteps) {
          P.alive = false;
        } else {
          const float mus = P.mus;
          const float s = advance(P, p);
          int jNew = P.j, mNew = 0;
          float muaNew = 0.f;
          if (!P.sameVoxel) {
            jNew = voxel_of(p, P.i);
            mNew = p.M[jNew];
            if (g.muaMap) muaNew = g.muaMap[jNew];
          }
          const float absorbed = absorb(P, s);
          if (!pass2) {
            tau += (double)s * (double)mus;
            if (boxed) D += (double)absorbed;
          } else {
            if (boxed) D -= (double)absorbed;
            double gv = -(double)s * D;
            if (boxed) gv += (double)P.weight * (double)s;
            sTerms.j[t * kTermPitch + nTerms] = P.j;
            sTerms.v[t * kTermPitch + nTerms] = gv;
            ++nTerms;
          }
          if (!P.sameVoxel) {
            // (at once: a packet trapped between two indices meets an interface at
            // every sub-step, and a state of its own would double its time)
            if (FRESNEL && P.ri != sMed[mNew].ri) fresnel(P, p, sMed, jNew, mNew, R);
            enter(jNew, mNew, muaNew);
          }
        }
        settle();
      }
      // a lane parks at most one term per sub-step
      if (++parked >= kTerms && __ballot(nTerms == kTerms)) {
        add_terms(grad, sTerms, nTerms);
        parked = 0;
      }
    } while (__popcll(__ballot(st == G_MOVE)) >= stay);
    else if (phase == G_SCATTER) {
      if (st == G_SCATTER) {
        ++K;  // the flight ended in an interaction
        roulette_scatter(P, p, p.cdfs, 0, R);
        settle();
      }
    } else {
      const unsigned long long bNew = __ballot(st == G_FETCH && !again);
      unsigned long long base = 0;
      if (bNew) {
        const int leader = __ffsll((long long)bNew) - 1;
        if (lane == leader) {
          base = atomicAdd(g.next, (unsigned long long)__popcll(bNew));
          if (atomicAdd(g.aborted, 0u)) base = g.nPackets;  // a failed launch stops the run
        }
        base = grad_bcast64(base, leader);
      }
      if (st == G_FETCH) {
        pass2 = again;
        if (!again) {
          k = base + (unsigned long long)__popcll(bNew & ((1ull << lane) - 1ull));
          D = 0.0;
          tau = 0.0;
          K = 0;
        }
        again = false;
        if (k >= g.nPackets) {
          st = G_DONE;
        } else {
          const LaunchRecord L = launches[k];
          R.start(g.firstPacket + k);
          unpack_launch(L, P, R);
          set_crossing_lengths(P, p);
          const int j = voxel_of(p, P.i);
          set_voxel(j, p.M[j], g.muaMap ? g.muaMap[j] : 0.f);
          settle();
        }
      }
    }
  }
  add_terms(grad, sTerms, nTerms);
  // wavefront then workgroup reduction of the four sums
  __syncthreads();
  if (t < 4) {
    double sum = 0.0;
    for (int q = 0; q < 256; ++q) sum += sSum[t][q];
    unsafeAtomicAdd(&g.sums[t], sum);
  }
}

// dJ/dmua in linear order, the copies summed, scaled to power / N
__global__ void mc_grad_output(double* out, const double* grad, int copies, int64_t LB, VoxelMap map, double power, double N, int64_t L) {
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= L) return;
  const int64_t i = map(j);
  double sum = 0.0;
  for (int c = 0; c < copies; ++c) sum += grad[c * LB + i];
  out[j] = power * sum / N;
}

}  // namespace mcm

using namespace mcm;

// Largest number of packets per launch (64-byte records).
constexpr uint64_t kGradLaunchPackets = 1ull << 22;

// Records for n packets, or fewer (then n becomes that) where there is no memory
// for as many.
static int ensure_grad_records(mcm_mc_plan* pl, uint64_t& n) {
  if (n <= pl->gradRecCap) return MCM_OK;
  MCM_HIP(hipStreamSynchronize(pl->stream));
  for (;; n = (n + 1) / 2) {
    free_buf(pl->gradRec);
    pl->gradRecCap = 0;
    if (hipMalloc(&pl->gradRec.p, (size_t)n * sizeof(LaunchRecord)) == hipSuccess) break;
    (void)hipGetLastError();
    if (n <= kFewestLaunchPackets) return fail(MCM_ERR_OUT_OF_MEMORY, "Error: Out of memory (packet records for %llu packets)", (unsigned long long)n);
  }
  pl->gradRecCap = n;
  return MCM_OK;
}

extern "C" int mcm_mc_grad_run(mcm_mc_plan* pl, const mcm_mc_grad_input* in, mcm_mc_grad_output* out) {
  if (!pl || !in || !out) return fail(MCM_ERR_INVALID_ARGUMENT, "null argument");
  McTables& T = pl->T;
  if (pl->prm.criteriaActive) return fail(MCM_ERR_UNSUPPORTED, "gradients run without deposition criteria");
  if (in->iL < 0 || in->iL >= T.nL) return fail(MCM_ERR_INVALID_ARGUMENT, "wavelength index out of range");
  if (in->nPhotons < 2) return fail(MCM_ERR_INVALID_ARGUMENT, "nPhotons must be at least 2");
  const int64_t n3[3] = {T.nx, T.ny, T.nz};
  for (int a = 0; a < 3; ++a)
    if (in->box[2 * a] < 0 || in->box[2 * a + 1] > n3[a] || in->box[2 * a] >= in->box[2 * a + 1])
      return fail(MCM_ERR_INVALID_ARGUMENT, "box must satisfy 0 <= lo < hi <= grid size on every axis");
  if (in->muaMap)
    for (int64_t k = 0; k < T.L; ++k)
      if (!(in->muaMap[k] >= 0.f)) return fail(MCM_ERR_INVALID_ARGUMENT, "muaMap must be non-negative");
  MCM_HIP(hipSetDevice(pl->device));
  int rc = select_wavelength(pl, in->iL);
  if (rc) return rc;
  hipStream_t s = pl->stream;
  // device buffers live in the plan across calls: the map and the gradient in
  // the plan's voxel order, one linear buffer that the map is uploaded through
  // and the gradient downloaded from, and 64 bytes for the four sums, the abort
  // flag and the packet counter
  const int64_t LB = pl->prm.LB;
  const unsigned gL = (unsigned)((T.L + 255) / 256);
  if (!pl->gradOut.p) {
    if (!pl->gradMap.p) MCM_HIP(hipMalloc(&pl->gradMap.p, (size_t)LB * sizeof(float)));
    if (!pl->gradLin.p) MCM_HIP(hipMalloc(&pl->gradLin.p, (size_t)T.L * sizeof(double)));
    if (!pl->gradSmall.p) MCM_HIP(hipMalloc(&pl->gradSmall.p, 64));
    pl->gradCopies = start_copies(LB);
    if ((rc = zero_copies(pl->gradOut, pl->gradCopies, LB, s))) return rc;
  }
  const int copies = pl->gradCopies;
  if (in->muaMap) {
    MCM_HIP(hipMemcpyAsync(pl->gradLin.p, in->muaMap, (size_t)T.L * sizeof(float), hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(mc_to_bricks<float>, dim3(gL), dim3(256), 0, s, pl->gradMap.as<float>(), pl->gradLin.as<float>(), voxel_map(pl), T.L);
    MCM_HIP(hipGetLastError());
  }
  MCM_HIP(hipMemsetAsync(pl->gradOut.p, 0, (size_t)copies * LB * sizeof(double), s));
  MCM_HIP(hipMemsetAsync(pl->gradSmall.p, 0, 64, s));
  char* small = (char*)pl->gradSmall.p;
  GradArgs g;
  std::memset(&g, 0, sizeof g);
  g.muaMap = in->muaMap ? pl->gradMap.as<float>() : nullptr;
  for (int a = 0; a < 6; ++a) g.box[a] = (int)in->box[a];
  g.key0 = (uint32_t)in->seed;
  g.key1 = (uint32_t)(in->seed >> 32);
  g.stream = (uint32_t)in->iL;
  g.grad = pl->gradOut.as<double>();
  g.copies = copies;
  g.LB = LB;
  g.sums = (double*)small;                          // bytes 0..31
  g.next = (unsigned long long*)(small + 32);       // bytes 32..39
  g.aborted = (unsigned*)(small + 40);              // bytes 40..43
  g.replay = out->dJ_dmua != nullptr;              // J and dJ/dlog s need pass 1 only
  int per = 0;
  const void* kern = T.fresnelPossible ? (const void*)mc_grad<true> : (const void*)mc_grad<false>;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kern, 256, 0) != hipSuccess || per < 1) per = 2;
  uint64_t most = kGradLaunchPackets;
  for (uint64_t done = 0; done < in->nPhotons; done += g.nPackets) {
    g.firstPacket = done;
    g.nPackets = std::min<uint64_t>(in->nPhotons - done, most);
    const uint64_t asked = g.nPackets;
    if ((rc = ensure_grad_records(pl, g.nPackets))) return rc;
    if (g.nPackets < asked) most = g.nPackets;
    if (done) MCM_HIP(hipMemsetAsync(g.next, 0, sizeof *g.next, s));
    LaunchRecord* rec = pl->gradRec.as<LaunchRecord>();
    const dim3 b(256), grid(launch_blocks(pl, per * cu_count(pl->device), g.nPackets));
    hipLaunchKernelGGL(mc_grad_launch, grid, b, 0, s, pl->prm, g, rec);
    if (T.fresnelPossible) hipLaunchKernelGGL(mc_grad<true>, grid, b, 0, s, pl->prm, g, rec);
    else hipLaunchKernelGGL(mc_grad<false>, grid, b, 0, s, pl->prm, g, rec);
    MCM_HIP(hipGetLastError());
  }
  unsigned char hs[64];
  MCM_HIP(hipMemcpyAsync(hs, small, 64, hipMemcpyDeviceToHost, s));
  const double N = (double)in->nPhotons;
  const double power = T.spectrum[(size_t)in->iL];
  if (out->dJ_dmua) {
    hipLaunchKernelGGL(mc_grad_output, dim3(gL), dim3(256), 0, s, pl->gradLin.as<double>(), pl->gradOut.as<double>(), copies, LB, voxel_map(pl), power, N, T.L);
    MCM_HIP(hipGetLastError());
    if ((rc = pl->stage.download(out->dJ_dmua, pl->gradLin.p, (size_t)T.L * sizeof(double), pl->device, s))) return rc;
  }
  MCM_HIP(hipStreamSynchronize(s));
  double sums[4];
  unsigned aborted = 0;
  std::memcpy(sums, hs, sizeof sums);
  std::memcpy(&aborted, hs + 40, sizeof aborted);
  if (aborted) return fail(MCM_ERR_INVALID_ARGUMENT, "all packets launch outside the simulation cuboid");
  auto se = [&](double sx, double sx2) { return power * std::sqrt(std::max(0.0, sx2 - sx * sx / N) / (N * (N - 1))); };
  out->J = power * sums[0] / N;
  out->J_se = se(sums[0], sums[1]);
  out->dJ_dlogmus = power * sums[2] / N;
  out->dJ_dlogmus_se = se(sums[2], sums[3]);
  return MCM_OK;
}
