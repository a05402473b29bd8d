// Heat diffusion + Arrhenius damage on gfx950: kernels and the C ABI
// (mcm_heat_plan_*, mcm_heat_run).  Replaces finiteElementHeatPropagator.c
// (+MCmatlab/src/finiteElementHeatPropagator.c:688-821).
//
// One Douglas-Gunn ADI step (:767-782) is three line-sweep kernels instead of
// the reference's six loops:
//   x sweep   substeps 1a + 1b: the explicit right-hand side (full 7-point
//             stencil, x half-weighted, plus the source) built on the fly and
//             solved along x;
//   y sweep   substeps 2a + 2b: the -dt/2 L_y correction and the y solve;
//   z sweep   substeps 3a + 3b: the -dt/2 L_z correction, the z solve, the
//             Arrhenius damage update and the per-medium maximum temperature.
// FP64 (default), lines of up to 512 voxels: the sweeps solve for increments
// (below) by a partition method with parallel cyclic reduction between the
// chunks of a line; along x a wavefront holds contiguous voxels, along y and z
// a workgroup holds 16 neighbouring lines in registers.  FP32 (the reference's
// arithmetic) and longer lines: one lane per line running the Thomas
// recurrence over blocks of loaded elements; FP32 lines of up to 431 voxels
// (line32_lines) run it on lines staged in LDS.
// The explicit (forward Euler) scheme is one kernel per step.
//
// Arithmetic follows the reference's expressions (built without FMA
// contraction); in FP32 it is the reference's operation for operation.
// Per-medium maxima use an order-preserving integer key of the FP64 value:
// each lane keeps a running maximum over its current run of one medium and
// folds it into LDS when the medium changes; each workgroup folds LDS into
// the global keys at the end.
// The discrete adjoint of the FP64 DG-ADI step (transposed line solves and
// stencils) follows the forward kernels.
#include <hip/hip_runtime.h>

#include <array>
#include <map>
#include <mutex>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <type_traits>
#include <vector>

#include "mcm_common.h"

namespace mcm {

constexpr int kHeatTPB = 256;

__host__ __device__ inline unsigned long long order_key(double v) {
  unsigned long long b;
  memcpy(&b, &v, 8);
  return (b >> 63) ? ~b : (b | 0x8000000000000000ull);
}
__host__ __device__ inline double key_value(unsigned long long k) {
  const unsigned long long b = (k >> 63) ? (k & 0x7FFFFFFFFFFFFFFFull) : ~k;
  double v;
  memcpy(&v, &b, 8);
  return v;
}

template <typename RT>
struct HeatArgs {
  int nx, ny, nz, nM;
  int sinked, lightsOn, calcDamage;
  RT dt;
  RT Rgas, czero;
  const uint8_t* M;
  const float* Q;        // dTdt_abs
  const RT* c;           // [nM * nM * 3]: c[a + b nM + d nM^2]
  const RT* logA;
  const RT* E;
  const RT* T1;          // temperature at the start of the step
  RT* T2;                // result (and intermediate) of the step
  RT* B;                 // Thomas scratch: forward-eliminated diagonal
  float* fac[3];         // FP32: eliminated diagonals of the x, y and z lines for this dt
  RT* Om;                // damage integral (calcDamage)
  unsigned long long* maxKey;  // [nM] order_key of the running maximum
  // sensor record of T1 (the state before the step), written by the first
  // workgroup of the step's first kernel: column sCol (+ *sColBase)
  int nS;
  const long long* sIdx;
  const RT* sW;
  double* sOut;
  const long long* sColBase;
  long long sCol;
};

// recordTempSensors (:652-663): trilinear interpolation of T into column
// `col` of the sensor record, sensors s = first, first + step, ...
template <typename RT>
__device__ inline void sensors_at(const RT* T, int nx, int nxy, const long long* idx, const RT* w, int nS, double* out, long long col,
                                  int first, int step) {
  for (int s = first; s < nS; s += step) {
    const long long k = idx[s];
    const RT wx = w[s], wy = w[s + nS], wz = w[s + 2 * nS];
    out[s + col * nS] = (double)((1 - wx) * (1 - wy) * (1 - wz) * T[k] + (1 - wx) * (1 - wy) * wz * T[k + nxy] +
                                 (1 - wx) * wy * (1 - wz) * T[k + nx] + (1 - wx) * wy * wz * T[k + nx + nxy] +
                                 wx * (1 - wy) * (1 - wz) * T[k + 1] + wx * (1 - wy) * wz * T[k + 1 + nxy] +
                                 wx * wy * (1 - wz) * T[k + 1 + nx] + wx * wy * wz * T[k + 1 + nx + nxy]);
  }
}

// The step kernels' share of the sensor record (first workgroup only).
template <typename RT>
__device__ inline void step_sensors(const HeatArgs<RT>& a) {
  if (a.nS == 0 || blockIdx.x != 0) return;
  const long long col = a.sCol + (a.sColBase ? *a.sColBase : 0);
  sensors_at(a.T1, a.nx, a.nx * a.ny, a.sIdx, a.sW, a.nS, a.sOut, col, (int)threadIdx.x, (int)blockDim.x);
}

template <typename RT>
__device__ inline bool frozen(const HeatArgs<RT>& a, int x, int y, int z) {
  return a.sinked && (x == 0 || x == a.nx - 1 || y == 0 || y == a.ny - 1 || z == 0 || z == a.nz - 1);
}

template <typename RT>
__device__ inline RT cc(const HeatArgs<RT>& a, int m, int n, int d) {
  return a.c[m + n * a.nM + d * a.nM * a.nM];
}

// Running maxima per medium.  The keys in LDS start from the global running
// maxima, so a voxel that does not raise its medium's maximum touches no
// atomic (a stale start is harmless: the keys only grow), and a workgroup
// writes back only what it raised.  Like the reference's comparison
// (maxT < T), a NaN raises nothing.  Starting every workgroup from -inf cost
// one LDS atomic per lane and one same-address global atomic per workgroup,
// medium and step.
struct MaxRun {
  int m = -1;
  double v = 0;  // the maximum of medium m as far as this lane knows
  __device__ void add(int mm, double t, unsigned long long* s) {
    if (mm != m) {
      m = mm;
      v = key_value(__hip_atomic_load(&s[m], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
    }
    if (t > v) {
      atomicMax(&s[m], order_key(t));
      v = t;
    }
  }
};

__device__ inline void fold_lds_max(unsigned long long* s, unsigned long long* g, int nM) {
  __syncthreads();
  for (int k = threadIdx.x; k < nM; k += blockDim.x)
    if (s[k] > g[k]) atomicMax(&g[k], s[k]);
}

// Workgroup b of n, renumbered so that each of the 8 XCDs (which take
// workgroups in turn) works on consecutive ones and finds its neighbours'
// data in its own L2.
__device__ inline int xcd_contiguous(int b, int n) {
  const int q = n >> 3, r = n & 7, x = b & 7;
  return x * q + min(x, r) + (b >> 3);
}

enum : int { SWEEP_X = 0, SWEEP_Y = 1, SWEEP_Z = 2 };
constexpr int kLdsCoef = 1536;  // coefficient tables up to 22 media live in LDS

template <typename RT>
__device__ inline RT coef(const RT* c, int nM, int m, int nb, int d) {
  return c[d * nM * nM + (int)(__umul24((unsigned)nb, (unsigned)nM) + (unsigned)m)];
}

// Per-workgroup copies of the small per-medium tables.
template <typename RT>
struct HeatLds {
  RT c[kLdsCoef];
  RT logA[256];
  RT E[256];
  unsigned long long maxKey[256];
};

template <typename RT>
__device__ inline const RT* stage_tables(const HeatArgs<RT>& a, HeatLds<RT>& s) {
  const int nc = a.nM * a.nM * 3;
  if (nc <= kLdsCoef)
    for (int k = threadIdx.x; k < nc; k += blockDim.x) s.c[k] = a.c[k];
  for (int k = threadIdx.x; k < a.nM; k += blockDim.x) {
    s.logA[k] = a.logA[k];
    s.E[k] = a.E[k];
    s.maxKey[k] = a.maxKey[k];
  }
  __syncthreads();
  return nc <= kLdsCoef ? s.c : a.c;
}

// One grid line: the explicit part of the substep (KIND X: the full
// right-hand side of substep 1a; Y/Z: the -dt/2 L_d T correction of 2a/3a),
// Thomas forward elimination, back substitution, and for Z the Arrhenius
// update and the running maxima.  Expressions and their order are those of
// the reference (finiteElementHeatPropagator.c:288-646); only the memory
// access is reorganised: each lane loads a block of U consecutive elements
// of its line (and their stencil neighbours) before running the sequential
// recurrence over them, so a wavefront has U loads in flight instead of one.
//   i0, st, n : first voxel, stride and length of the line (axis d)
//   lf        : the whole line lies on a fixed-temperature boundary
//   s1/k1/n1, s2/k2/n2 : stride, coordinate and extent of the two other axes
template <typename RT, int KIND, int U>
__device__ void sweep_line(const HeatArgs<RT>& a, const RT* cT, const HeatLds<RT>& L, int i0, int st, int n, bool lf, int d, int s1,
                           int k1, int n1, int s2, int k2, int n2, MaxRun* run, unsigned long long* sMax) {
  constexpr bool kIncrement = std::is_same<RT, double>::value;  // FP64 sweeps solve for increments (see below)
  const int nM = a.nM;
  const RT dt = a.dt;
  const bool sk = a.sinked;
  RT tprev = 0, bprev = 1;
  for (int k0 = 0; k0 < n; k0 += U) {
    RT Tw[U + 2];
    int Mw[U + 2];
    RT R0[U], Ta[U], Tb[U], Tc[U], Td[U];
    int Ma[U], Mb[U], Mc[U], Md[U];
    float Qv[U];
#pragma unroll
    for (int u = 0; u < U + 2; ++u) {
      const int k = k0 - 1 + u;
      const bool ok = k >= 0 && k < n;
      const int i = i0 + k * st;
      Tw[u] = ok ? a.T1[i] : (RT)0;
      Mw[u] = ok ? (int)a.M[i] : 0;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + u;
      const bool ok = k < n;
      const int i = i0 + k * st;
      if (KIND == SWEEP_X) {
        const bool a1 = ok && k1 > 0, b1 = ok && k1 < n1 - 1, a2 = ok && k2 > 0, b2 = ok && k2 < n2 - 1;
        Ta[u] = a1 ? a.T1[i - s1] : (RT)0;
        Ma[u] = a1 ? (int)a.M[i - s1] : 0;
        Tb[u] = b1 ? a.T1[i + s1] : (RT)0;
        Mb[u] = b1 ? (int)a.M[i + s1] : 0;
        Tc[u] = a2 ? a.T1[i - s2] : (RT)0;
        Mc[u] = a2 ? (int)a.M[i - s2] : 0;
        Td[u] = b2 ? a.T1[i + s2] : (RT)0;
        Md[u] = b2 ? (int)a.M[i + s2] : 0;
        Qv[u] = ok ? a.Q[i] : 0.f;
      } else {
        R0[u] = ok ? a.T2[i] : (RT)0;
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + u;
      if (k >= n) break;
      const int i = i0 + k * st;
      const int m = Mw[u + 1];
      const bool fz = lf || (sk && (k == 0 || k == n - 1));
      RT t;
      if (KIND == SWEEP_X) {
        RT dTdt = 0;
        if (!fz) {
          dTdt = a.lightsOn ? (RT)Qv[u] : (RT)0;
          if (k != 0) dTdt += (Tw[u] - Tw[u + 1]) * coef(cT, nM, m, Mw[u], 0) / (kIncrement ? 1 : 2);
          if (k != n - 1) dTdt += (Tw[u + 2] - Tw[u + 1]) * coef(cT, nM, m, Mw[u + 2], 0) / (kIncrement ? 1 : 2);
          if (k1 != 0) dTdt += (Ta[u] - Tw[u + 1]) * coef(cT, nM, m, Ma[u], 1);
          if (k1 != n1 - 1) dTdt += (Tb[u] - Tw[u + 1]) * coef(cT, nM, m, Mb[u], 1);
          if (k2 != 0) dTdt += (Tc[u] - Tw[u + 1]) * coef(cT, nM, m, Mc[u], 2);
          if (k2 != n2 - 1) dTdt += (Td[u] - Tw[u + 1]) * coef(cT, nM, m, Md[u], 2);
        }
        t = kIncrement ? dt * dTdt : Tw[u + 1] + dt * dTdt;
      } else {
        t = R0[u];
        if (!kIncrement && !fz) {
          RT dTdt = 0;
          if (k != 0) dTdt -= (Tw[u] - Tw[u + 1]) * coef(cT, nM, m, Mw[u], d) / 2;
          if (k != n - 1) dTdt -= (Tw[u + 2] - Tw[u + 1]) * coef(cT, nM, m, Mw[u + 2], d) / 2;
          t = t + dt * dTdt;
        }
      }
      RT b = 1;
      if (!fz) {
        if (k < n - 1) b += dt / 2 * coef(cT, nM, m, Mw[u + 2], d);
        if (k > 0) {
          const int mp = Mw[u];
          b += dt / 2 * coef(cT, nM, m, mp, d);
          const RT w = -dt / 2 * coef(cT, nM, m, mp, d) / bprev;
          if (k > 1 || !sk) b += w * dt / 2 * coef(cT, nM, mp, m, d);
          t -= w * tprev;
        }
      }
      a.T2[i] = t;
      a.B[i] = b;
      tprev = t;
      bprev = b;
    }
  }
  RT xnext = 0;
  for (int kt = n - 1; kt >= 0; kt -= U) {
    RT Dv[U], Bv[U], T1v[U], Omv[U];
    int Mi[U], Mn[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = kt - u;
      const bool ok = k >= 0;
      const int i = i0 + k * st;
      Dv[u] = ok ? a.T2[i] : (RT)0;
      Bv[u] = ok ? a.B[i] : (RT)1;
      Mi[u] = ok ? (int)a.M[i] : 0;
      Mn[u] = ok && k < n - 1 ? (int)a.M[i + st] : 0;
      if (KIND == SWEEP_Z) {
        T1v[u] = ok ? a.T1[i] : (RT)0;
        Omv[u] = ok && a.calcDamage ? a.Om[i] : (RT)0;
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = kt - u;
      if (k < 0) break;
      const int i = i0 + k * st;
      const int m = Mi[u];
      const bool fz = lf || (sk && (k == 0 || k == n - 1));
      RT t = Dv[u];
      if (!fz) {
        t = (t + (k == n - 1 ? (RT)0 : dt / 2 * coef(cT, nM, m, Mn[u], d) * xnext)) / Bv[u];
        a.T2[i] = t;
      }
      xnext = t;
      if (KIND == SWEEP_Z) {
        if (kIncrement) {
          t = T1v[u] + t;
          a.T2[i] = t;
        }
        if (a.calcDamage && L.E[m] != 0) a.Om[i] = Omv[u] + dt * (RT)exp(L.logA[m] - L.E[m] / (a.Rgas * ((t + T1v[u]) / 2 + a.czero)));
        run->add(m, (double)t, sMax);
      }
    }
  }
}

constexpr int kSweepU = 8;

// FP32 sweeps of lines that fit in LDS (line32_lines).  The reference's recurrence is
// sequential along a line and is kept operation for operation, so its length
// cannot be cut; what a lane per line loses is the latency of its loads and
// the few lanes (100^3: 157 wavefronts for 256 CUs).  Here a workgroup takes TL
// lines: all its threads compute the right-hand sides and the rows'
// coefficients voxel by voxel (coalesced) into LDS, TL lanes run the recurrence
// there, and all threads write the lines back with the damage and maxima.
// 100^3: 53 us a step (three sweeps; 390 with a lane per line), of which 30
// remain without the recurrences.  Rows are read a group ahead of the recurrence
// (70 us when each group waited for its own reads).
// TL: as many lines (32, 16, 8) as fit four numbers per voxel into 54 KB: lines
// of up to 107, 215 and 431 voxels.
constexpr int kLine32Floats = 54 * 1024 / 16;
inline int line32_lines(int n) {
  const int pitch = n | 1;
  return 32 * pitch <= kLine32Floats ? 32 : 16 * pitch <= kLine32Floats ? 16 : 8 * pitch <= kLine32Floats ? 8 : 0;
}

// The eliminated diagonal depends on the media and dt only: LINES_BUILD computes
// it into a.fac, LINES_FACTORED reads it, which leaves a multiply and a
// subtraction per row in the downward recurrence (LINES_PLAIN computes it on
// the way, a division and five more operations per row).
enum : int { LINES_PLAIN = 0, LINES_FACTORED = 1, LINES_BUILD = 2 };
constexpr int kLine32TPB = 512;

// Runs visit(k, load(k)) for k = from, from + step, ... up to and without `end`
// (step 1 or -1), loading a group of rows while the group before is visited: the
// LDS latency stays off the recurrence's chain.
template <class Load, class Visit>
__device__ inline void row_groups(int from, int end, int step, Load&& load, Visit&& visit) {
  constexpr int V = 8;
  const int count = (end - from) * step;
  int k = from, left = count;
  if (left >= V) {
    decltype(load(0)) cur[V], next[V];
#pragma unroll
    for (int v = 0; v < V; ++v) cur[v] = load(k + v * step);
    for (; left >= V; left -= V, k += V * step) {
      const int ahead = left >= 2 * V ? k + V * step : k;  // the last whole group reloads itself
#pragma unroll
      for (int v = 0; v < V; ++v) next[v] = load(ahead + v * step);
#pragma unroll
      for (int v = 0; v < V; ++v) visit(k + v * step, cur[v]);
#pragma unroll
      for (int v = 0; v < V; ++v) cur[v] = next[v];
    }
  }
  for (; left > 0; --left, k += step) visit(k, load(k));
}

template <int KIND, int TL, int MODE, bool LDS_COEF>
__global__ void __launch_bounds__(kLine32TPB) heat_sweep_lines32(HeatArgs<float> a) {
  extern __shared__ float sLine[];
  __shared__ HeatLds<float> L;
  constexpr bool X = KIND == SWEEP_X, Z = KIND == SWEEP_Z;
  constexpr bool FACTORED = MODE == LINES_FACTORED, BUILD = MODE == LINES_BUILD;
  constexpr int d = KIND;
  if (X && !BUILD) step_sensors(a);
  (void)stage_tables(a, L);
  const float* cT = LDS_COEF ? L.c : a.c;  // LDS or global, never a generic pointer
  const int nx = a.nx, ny = a.ny, nz = a.nz, nxy = nx * ny, nM = a.nM;
  const int n = X ? nx : KIND == SWEEP_Y ? ny : nz, st = X ? 1 : KIND == SWEEP_Y ? nx : nxy;
  const int pitch = n | 1;  // odd: the recurrence's lanes fall into different banks
  float* const sR = sLine;                    // right-hand side, then the solution
  float* const sB = sLine + TL * pitch;       // eliminated diagonal (not FACTORED: dt/2 c(m, before) first)
  float* const sP = sLine + 2 * TL * pitch;   // dt/2 c(m, after)
  float* const sS = sLine + 3 * TL * pitch;   // c(before, m); FACTORED: the row's multiplier
  const int blk = xcd_contiguous(blockIdx.x, gridDim.x);
  const int tiles = (nx + TL - 1) / TL;  // y and z sweeps: TL consecutive x at one z (y)
  const int o = X ? 0 : blk / tiles, c0 = X ? blk * TL : (blk - o * tiles) * TL;
  const int cols = min(TL, (X ? ny * nz : nx) - c0);
  const float dt = a.dt;
  const bool sk = a.sinked;
  float* __restrict__ fac = a.fac[KIND];
  auto line_frozen = [&](int c) {
    if (!sk) return false;
    if (X) {
      const int y = (c0 + c) % ny, z = (c0 + c) / ny;
      return y == 0 || y == ny - 1 || z == 0 || z == nz - 1;
    }
    const int x = c0 + c, nOther = KIND == SWEEP_Y ? nz : ny;
    return x == 0 || x == nx - 1 || o == 0 || o == nOther - 1;
  };
  // G threads a line, each G voxels apart (a thread stays on its line, so its
  // coordinates are worked out once); consecutive threads hold consecutive x
  constexpr int G = kLine32TPB / TL;
  const int cRaw = X ? (int)threadIdx.x / G : (int)threadIdx.x % TL, kk = X ? (int)threadIdx.x % G : (int)threadIdx.x / TL;
  const bool mine = cRaw < cols;
  const int c = mine ? cRaw : cols - 1;
  const int i0 = X ? (c0 + c) * nx : KIND == SWEEP_Y ? c0 + c + o * nxy : c0 + c + o * nx;
  const bool lf = line_frozen(c);
  const int yLine = X ? (c0 + c) % ny : 0, zLine = X ? (c0 + c) / ny : 0;
  const int oym = yLine > 0 ? -nx : 0, oyp = yLine < ny - 1 ? nx : 0, ozm = zLine > 0 ? -nxy : 0, ozp = zLine < nz - 1 ? nxy : 0;
  // all lookups and loads are done (clamped) and unwanted terms dropped by
  // selects, so that the loads of an unrolled group are in flight together
  constexpr int U = 4;
  for (int k0 = kk; k0 < n; k0 += U * G) {
    float T[U], Tl[U], Tr[U], R0[U], Ta[U], Tb[U], Tc[U], Td[U], Q[U], F[U], Fl[U];
    int M[U], Ml[U], Mr[U], Ma[U], Mb[U], Mc[U], Md[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = min(k0 + u * G, n - 1), i = i0 + k * st, il = k > 0 ? i - st : i, ir = k < n - 1 ? i + st : i;
      M[u] = a.M[i], Ml[u] = a.M[il], Mr[u] = a.M[ir];
      if (FACTORED) F[u] = fac[i], Fl[u] = fac[il];
      if (BUILD) continue;
      T[u] = a.T1[i], Tl[u] = a.T1[il], Tr[u] = a.T1[ir];
      if (X) {
        Ta[u] = a.T1[i + oym], Tb[u] = a.T1[i + oyp], Tc[u] = a.T1[i + ozm], Td[u] = a.T1[i + ozp];
        Ma[u] = a.M[i + oym], Mb[u] = a.M[i + oyp], Mc[u] = a.M[i + ozm], Md[u] = a.M[i + ozp];
        Q[u] = a.Q[i];
      } else {
        R0[u] = a.T2[i];
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + u * G;
      if (!mine || k >= n) break;
      const int m = M[u], q = c * pitch + k;
      const float cl = coef(cT, nM, m, Ml[u], d), cr = coef(cT, nM, m, Mr[u], d);
      sP[q] = dt / 2 * cr;
      if (FACTORED) {
        sB[q] = F[u];
        sS[q] = -(dt / 2 * cl) / Fl[u];
      } else {
        sB[q] = dt / 2 * cl;
        sS[q] = coef(cT, nM, Ml[u], m, d);
      }
      if (BUILD) continue;
      const bool fz = lf || (sk && (k == 0 || k == n - 1));
      if (X) {
        float dTdt = a.lightsOn ? Q[u] : 0.f;
        if (k != 0) dTdt += (Tl[u] - T[u]) * cl / 2;
        if (k != n - 1) dTdt += (Tr[u] - T[u]) * cr / 2;
        if (yLine != 0) dTdt += (Ta[u] - T[u]) * coef(cT, nM, m, Ma[u], 1);
        if (yLine != ny - 1) dTdt += (Tb[u] - T[u]) * coef(cT, nM, m, Mb[u], 1);
        if (zLine != 0) dTdt += (Tc[u] - T[u]) * coef(cT, nM, m, Mc[u], 2);
        if (zLine != nz - 1) dTdt += (Td[u] - T[u]) * coef(cT, nM, m, Md[u], 2);
        sR[q] = T[u] + dt * (fz ? 0.f : dTdt);
      } else {
        float dTdt = 0;
        if (k != 0) dTdt -= (Tl[u] - T[u]) * cl / 2;
        if (k != n - 1) dTdt -= (Tr[u] - T[u]) * cr / 2;
        sR[q] = fz ? R0[u] : R0[u] + dt * dTdt;
      }
    }
  }
  __syncthreads();
  if ((int)threadIdx.x < cols && !line_frozen(threadIdx.x)) {
    float* const r = sR + threadIdx.x * pitch;
    float* const b = sB + threadIdx.x * pitch;
    const float* const p = sP + threadIdx.x * pitch;
    const float* const q = sS + threadIdx.x * pitch;
    const int n1 = sk ? n - 1 : n;  // rows 1 .. n1-1 are eliminated; with frozen ends the last row stands
    float tprev = BUILD ? 0.f : r[0], bprev = 1;
    if (!FACTORED) {
      if (!sk && n > 1) bprev += p[0];
      b[0] = bprev;
    }
    struct Row {
      float r, b, p, q;
    };
    auto row_at = [&](int k) {
      Row w{};
      w.q = q[k];
      if (!BUILD) w.r = r[k];
      if (!FACTORED) w.b = b[k], w.p = p[k];
      return w;
    };
    auto eliminate = [&](int k, const Row& row) {
      float w = row.q;
      if (!FACTORED) {
        float bb = 1;
        if (k < n - 1) bb += row.p;
        bb += row.b;
        w = -row.b / bprev;
        if (k > 1 || !sk) bb += w * dt / 2 * row.q;
        bprev = bb;
        b[k] = bprev;
      }
      if (!BUILD) {
        tprev = row.r - w * tprev;
        r[k] = tprev;
      }
    };
    row_groups(1, n1, 1, row_at, eliminate);
  }
  // Back substitution divides by the eliminated diagonal b in every row, and a
  // correctly rounded division is the longest part of the recurrence's chain.
  // With y = 1 / b rounded to nearest, computed here by all threads, the chain
  // is q = a y and two corrections q += (a - b q) y with fused multiply-adds,
  // which round to the same bits as a / b (Markstein, "Computation of elementary
  // functions on the IBM RISC System/6000 processor", 1990) as long as nothing
  // leaves the normal range.  The rows keep the range of |a| on the way; a line
  // that left it is repeated with divisions.
  const bool divides = (int)threadIdx.x < cols && !line_frozen(threadIdx.x);
  if (!BUILD) {
    __syncthreads();
    for (int k = kk; k < n; k += G) sS[c * pitch + k] = 1.0f / sB[c * pitch + k];
    __syncthreads();
  }
  if (!BUILD && divides) {
    const float* const r = sR + threadIdx.x * pitch;
    const float* const b = sB + threadIdx.x * pitch;
    const float* const p = sP + threadIdx.x * pitch;
    float* const x = sS + threadIdx.x * pitch;  // y, then the solution
    // the last row (no term from beyond; frozen: stands), then the others that
    // are not frozen
    const int kEnd = sk ? 1 : 0;
    float lo = 1.f, hi = 1.f, bhi = 1.f;
    float xnext = sk ? r[n - 1] : (r[n - 1] + 0.f) / b[n - 1];
    x[n - 1] = xnext;
    struct Row {
      float r, b, p, y;
    };
    auto row_at = [&](int k) { return Row{r[k], b[k], p[k], x[k]}; };
    auto substitute = [&](int k, const Row& row) {
      const float t = row.r + row.p * xnext;
      float v = t * row.y;
      v = fmaf(fmaf(-row.b, v, t), row.y, v);
      v = fmaf(fmaf(-row.b, v, t), row.y, v);
      xnext = v;
      x[k] = v;
      lo = fminf(lo, t == 0.f ? 1.f : fabsf(t));
      hi = fmaxf(hi, fabsf(t));
      bhi = fmaxf(bhi, row.b);
    };
    row_groups(n - 2, kEnd - 1, -1, row_at, substitute);
    if (!(lo >= 0x1p-100f && hi <= 0x1p100f && bhi <= 0x1p20f)) {
      xnext = x[n - 1];
      for (int k = n - 2; k >= kEnd; --k) {
        xnext = (r[k] + p[k] * xnext) / b[k];
        x[k] = xnext;
      }
    }
    if (sk) x[0] = r[0];
  }
  __syncthreads();
  MaxRun run;
  for (int k0 = kk; k0 < n; k0 += U * G) {
    int m[U];
    float t0[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = i0 + min(k0 + u * G, n - 1) * st;
      if (Z && !BUILD) m[u] = a.M[i], t0[u] = a.T1[i];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + u * G, i = i0 + k * st, q = c * pitch + k;
      if (!mine || k >= n) break;
      if (BUILD) {
        fac[i] = sB[q];
        continue;
      }
      const float t = lf ? sR[q] : sS[q];
      a.T2[i] = t;
      if (Z) {
        if (a.calcDamage && L.E[m[u]] != 0)
          a.Om[i] += dt * (float)exp(L.logA[m[u]] - L.E[m[u]] / (a.Rgas * ((t + t0[u]) / 2 + a.czero)));
        run.add(m[u], (double)t, L.maxKey);
      }
    }
  }
  if (Z && !BUILD) fold_lds_max(L.maxKey, a.maxKey, nM);
}

// substeps 1a + 1b (finiteElementHeatPropagator.c:288-312, :352-389): lane per (y, z) x-line
template <typename RT, bool LDS_COEF>
__global__ void __launch_bounds__(kHeatTPB) heat_sweep_x(HeatArgs<RT> a) {
  __shared__ HeatLds<RT> L;
  step_sensors(a);
  (void)stage_tables(a, L);
  const RT* cT = LDS_COEF ? L.c : a.c;  // LDS or global, never a generic pointer
  const int line = blockIdx.x * blockDim.x + threadIdx.x;
  if (line >= a.ny * a.nz) return;
  const int y = line % a.ny, z = line / a.ny;
  const bool lf = a.sinked && (y == 0 || y == a.ny - 1 || z == 0 || z == a.nz - 1);
  sweep_line<RT, SWEEP_X, kSweepU>(a, cT, L, y * a.nx + z * a.nx * a.ny, 1, a.nx, lf, 0, a.nx, y, a.ny, a.nx * a.ny, z, a.nz, nullptr,
                                   nullptr);
}

// substeps 2a + 2b (:429-448, :486-521): lane per (x, z) y-line, lanes along x
template <typename RT, bool LDS_COEF>
__global__ void __launch_bounds__(kHeatTPB) heat_sweep_y(HeatArgs<RT> a) {
  __shared__ HeatLds<RT> L;
  (void)stage_tables(a, L);
  const RT* cT = LDS_COEF ? L.c : a.c;  // LDS or global, never a generic pointer
  const int line = blockIdx.x * blockDim.x + threadIdx.x;
  if (line >= a.nx * a.nz) return;
  const int x = line % a.nx, z = line / a.nx;
  const bool lf = a.sinked && (x == 0 || x == a.nx - 1 || z == 0 || z == a.nz - 1);
  sweep_line<RT, SWEEP_Y, kSweepU>(a, cT, L, x + z * a.nx * a.ny, a.nx, a.ny, lf, 1, 0, 0, 1, 0, 0, 1, nullptr, nullptr);
}

// substeps 3a + 3b (:546-565, :606-646) with the Arrhenius update and the
// per-medium maximum: lane per (x, y) z-line, lanes along x
template <typename RT, bool LDS_COEF>
__global__ void __launch_bounds__(kHeatTPB) heat_sweep_z(HeatArgs<RT> a) {
  __shared__ HeatLds<RT> L;
  (void)stage_tables(a, L);
  const RT* cT = LDS_COEF ? L.c : a.c;  // LDS or global, never a generic pointer
  const int line = blockIdx.x * blockDim.x + threadIdx.x;
  if (line < a.nx * a.ny) {
    const int x = line % a.nx, y = line / a.nx;
    const bool lf = a.sinked && (x == 0 || x == a.nx - 1 || y == 0 || y == a.ny - 1);
    MaxRun run;
    sweep_line<RT, SWEEP_Z, kSweepU>(a, cT, L, line, a.nx * a.ny, a.nz, lf, 2, 0, 0, 1, 0, 0, 1, &run, L.maxKey);
  }
  fold_lds_max(L.maxKey, a.maxKey, a.nM);
}

// ---------------------------------------------------------------------------
// Wavefront-parallel tridiagonal solve (FP64 sweeps)
//
// A system  a[r] x[r-1] + b[r] x[r] + c[r] x[r+1] = d[r]  of up to W*S rows
// is spread over a segment of W lanes (W = 64 or 32; a wavefront solves
// 64 / W systems side by side), S consecutive rows per lane (row
// r = lane * S + s, lane counted within the segment); unused rows are
// a = c = 0, b = 1, d = 0.  The matrices of the heat step are strictly
// diagonally dominant, so no pivoting is needed.  With U the lanes' last
// unknowns and UL the one of the lane before:
//   1. each lane eliminates downwards and keeps three numbers per row,
//      x[s] = p[s] - q[s] UL - g[s] x[s+1];
//   2. its first unknown in terms of UL and U goes to the lane before, which
//      leaves one tridiagonal equation per lane in U with a unit diagonal;
//   3. that W-row system is solved by parallel cyclic reduction, at most
//      log2(W) steps of lane moves that never cross a segment's edge.  The
//      couplings are products of S off-diagonal/diagonal ratios and square at
//      every step, so they fall fast: once all of a wavefront's are at most
//      2^-30, one correction with the neighbours' right-hand sides leaves a
//      relative error of 2^-60 and the steps end (time steps of up to 1.5
//      times the explicit limit have ratios of about 0.1: no step at S = 13,
//      one at S = 8, two at S = 4; larger time steps take more);
//   4. each lane recovers its unknowns upwards from U and UL.
// Same solution as the sequential Thomas recurrence up to rounding.
__device__ inline double lane_shfl(double v, int src) { return __shfl(v, src < 0 ? 0 : (src > 63 ? 63 : src), 64); }
__device__ inline int lane_shfl(int v, int src) { return __shfl(v, src < 0 ? 0 : (src > 63 ? 63 : src), 64); }

// v of lane wl + h (UP) or wl - h of the same W-lane segment; a lane whose
// source lies outside its segment gets an unspecified value, which callers
// mask.
template <int W, bool UP, typename V>
__device__ inline V seg_shift(V v, int h) {
  const int wl = __lane_id();
  return lane_shfl(v, UP ? wl + h : wl - h);
}

// 1 / b for the well-scaled pivots of the solver: hardware reciprocal estimate
// refined by two Newton steps (a few ulp), instead of the correctly rounded
// division sequence.
__device__ inline double prcp(double b) {
  double r = __builtin_amdgcn_rcp(b);
  r = fma(fma(-b, r, 1.0), r, r);
  r = fma(fma(-b, r, 1.0), r, r);
  return r;
}

// couplings below this are dropped after one correction step (line_solve)
constexpr double kDecoupled = 0x1p-30;

template <int S, int W = 64>
__device__ inline void line_solve(const double (&a)[S], const double (&b)[S], const double (&c)[S], const double (&d)[S], double (&x)[S]) {
  // a line per W-lane segment of the wavefront; lane is the index within it
  static_assert(W == 32 || W == 64, "segments of 32 or 64 lanes");
  const int lane = __lane_id() & (W - 1);
  // 1: x[s] = p[s] - q[s] UL - g[s] x[s+1]
  double g[S], p[S], q[S];
  {
    const double r = prcp(b[0]);
    g[0] = c[0] * r;
    p[0] = d[0] * r;
    q[0] = a[0] * r;
  }
#pragma unroll
  for (int s = 1; s < S; ++s) {
    const double r = prcp(fma(-a[s], g[s - 1], b[s]));
    g[s] = c[s] * r;
    p[s] = fma(-a[s], p[s - 1], d[s]) * r;
    q[s] = -a[s] * q[s - 1] * r;
  }
  // 2: x[0] = P - Q UL + R U
  double P = 0.0, Q = 0.0, R = 1.0;
#pragma unroll
  for (int s = S - 2; s >= 0; --s) {
    P = fma(-g[s], P, p[s]);
    Q = fma(-g[s], Q, q[s]);
    R = -g[s] * R;
  }
  // shuffles run in every lane (a lane reading from a lane that is inactive
  // at the shuffle gets 0), then lanes without the neighbour are masked
  double Pn = seg_shift<W, true>(P, 1), Qn = seg_shift<W, true>(Q, 1), Rn = seg_shift<W, true>(R, 1);
  if (lane == W - 1) Pn = Qn = Rn = 0.0;
  const double e = g[S - 1], ib = prcp(fma(-e, Qn, 1.0));
  double pa = q[S - 1] * ib, pc = e * Rn * ib, pd = fma(-e, Pn, p[S - 1]) * ib;
  // 3: U + pa U(lane - h) + pc U(lane + h) = pd
  double U = pd;
#pragma unroll
  for (int h = 1; h < W; h <<= 1) {
    double dm = seg_shift<W, false>(pd, h), dp = seg_shift<W, true>(pd, h);
    dm = lane >= h ? dm : 0.0;
    dp = lane + h < W ? dp : 0.0;
    if (__all(fmax(fabs(pa), fabs(pc)) <= kDecoupled)) {
      pd = fma(-pc, dp, fma(-pa, dm, pd));
      break;
    }
    double am = seg_shift<W, false>(pa, h), cm = seg_shift<W, false>(pc, h);
    double ap = seg_shift<W, true>(pa, h), cp = seg_shift<W, true>(pc, h);
    am = lane >= h ? am : 0.0;
    cm = lane >= h ? cm : 0.0;
    ap = lane + h < W ? ap : 0.0;
    cp = lane + h < W ? cp : 0.0;
    const double r = prcp(fma(-pc, ap, fma(-pa, cm, 1.0)));
    pd = fma(-pc, dp, fma(-pa, dm, pd)) * r;
    pa = -pa * am * r;
    pc = -pc * cp * r;
  }
  U = pd;
  // 4
  double UL = seg_shift<W, false>(U, 1);
  if (lane == 0) UL = 0.0;
  x[S - 1] = U;
#pragma unroll
  for (int s = S - 2; s >= 0; --s) x[s] = fma(-g[s], x[s + 1], fma(-q[s], UL, p[s]));
}

// The FP64 sweeps work on increments: with u the temperature at the start of
// the step, A_d = I - dt/2 L_d and L = L_x + L_y + L_z,
//   A_x dx = dt (L u + Q),  A_y dy = dx,  A_z dz = dy,  T = u + dz
// is the Douglas-Gunn step written for T1 - u, T2 - u and T3 - u instead of
// the substeps' temperatures T1, T2, T3 (A_y (T2 - u) = T1 - dt/2 L_y u - A_y u
// = T1 - u, and likewise along z).  The y and z sweeps then need neither u's
// stencil nor u itself before the end, and rounding enters relative to the
// increment.  Frozen voxels have increment 0.

// substeps 1a + 1b in FP64, a (y, z) x-line per W lanes: lane l holds voxels
// x = l*S .. l*S+S-1, so every load of the wavefront is contiguous.  Bound by
// instruction issue (52 us at 200^3; 75 us with all six reduction steps and
// workgroups dealt to the XCDs in turn).
template <int S, int W, bool LDS_COEF>
__global__ void __launch_bounds__(kHeatTPB) heat_sweep_x_wave(HeatArgs<double> a) {
  // the coefficient table in LDS when it fits (LDS_COEF), else read from
  // global memory; one or the other, so every lookup is a plain LDS or
  // global load rather than a generic one
  __shared__ double sc[LDS_COEF ? kLdsCoef : 1];
  step_sensors(a);
  if (LDS_COEF) {
    const int nc = a.nM * a.nM * 3;
    for (int k = threadIdx.x; k < nc; k += blockDim.x) sc[k] = a.c[k];
    __syncthreads();
  }
  const double* __restrict__ cT = LDS_COEF ? sc : a.c;
  // a line per W-lane segment; a segment past the last line solves the
  // last line again and stores nothing
  const int wl = __lane_id(), lane = wl & (W - 1);
  const int line = (xcd_contiguous(blockIdx.x, gridDim.x) * (kHeatTPB / 64) + (threadIdx.x >> 6)) * (64 / W) + wl / W;
  const int nx = a.nx, ny = a.ny, nz = a.nz, nxy = nx * ny, nM = a.nM;
  const bool valid = line < ny * nz;
  const int y = (valid ? line : ny * nz - 1) % ny, z = (valid ? line : ny * nz - 1) / ny;
  const int i0 = y * nx + z * nxy;
  const bool sk = a.sinked;
  const bool lf = sk && (y == 0 || y == ny - 1 || z == 0 || z == nz - 1);
  const double* __restrict__ T1 = a.T1;
  const uint8_t* __restrict__ Mg = a.M;
  const float* __restrict__ Q = a.Q;
  const double dt = a.dt;
  double T[S];
  int Mv[S];
  // neighbouring lines and the source, loaded up front (clamped addresses)
  double Tym[S], Typ[S], Tzm[S], Tzp[S];
  int Mym[S], Myp[S], Mzm[S], Mzp[S];
  float Qv[S];
  const int oym = y != 0 ? -nx : 0, oyp = y != ny - 1 ? nx : 0, ozm = z != 0 ? -nxy : 0, ozp = z != nz - 1 ? nxy : 0;
  const bool vec = S % 4 == 0 && (nx & 3) == 0 && lane * S + S <= nx;
  if (vec) {
    // a lane's S voxels of each line are consecutive and 32-byte aligned:
    // 16-byte loads for T and Q, 4-byte loads for M
    const int b = i0 + lane * S;
#pragma unroll
    for (int s = 0; s < S; s += 2) {
      const double2 t = *(const double2*)(T1 + b + s), tym = *(const double2*)(T1 + b + oym + s), typ = *(const double2*)(T1 + b + oyp + s);
      const double2 tzm = *(const double2*)(T1 + b + ozm + s), tzp = *(const double2*)(T1 + b + ozp + s);
      T[s] = t.x, T[s + 1] = t.y;
      Tym[s] = tym.x, Tym[s + 1] = tym.y;
      Typ[s] = typ.x, Typ[s + 1] = typ.y;
      Tzm[s] = tzm.x, Tzm[s + 1] = tzm.y;
      Tzp[s] = tzp.x, Tzp[s + 1] = tzp.y;
    }
#pragma unroll
    for (int s = 0; s < S; s += 4) {
      const float4 q = *(const float4*)(Q + b + s);
      Qv[s] = q.x, Qv[s + 1] = q.y, Qv[s + 2] = q.z, Qv[s + 3] = q.w;
      const uint32_t m = *(const uint32_t*)(Mg + b + s), mym = *(const uint32_t*)(Mg + b + oym + s);
      const uint32_t myp = *(const uint32_t*)(Mg + b + oyp + s), mzm = *(const uint32_t*)(Mg + b + ozm + s);
      const uint32_t mzp = *(const uint32_t*)(Mg + b + ozp + s);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        Mv[s + u] = (int)((m >> (8 * u)) & 0xffu);
        Mym[s + u] = (int)((mym >> (8 * u)) & 0xffu);
        Myp[s + u] = (int)((myp >> (8 * u)) & 0xffu);
        Mzm[s + u] = (int)((mzm >> (8 * u)) & 0xffu);
        Mzp[s + u] = (int)((mzp >> (8 * u)) & 0xffu);
      }
    }
  } else {
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const int k = lane * S + s;
      const int i = i0 + (k < nx ? k : 0);
      T[s] = k < nx ? T1[i] : 0.0;
      Mv[s] = k < nx ? (int)Mg[i] : 0;
      Tym[s] = T1[i + oym];
      Typ[s] = T1[i + oyp];
      Tzm[s] = T1[i + ozm];
      Tzp[s] = T1[i + ozp];
      Mym[s] = Mg[i + oym];
      Myp[s] = Mg[i + oyp];
      Mzm[s] = Mg[i + ozm];
      Mzp[s] = Mg[i + ozp];
      Qv[s] = Q[i];
    }
  }
  const double Tl = seg_shift<W, false>(T[S - 1], 1), Tr = seg_shift<W, true>(T[0], 1);
  const int Ml = seg_shift<W, false>(Mv[S - 1], 1), Mr = seg_shift<W, true>(Mv[0], 1);
  double ca[S], cb[S], cc_[S], cd[S], xs[S];
  const double h = dt / 2;
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const int k = lane * S + s;
    const int m = Mv[s];
    const double TL = s > 0 ? T[s - 1] : Tl, TR = s < S - 1 ? T[s + 1] : Tr;
    const int ML = s > 0 ? Mv[s - 1] : Ml, MR = s < S - 1 ? Mv[s + 1] : Mr;
    // Every lookup is done and unwanted ones dropped by selects (no branch).
    // Neighbours outside the grid: along y and z the clamped addresses above
    // read the voxel itself, whose difference is 0; along x the coefficient
    // is made 0 (and the difference finite).
    const bool on = k < nx && !lf && !(sk && (k == 0 || k == nx - 1));
    const bool hasL = on && k > 0, hasR = on && k < nx - 1;
    const double cL = coef(cT, nM, m, ML, 0), cR = coef(cT, nM, m, MR, 0);
    const double cl = hasL ? cL : 0.0, cr = hasR ? cR : 0.0;
    double dTdt = a.lightsOn ? (double)Qv[s] : 0.0;
    dTdt = fma(hasL ? TL - T[s] : 0.0, cl, dTdt);
    dTdt = fma(hasR ? TR - T[s] : 0.0, cr, dTdt);
    dTdt = fma(Tym[s] - T[s], coef(cT, nM, m, Mym[s], 1), dTdt);
    dTdt = fma(Typ[s] - T[s], coef(cT, nM, m, Myp[s], 1), dTdt);
    dTdt = fma(Tzm[s] - T[s], coef(cT, nM, m, Mzm[s], 2), dTdt);
    dTdt = fma(Tzp[s] - T[s], coef(cT, nM, m, Mzp[s], 2), dTdt);
    cd[s] = on ? dt * dTdt : 0.0;
    ca[s] = -h * cl;
    cc_[s] = -h * cr;
    cb[s] = fma(h, cl + cr, 1.0);
  }
  line_solve<S, W>(ca, cb, cc_, cd, xs);
  double* __restrict__ T2 = a.T2;
  if (!valid) return;
  if (vec) {
#pragma unroll
    for (int s = 0; s < S; s += 2) *(double2*)(T2 + i0 + lane * S + s) = make_double2(xs[s], xs[s + 1]);
  } else {
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const int k = lane * S + s;
      if (k < nx) T2[i0 + k] = xs[s];
    }
  }
}

// The same solve for lines along y or z by a whole workgroup: 16 neighbouring
// lines (one cache line of doubles per row of voxels), NC chunks of S voxels
// each, thread t holding chunk t / 16 of line t % 16 in registers.  Steps 2-4
// exchange between chunks through LDS, two barriers when the couplings fall
// below kDecoupled at once (S large enough) and one more per reduction step.
// Bound by memory: at 200^3 the y sweep moves 136 MB in 24.9 us (5.5 TB/s; a
// 64 MiB copy reaches 8.1).  Lines staged through LDS tiles, with u's stencil
// in the y and z sweeps, took 60.9 (y) and 96.4 us (z); four lines per
// wavefront without LDS 40.2 and 83.0 us (32-byte pieces of cache lines).
template <int NC>
struct LineLds {
  double v[2][3][NC * 16];  // two buffers used in turn
  int coupled[8];           // per reduction step: some coupling is above kDecoupled
};

template <int S, int NC>
__device__ inline void block_line_solve(const double (&a)[S], const double (&b)[S], const double (&c)[S], const double (&d)[S], double (&x)[S],
                                        LineLds<NC>& L) {
  const int t = threadIdx.x, ch = t >> 4;
  double g[S], p[S], q[S];
  {
    const double r = prcp(b[0]);
    g[0] = c[0] * r;
    p[0] = d[0] * r;
    q[0] = a[0] * r;
  }
#pragma unroll
  for (int s = 1; s < S; ++s) {
    const double r = prcp(fma(-a[s], g[s - 1], b[s]));
    g[s] = c[s] * r;
    p[s] = fma(-a[s], p[s - 1], d[s]) * r;
    q[s] = -a[s] * q[s - 1] * r;
  }
  double P = 0.0, Q = 0.0, R = 1.0;
#pragma unroll
  for (int s = S - 2; s >= 0; --s) {
    P = fma(-g[s], P, p[s]);
    Q = fma(-g[s], Q, q[s]);
    R = -g[s] * R;
  }
  L.v[0][0][t] = P;
  L.v[0][1][t] = Q;
  L.v[0][2][t] = R;
  if (t < 8) L.coupled[t] = 0;
  __syncthreads();
  // entry of chunk ch + h (0 outside the line)
  auto at = [&](int buf, int k, int h) {
    const bool in = ch + h >= 0 && ch + h < NC;
    const double v = L.v[buf][k][in ? t + 16 * h : t];
    return in ? v : 0.0;
  };
  const double Pn = at(0, 0, 1), Qn = at(0, 1, 1), Rn = at(0, 2, 1);
  const double e = g[S - 1], ib = prcp(fma(-e, Qn, 1.0));
  double pa = q[S - 1] * ib, pc = e * Rn * ib, pd = fma(-e, Pn, p[S - 1]) * ib;
  double U = 0.0, UL = 0.0;
  int buf = 1;
  for (int h = 1, step = 0;; h <<= 1, ++step) {
    L.v[buf][0][t] = pd;
    L.v[buf][1][t] = pa;
    L.v[buf][2][t] = pc;
    if (!(fmax(fabs(pa), fabs(pc)) <= kDecoupled)) L.coupled[step] = 1;
    __syncthreads();
    const double dm = at(buf, 0, -h), dp = at(buf, 0, h);
    if (h >= NC || !L.coupled[step]) {
      U = fma(-pc, dp, fma(-pa, dm, pd));
      UL = fma(-at(buf, 2, -1), at(buf, 0, h - 1), fma(-at(buf, 1, -1), at(buf, 0, -h - 1), at(buf, 0, -1)));
      break;
    }
    const double am = at(buf, 1, -h), cm = at(buf, 2, -h), ap = at(buf, 1, h), cp = at(buf, 2, h);
    const double r = prcp(fma(-pc, ap, fma(-pa, cm, 1.0)));
    pd = fma(-pc, dp, fma(-pa, dm, pd)) * r;
    pa = -pa * am * r;
    pc = -pc * cp * r;
    buf ^= 1;
  }
  x[S - 1] = U;
#pragma unroll
  for (int s = S - 2; s >= 0; --s) x[s] = fma(-g[s], x[s + 1], fma(-q[s], UL, p[s]));
}

// per-axis coefficient tables of up to this many entries go to LDS in the y/z
// kernels (22 media, like kLdsCoef)
constexpr int kAxisCoef = 512;

// What a thread of a y/z kernel works on: chunk `ch` (voxels k0 .. k0+S-1) of
// the line at x and the other coordinate o.
struct LinePos {
  int x, o, k0, base;
  bool valid;  // false: a copy of the last line, which stores nothing
};
template <int S, int NC, int AXIS>
__device__ inline LinePos line_pos(int nx, int ny) {
  LinePos L;
  const int ntx = (nx + 15) >> 4, blk = xcd_contiguous(blockIdx.x, gridDim.x);
  L.o = blk / ntx;
  const int xw = ((blk - L.o * ntx) << 4) + (threadIdx.x & 15);
  L.valid = xw < nx;
  L.x = L.valid ? xw : nx - 1;
  L.k0 = (threadIdx.x >> 4) * S;
  L.base = L.x + L.o * (AXIS == 1 ? nx * ny : nx);
  return L;
}

// Arrhenius updates collected per wavefront: the voxels whose medium can be
// damaged are few and scattered over lanes, so a wavefront appends them to a
// queue and evaluates 64 at a time with all its lanes.
constexpr int kBurnQueue = 128;
struct BurnQueue {
  double th[kBurnQueue];  // mean temperature of the step [K]
  int i[kBurnQueue], m[kBurnQueue];
};
__device__ inline void burn(const HeatArgs<double>& a, const BurnQueue& B, int e, const double* sLogA, const double* sE) {
  const int m = B.m[e], i = B.i[e];
  const double rt = a.Rgas * B.th[e];
  double r = prcp(rt);
  if (!__builtin_isfinite(r)) r = __builtin_amdgcn_rcp(rt);  // 0 and infinities, where the refinement has no value
  a.Om[i] += a.dt * exp(fma(-sE[m], r, sLogA[m]));
}

// substeps 2a + 2b (KIND Y) and 3a + 3b with the Arrhenius update and the
// per-medium maxima (KIND Z) in FP64.  50 us for z at 200^3, half of it the
// damage and maxima; exponentials evaluated where their voxels lie (13 rounds
// with 3 of 16 lanes) cost 30 us more.
template <int S, int NC, int KIND, bool LDS_COEF>
__global__ void __launch_bounds__(NC * 16) heat_sweep_yz(HeatArgs<double> a) {
  constexpr bool Z = KIND == SWEEP_Z;
  constexpr int d = Z ? 2 : 1;
  __shared__ LineLds<NC> lds;
  __shared__ double sC[LDS_COEF ? kAxisCoef : 1];
  __shared__ double sLogA[Z ? 256 : 1], sE[Z ? 256 : 1];
  __shared__ unsigned long long sMax[Z ? 256 : 1];
  __shared__ BurnQueue sBurn[Z ? NC / 4 : 1];
  const int nx = a.nx, ny = a.ny, nz = a.nz, nM = a.nM;
  const int n = Z ? nz : ny, nOther = Z ? ny : nz, st = Z ? nx * ny : nx;
  const LinePos L = line_pos<S, NC, d>(nx, ny);
  double* __restrict__ T2 = a.T2;
  const double* __restrict__ T1 = a.T1;
  const uint8_t* __restrict__ Mg = a.M;
  double cd[S], T[Z ? S : 1];
  int Mv[S];
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const int i = L.base + min(L.k0 + s, n - 1) * st;
    cd[s] = T2[i];
    Mv[s] = Mg[i];
    if (Z) T[s] = T1[i];
  }
  const int Ml = Mg[L.base + min(max(L.k0 - 1, 0), n - 1) * st], Mr = Mg[L.base + min(L.k0 + S, n - 1) * st];
  if (LDS_COEF)
    for (int k = threadIdx.x; k < nM * nM; k += blockDim.x) sC[k] = a.c[k + d * nM * nM];
  if (Z)
    for (int k = threadIdx.x; k < nM; k += blockDim.x) {
      sLogA[k] = a.logA[k];
      sE[k] = a.E[k];
      sMax[k] = a.maxKey[k];
    }
  __syncthreads();
  const double* __restrict__ cT = LDS_COEF ? sC : a.c + d * nM * nM;  // LDS or global, never a generic pointer
  const bool sk = a.sinked, lf = sk && (L.x == 0 || L.x == nx - 1 || L.o == 0 || L.o == nOther - 1);
  const double h = a.dt / 2;
  double ca[S], cb[S], cc_[S], xs[S];
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const int k = L.k0 + s;
    const double cl = coef(cT, nM, Mv[s], s > 0 ? Mv[s - 1] : Ml, 0), cr = coef(cT, nM, Mv[s], s < S - 1 ? Mv[s + 1] : Mr, 0);
    const bool on = k < n && !lf && !(sk && (k == 0 || k == n - 1));
    ca[s] = on && k > 0 ? -h * cl : 0.0;
    cc_[s] = on && k < n - 1 ? -h * cr : 0.0;
    cb[s] = 1.0 - (ca[s] + cc_[s]);
    cd[s] = k < n ? cd[s] : 0.0;
  }
  block_line_solve<S, NC>(ca, cb, cc_, cd, xs, lds);
  if (!Z) {
#pragma unroll
    for (int s = 0; s < S; ++s)
      if (L.valid && L.k0 + s < n) T2[L.base + (L.k0 + s) * st] = xs[s];
    return;
  }
  MaxRun run;
  BurnQueue& B = sBurn[threadIdx.x >> 6];
  const int lane = __lane_id();
  int queued = 0;  // wavefront-uniform
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const int k = L.k0 + s, i = L.base + k * st, m = Mv[s];
    const bool live = L.valid && k < n;
    const double t = T[s] + xs[s];
    if (live) {
      T2[i] = t;
      run.add(m, t, sMax);
    }
    const bool burns = live && a.calcDamage && sE[m] != 0;
    const unsigned long long bal = __ballot(burns);
    if (bal) {
      if (burns) {
        const int e = queued + __popcll(bal & ((1ull << lane) - 1ull));
        B.th[e] = (t + T[s]) / 2 + a.czero;
        B.i[e] = i;
        B.m[e] = m;
      }
      queued += __popcll(bal);
      if (queued >= 64) {
        queued -= 64;
        wave_lds_fence();
        burn(a, B, queued + lane, sLogA, sE);
        wave_lds_fence();
      }
    }
  }
  wave_lds_fence();
  if (lane < queued) burn(a, B, lane, sLogA, sE);
  fold_lds_max(sMax, a.maxKey, nM);
}

// whether the wavefront solvers take a line of n voxels (else the sequential
// lane-per-line kernels)
inline bool wave_line(int n) { return n <= 512; }

// Calls f(integral_constant S, integral_constant W) with the rows per lane and
// lanes per line of the x sweeps.
template <class F>
inline void with_x_shape(int n, F&& f) {
  using std::integral_constant;
  if (n <= 64) return f(integral_constant<int, 2>(), integral_constant<int, 32>());
  if (n <= 128) return f(integral_constant<int, 4>(), integral_constant<int, 32>());
  if (n <= 256) return f(integral_constant<int, 4>(), integral_constant<int, 64>());
  return f(integral_constant<int, 8>(), integral_constant<int, 64>());
}

// The same with the rows per thread and chunks per line of the y and z
// sweeps: the fewest rows of the compiled ones that hold the line in 16
// chunks (32 chunks beyond 256 voxels).
template <class F>
inline void with_yz_shape(int n, F&& f) {
  using std::integral_constant;
  using C16 = integral_constant<int, 16>;
  using C32 = integral_constant<int, 32>;
  if (n <= 32) return f(integral_constant<int, 2>(), C16());
  if (n <= 64) return f(integral_constant<int, 4>(), C16());
  if (n <= 96) return f(integral_constant<int, 6>(), C16());
  if (n <= 128) return f(integral_constant<int, 8>(), C16());
  if (n <= 160) return f(integral_constant<int, 10>(), C16());
  if (n <= 208) return f(integral_constant<int, 13>(), C16());
  if (n <= 256) return f(integral_constant<int, 16>(), C16());
  if (n <= 416) return f(integral_constant<int, 13>(), C32());
  return f(integral_constant<int, 16>(), C32());
}

// v of the lane before (after) in the wavefront; lane 0 (63) gets 0
template <typename V>
__device__ inline V lane_before(V v) {
  return __shfl_up(v, 1, 64);
}
template <typename V>
__device__ inline V lane_after(V v) {
  return __shfl_down(v, 1, 64);
}

// Forward Euler step (no reference counterpart; the 7-point right-hand side
// of substep 1a with all three axes fully weighted, the damage update and
// the per-medium maxima of the DG-ADI step).  A thread owns a column and
// marches up a run of zRun z planes (chosen per plan by timing, see
// tune_explicit); the threads of a workgroup own consecutive voxels of the
// plane, whatever the row length.  The z neighbours are carried in registers,
// the x neighbours come from the neighbouring lanes (the wavefront's first and
// last lane load theirs), the y neighbours are loaded, and all loads of a plane
// are issued one plane ahead of their use (the voxel above two ahead).
//
// 225x190x171, lights on and off: 39 us a step (3.4 to 4 TB/s of compulsory
// bytes), bound by instruction issue together with the memory's latency;
// staging each plane through LDS behind two barriers took 53 us (45 of them
// once maxima no longer went through global atomics).  Two planes ahead, or
// register roles rotated instead of copied, need 4 wavefronts' registers
// instead of 5 and were slower on large grids.  Addresses are a plane's base in
// scalar registers plus a 32-bit byte offset in the plane (OFF = uint32_t;
// planes of 2^28 voxels or more use 64-bit offsets); a coefficient's address is
// one multiply-add.
template <typename RT, bool LDS_COEF, typename OFF>
__global__ void __launch_bounds__(kHeatTPB) heat_explicit_march(HeatArgs<RT> a, int zRun) {
  __shared__ HeatLds<RT> L;
  step_sensors(a);
  const int nx = a.nx, ny = a.ny, nz = a.nz, nxy = nx * ny, nM = a.nM;
  const int npb = (nxy + kHeatTPB - 1) / kHeatTPB, blk = xcd_contiguous(blockIdx.x, gridDim.x);
  const int zi = blk / npb;
  const int p0 = (blk - zi * npb) * kHeatTPB + threadIdx.x, z0 = zi * zRun, zEnd = min(z0 + zRun, nz);
  const bool ok = p0 < nxy;
  const int p = ok ? p0 : nxy - 1, x = p % nx, y = p / nx;
  const bool sideFrozen = a.sinked && (x == 0 || x == nx - 1 || y == 0 || y == ny - 1);
  const bool first = __lane_id() == 0, last = __lane_id() == 63;
  // Neighbours outside the grid are the voxel itself (difference 0).
  const bool noL = x == 0, noR = x == nx - 1;
  const OFF oP = (OFF)p, oYm = (OFF)(y > 0 ? p - nx : p), oYp = (OFF)(y < ny - 1 ? p + nx : p);
  const OFF oE = (OFF)(first ? max(p - 1, 0) : min(p + 1, nxy - 1));
  auto ldT = [&](int z, OFF o) { return *(const RT*)((const char*)(a.T1 + (int64_t)z * nxy) + (OFF)(o * (OFF)sizeof(RT))); };
  auto ldM = [&](int z, OFF o) { return (unsigned)*(const uint8_t*)((const char*)(a.M + (int64_t)z * nxy) + o); };
  struct Side {  // a plane's neighbours within the plane and its source
    RT ym, yp, e;
    unsigned mym, myp, me;
    float q;
  };
  auto load_side = [&](int z) {
    Side s;
    z = min(z, nz - 1);
    s.ym = ldT(z, oYm);
    s.yp = ldT(z, oYp);
    s.mym = ldM(z, oYm);
    s.myp = ldM(z, oYp);
    s.e = 0;
    s.me = 0;
    if (first || last) {
      s.e = ldT(z, oE);
      s.me = ldM(z, oE);
    }
    s.q = a.lightsOn ? *(const float*)((const char*)(a.Q + (int64_t)z * nxy) + (OFF)(oP * (OFF)4)) : 0.f;
    return s;
  };
  auto clampz = [&](int z) { return min(max(z, 0), nz - 1); };
  RT tBelow = ldT(clampz(z0 - 1), oP), tHere = ldT(z0, oP), tAbove = ldT(clampz(z0 + 1), oP);
  unsigned mBelow = ldM(clampz(z0 - 1), oP), mHere = ldM(z0, oP), mAbove = ldM(clampz(z0 + 1), oP);
  Side here = load_side(z0);
  (void)stage_tables(a, L);
  const char* cT = (const char*)(LDS_COEF ? L.c : a.c);  // LDS or global, never a generic pointer
  const unsigned pitch = (unsigned)(nM * sizeof(RT)), axis = pitch * (unsigned)nM;
  const RT dt = a.dt;
  MaxRun run;
  for (int z = z0; z < zEnd; ++z) {
    const Side next = load_side(z + 1);
    const RT tNext = ldT(min(z + 2, nz - 1), oP);
    const unsigned mNext = ldM(min(z + 2, nz - 1), oP);
    RT tl = lane_before(tHere), tr = lane_after(tHere);
    unsigned ml = lane_before(mHere), mr = lane_after(mHere);
    if (first) tl = here.e, ml = here.me;
    if (last) tr = here.e, mr = here.me;
    if (noL) tl = tHere;
    if (noR) tr = tHere;
    const unsigned row0 = mHere * (unsigned)sizeof(RT), row1 = row0 + axis, row2 = row1 + axis;
    auto cf = [&](unsigned row, unsigned m) { return *(const RT*)(cT + (__umul24(m, pitch) + row)); };
    const RT cl = cf(row0, ml), cr = cf(row0, mr), cym = cf(row1, here.mym), cyp = cf(row1, here.myp), czm = cf(row2, mBelow), czp = cf(row2, mAbove);
    RT dTdt = (RT)here.q;
    dTdt += (tl - tHere) * cl;
    dTdt += (tr - tHere) * cr;
    dTdt += (here.ym - tHere) * cym;
    dTdt += (here.yp - tHere) * cyp;
    dTdt += (tBelow - tHere) * czm;
    dTdt += (tAbove - tHere) * czp;
    if (sideFrozen || (a.sinked && (z == 0 || z == nz - 1))) dTdt = 0;
    const RT t = tHere + dt * dTdt;
    if (ok) {
      *(RT*)((char*)(a.T2 + (int64_t)z * nxy) + (OFF)(oP * (OFF)sizeof(RT))) = t;
      if (a.calcDamage && L.E[mHere] != 0)
        a.Om[(int64_t)z * nxy + p] += dt * (RT)exp(L.logA[mHere] - L.E[mHere] / (a.Rgas * ((t + tHere) / 2 + a.czero)));
      run.add((int)mHere, (double)t, L.maxKey);
    }
    tBelow = tHere;
    mBelow = mHere;
    tHere = tAbove;
    mHere = mAbove;
    tAbove = tNext;
    mAbove = mNext;
    here = next;
  }
  fold_lds_max(L.maxKey, a.maxKey, a.nM);
}

// Sensor record of T into column `col` on its own (the final state of a
// run, recorded when the record is read).
template <typename RT>
__global__ void heat_sensors(const RT* T, int nx, int nxy, const long long* idx, const RT* w, int nS, double* out, long long col) {
  sensors_at(T, nx, nxy, idx, w, nS, out, col, (int)threadIdx.x, (int)blockDim.x);
}

// step counter of graph-replayed steps: set before a series of replays,
// advanced by the last node of each replay
__global__ void heat_step_counter(long long* c, long long value, int add) {
  if (threadIdx.x == 0) *c = add ? *c + value : value;
}

template <typename RT>
__global__ void heat_load(RT* dst, const float* src32, const double* src64, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = src64 ? (RT)src64[i] : (RT)src32[i];
}

template <typename RT>
__global__ void heat_store(const RT* src, float* dst32, double* dst64, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    if (dst32) dst32[i] = (float)src[i];
    if (dst64) dst64[i] = (double)src[i];
  }
}

__global__ void heat_init_keys(unsigned long long* k, int n) {
  const int i = threadIdx.x + blockIdx.x * blockDim.x;
  if (i < n) k[i] = order_key(-INFINITY);
}


// ---------------------------------------------------------------------------
// Discrete adjoint of the FP64 DG-ADI step (no reference counterpart).
//
// With D the non-frozen voxels and L_d the conduction operators
// ((L_d u)_i = sum over the d-neighbours n of c[M_i, M_n, d] (u_n - u_i)),
// one step is
//   T*   = u + dt D (L_x/2 + L_y + L_z) u + dt lightsOn D Q
//   T1   = A_x^-1 T*,  T2 = A_y^-1 (T1 - dt/2 D L_y u),  T3 = A_z^-1 (T2 - dt/2 D L_z u)
// with A_d = I - dt/2 D L_d.  For an adjoint lam of T3 the adjoints are
//   mu3 = A_z^-T lam,  mu2 = A_y^-T mu3,  mu1 = A_x^-T mu2
//   lam_u = mu1 + dt (L_x/2 + L_y + L_z)^T D mu1 - dt/2 L_y^T D mu2 - dt/2 L_z^T D mu3
//   lam_Q = dt lightsOn D mu1
// and the damage of the step, dt A exp(-E / (R ((T3 + u)/2 + 273.15))),
// adds dt A exp(.) E / (R theta^2) / 2 to the adjoints of both u and T3.

// adjoint of the step's damage term for the target voxels
// dJ/dT of the damage of one step (of length dt, from xa to xb) at either end
__device__ inline double adj_damage(const HeatArgs<double>& a, double dt, int m, double xa, double xb) {
  const double E = a.E[m], th = (xa + xb) / 2 + a.czero;
  return dt * exp(a.logA[m] - E / (a.Rgas * th)) * E / (a.Rgas * th * th) / 2;
}

__global__ void heat_adj_damage(HeatArgs<double> a, const double* __restrict__ x0, const double* __restrict__ x1,
                                const uint8_t* __restrict__ target, double* lam, int64_t L) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= L || !target[i]) return;
  const int m = a.M[i];
  if (a.E[m] != 0) lam[i] += adj_damage(a, a.dt, m, x0[i], x1[i]);
}

// A_d^T y = r on every line along axis d: lane per line, Thomas recurrence;
// `beta` holds the eliminated diagonal.
template <int AXIS>
__global__ void __launch_bounds__(kHeatTPB) heat_adj_solve(HeatArgs<double> a, const double* __restrict__ r, double* y, double* beta) {
  const int nx = a.nx, ny = a.ny, nz = a.nz, nxy = nx * ny;
  const int line = blockIdx.x * blockDim.x + threadIdx.x;
  int i0, st, n;
  bool lf;
  if (AXIS == 0) {
    if (line >= ny * nz) return;
    const int yy = line % ny, zz = line / ny;
    i0 = yy * nx + zz * nxy, st = 1, n = nx;
    lf = a.sinked && (yy == 0 || yy == ny - 1 || zz == 0 || zz == nz - 1);
  } else if (AXIS == 1) {
    if (line >= nx * nz) return;
    const int xx = line % nx, zz = line / nx;
    i0 = xx + zz * nxy, st = nx, n = ny;
    lf = a.sinked && (xx == 0 || xx == nx - 1 || zz == 0 || zz == nz - 1);
  } else {
    if (line >= nxy) return;
    const int xx = line % nx, yy = line / nx;
    i0 = line, st = nxy, n = nz;
    lf = a.sinked && (xx == 0 || xx == nx - 1 || yy == 0 || yy == ny - 1);
  }
  const double h = a.dt / 2;
  // row k of A_d: (sub, diag, super) = (ak, bk, ck)
  auto row = [&](int k, double& ak, double& bk, double& ck) {
    ak = 0;
    bk = 1;
    ck = 0;
    if (lf || (a.sinked && (k == 0 || k == n - 1))) return;
    const int i = i0 + k * st, m = a.M[i];
    if (k > 0) {
      const double q = h * cc(a, m, a.M[i - st], AXIS);
      bk += q;
      ak = -q;
    }
    if (k < n - 1) {
      const double q = h * cc(a, m, a.M[i + st], AXIS);
      bk += q;
      ck = -q;
    }
  };
  double aPrev, bPrev, cPrev, ak, bk, ck;
  row(0, ak, bk, ck);
  double bet = bk, yy = r[i0];
  beta[i0] = bet;
  y[i0] = yy;
  for (int k = 1; k < n; ++k) {
    aPrev = ak;
    bPrev = bk;
    cPrev = ck;
    row(k, ak, bk, ck);
    // A^T row k: sub = c_(k-1), diag = b_k; A^T row k-1 has super = a_k
    const double w = cPrev / bet;
    bet = bk - w * ak;
    const int i = i0 + k * st;
    yy = r[i] - w * yy;
    beta[i] = bet;
    y[i] = yy;
    (void)aPrev;
    (void)bPrev;
  }
  double xn = y[i0 + (n - 1) * st] / beta[i0 + (n - 1) * st];
  y[i0 + (n - 1) * st] = xn;
  double aNext;
  {
    double t0, t1;
    row(n - 1, aNext, t0, t1);
  }
  for (int k = n - 2; k >= 0; --k) {
    const int i = i0 + k * st;
    xn = (y[i] - aNext * xn) / beta[i];
    y[i] = xn;
    double t0, t1;
    row(k, aNext, t0, t1);
  }
}

// Rows of A_d^T on S consecutive voxels k0 .. k0+S-1 of a line of n voxels (lf:
// the whole line is frozen; Ml, Mr: media of the voxels before and after).  The
// rows of A^T are (sub, diag, super) = (c_(k-1), b_k, a_(k+1)) of A's rows,
// which vanish where voxel k-1 (k+1) is frozen.
template <int S>
__device__ inline void adj_rows(const HeatArgs<double>& a, const double* cT, int n, int k0, bool lf, const int (&Mv)[S], int Ml, int Mr,
                                double (&ta)[S], double (&tb)[S], double (&tc)[S]) {
  const double h = a.dt / 2;
  const int nM = a.nM;
  auto moves = [&](int k) { return k >= 0 && k < n && !lf && !(a.sinked && (k == 0 || k == n - 1)); };
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const int k = k0 + s, m = Mv[s];
    const int ML = s > 0 ? Mv[s - 1] : Ml, MR = s < S - 1 ? Mv[s + 1] : Mr;
    const double toL = coef(cT, nM, m, ML, 0), toR = coef(cT, nM, m, MR, 0), fromL = coef(cT, nM, ML, m, 0), fromR = coef(cT, nM, MR, m, 0);
    const bool on = moves(k);
    ta[s] = k < n && moves(k - 1) ? -h * fromL : 0.0;
    tc[s] = k < n && moves(k + 1) ? -h * fromR : 0.0;
    tb[s] = 1.0 + (on && k > 0 ? h * toL : 0.0) + (on && k < n - 1 ? h * toR : 0.0);
  }
}

// A_d^T y = r on x lines of up to 512 voxels, a line per W lanes.
template <int S, int W, bool LDS_COEF>
__global__ void __launch_bounds__(kHeatTPB) heat_adj_solve_x(HeatArgs<double> a, const double* __restrict__ r, double* __restrict__ y) {
  __shared__ double sC[LDS_COEF ? kAxisCoef : 1];
  const int nx = a.nx, ny = a.ny, nz = a.nz;
  // a segment past the last line solves the last line again and stores nothing
  const int wl = __lane_id(), lane = wl & (W - 1);
  const int seg = (xcd_contiguous(blockIdx.x, gridDim.x) * (kHeatTPB / 64) + (threadIdx.x >> 6)) * (64 / W) + wl / W;
  const bool valid = seg < ny * nz;
  const int line = valid ? seg : ny * nz - 1;
  const int yy = line % ny, zz = line / ny, i0 = line * nx;
  const bool lf = a.sinked && (yy == 0 || yy == ny - 1 || zz == 0 || zz == nz - 1);
  double rv[S], xs[S], ta[S], tb[S], tc[S];
  int Mv[S];
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const int k = lane * S + s, i = i0 + min(k, nx - 1);
    const double v = r[i];
    rv[s] = k < nx ? v : 0.0;
    Mv[s] = a.M[i];
  }
  if (LDS_COEF)
    for (int k = threadIdx.x; k < a.nM * a.nM; k += blockDim.x) sC[k] = a.c[k];
  __syncthreads();
  const int Ml = seg_shift<W, false>(Mv[S - 1], 1), Mr = seg_shift<W, true>(Mv[0], 1);
  adj_rows<S>(a, LDS_COEF ? sC : a.c, nx, lane * S, lf, Mv, Ml, Mr, ta, tb, tc);
  line_solve<S, W>(ta, tb, tc, rv, xs);
  if (!valid) return;
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const int k = lane * S + s;
    if (k < nx) y[i0 + k] = xs[s];
  }
}

// A_d^T y = r along y (AXIS 1) or z (AXIS 2), lines of up to 512 voxels laid
// out over the workgroups like the forward y/z sweeps.
template <int S, int NC, int AXIS, bool LDS_COEF>
__global__ void __launch_bounds__(NC * 16) heat_adj_solve_yz(HeatArgs<double> a, const double* __restrict__ r, double* __restrict__ y) {
  __shared__ LineLds<NC> lds;
  __shared__ double sC[LDS_COEF ? kAxisCoef : 1];
  const int nx = a.nx, ny = a.ny, nz = a.nz, nM = a.nM;
  const int n = AXIS == 1 ? ny : nz, nOther = AXIS == 1 ? nz : ny, st = AXIS == 1 ? nx : nx * ny;
  const LinePos L = line_pos<S, NC, AXIS>(nx, ny);
  double rv[S], xs[S], ta[S], tb[S], tc[S];
  int Mv[S];
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const int k = L.k0 + s, i = L.base + min(k, n - 1) * st;
    const double v = r[i];
    rv[s] = k < n ? v : 0.0;
    Mv[s] = a.M[i];
  }
  const int Ml = a.M[L.base + min(max(L.k0 - 1, 0), n - 1) * st], Mr = a.M[L.base + min(L.k0 + S, n - 1) * st];
  if (LDS_COEF)
    for (int k = threadIdx.x; k < nM * nM; k += blockDim.x) sC[k] = a.c[k + AXIS * nM * nM];
  __syncthreads();
  const bool lf = a.sinked && (L.x == 0 || L.x == nx - 1 || L.o == 0 || L.o == nOther - 1);
  adj_rows<S>(a, LDS_COEF ? sC : a.c + AXIS * nM * nM, n, L.k0, lf, Mv, Ml, Mr, ta, tb, tc);
  block_line_solve<S, NC>(ta, tb, tc, rv, xs, lds);
  if (!L.valid) return;
#pragma unroll
  for (int s = 0; s < S; ++s)
    if (L.k0 + s < n) y[L.base + (L.k0 + s) * st] = xs[s];
}

__device__ inline bool heat_frozen(const HeatArgs<double>& a, int x, int y, int z) { return frozen(a, x, y, z); }

// lam_u of the step (plus the damage adjoint of u) and the source adjoint.
template <bool LDS_COEF>
__global__ void __launch_bounds__(kHeatTPB) heat_adj_combine(HeatArgs<double> a, const double* __restrict__ mu1, const double* __restrict__ mu2,
                                                            const double* __restrict__ mu3, const double* __restrict__ x0,
                                                            const double* __restrict__ x1, const uint8_t* __restrict__ target,
                                                            double* lamOut, double* dQ, int lightsOn, const double* __restrict__ xm,
                                                            double dtm) {
  __shared__ double sC[LDS_COEF ? kLdsCoef : 1];
  if (LDS_COEF) {
    for (int k = threadIdx.x; k < a.nM * a.nM * 3; k += blockDim.x) sC[k] = a.c[k];
    __syncthreads();
  }
  const double* __restrict__ cT = LDS_COEF ? sC : a.c;
  const int nx = a.nx, ny = a.ny, nz = a.nz, nxy = nx * ny;
  // whole workgroups per z plane, so that index arithmetic is 32-bit; each XCD
  // takes neighbouring planes and rows.  12.3 us at 96 x 80 x 72 with the damage
  // of the step before; 15.5 and 4.1 as two kernels in launch order.
  const int perPlane = (nxy + kHeatTPB - 1) / kHeatTPB, blk = xcd_contiguous(blockIdx.x, gridDim.x);
  const int z = blk / perPlane, p = (blk - z * perPlane) * kHeatTPB + threadIdx.x;
  if (p >= nxy) return;
  const int x = p % nx, y = p / nx;
  const int64_t i = (int64_t)z * nxy + p;
  const int m = a.M[i];
  const double dt = a.dt;
  // L_d^T (D w) at i for w = mu1, mu2, mu3.  Every neighbour is read, one outside
  // the grid as the voxel itself, and dropped by a select: all loads are under
  // way at once (14.2 us with a branch per neighbour, 12.3 so).
  const bool sk = a.sinked;
  const bool ix = sk && (x == 0 || x == nx - 1), iy = sk && (y == 0 || y == ny - 1), iz = sk && (z == 0 || z == nz - 1);
  const bool own = !(ix || iy || iz);
  const double w1 = own ? mu1[i] : 0.0, w2 = own ? mu2[i] : 0.0, w3 = own ? mu3[i] : 0.0;
  double t1[3] = {0, 0, 0}, t2 = 0, t3 = 0;
  const int xyz[3] = {x, y, z}, ext[3] = {nx, ny, nz}, step[3] = {1, nx, nxy};
  const bool fz[3] = {iy || iz, ix || iz, ix || iy};  // frozen by the other axes
#pragma unroll
  for (int d = 0; d < 3; ++d) {
#pragma unroll
    for (int s = -1; s <= 1; s += 2) {
      const int q = xyz[d] + s;
      const bool in = q >= 0 && q < ext[d], off = fz[d] || (sk && (q == 0 || q == ext[d] - 1));
      const int64_t j = in ? i + s * step[d] : i;
      const int mn = a.M[j];
      const double cin = coef(cT, a.nM, mn, m, d), cout = coef(cT, a.nM, m, mn, d);
      const double v1 = mu1[j], e1 = cin * (off ? 0.0 : v1) - cout * w1;
      t1[d] += in ? e1 : 0.0;
      if (d == 1) {
        const double v2 = mu2[j], e2 = cin * (off ? 0.0 : v2) - cout * w2;
        t2 += in ? e2 : 0.0;
      }
      if (d == 2) {
        const double v3 = mu3[j], e3 = cin * (off ? 0.0 : v3) - cout * w3;
        t3 += in ? e3 : 0.0;
      }
    }
  }
  double lam = mu1[i] + dt * (t1[0] / 2 + t1[1] + t1[2]) - dt / 2 * t2 - dt / 2 * t3;
  if (target[i] && a.E[m] != 0) {
    lam += adj_damage(a, dt, m, x0[i], x1[i]);
    // and what heat_adj_damage would add for the step before, from xm to x0
    if (xm) lam += adj_damage(a, dtm, m, xm[i], x0[i]);
  }
  lamOut[i] = lam;
  if (lightsOn) dQ[i] += dt * w1;
}

// Gradient with respect to the conduction coefficients c[a, b, d] (the
// reference's dTdtperdeltaT).  Perturbing c in the step's equations and
// applying the adjoints mu1..mu3 gives, with dL_d v at i = sum over the
// d-neighbours n of dc[M_i, M_n, d] (v_n - v_i),
//   dJ = dt/2 mu1^T D dL_x (u + T1)
//      + mu1^T D dL_y (dt u) + mu2^T D dL_y (dt/2 (T2 - u))
//      + mu1^T D dL_z (dt u) + mu3^T D dL_z (dt/2 (T3 - u)).
// The intermediate states follow from the step's two ends by undoing the
// line solves: T2 = A_z T3 + dt/2 D L_z u = T3 - dt/2 D L_z (T3 - u) and
// T1 = T2 - dt/2 D L_y (T2 - u).

// lo = hi - dt/2 D L_AXIS (hi - u)
template <int AXIS>
__global__ void __launch_bounds__(kHeatTPB) heat_adj_undo(HeatArgs<double> a, const double* __restrict__ hi, const double* __restrict__ u,
                                                         double* __restrict__ lo) {
  const int nx = a.nx, ny = a.ny, nz = a.nz, nxy = nx * ny;
  const int p = blockIdx.x * blockDim.x + threadIdx.x, z = blockIdx.y;
  if (p >= nxy) return;
  const int x = p % nx, y = p / nx;
  const int64_t i = (int64_t)z * nxy + p;
  const double vi = hi[i] - u[i];
  double l = 0;
  if (!heat_frozen(a, x, y, z)) {
    const int q = AXIS == 1 ? y : z, n = AXIS == 1 ? ny : nz;
    const int64_t st = AXIS == 1 ? nx : nxy;
    const int m = a.M[i];
    if (q > 0) l += coef(a.c, a.nM, m, (int)a.M[i - st], AXIS) * ((hi[i - st] - u[i - st]) - vi);
    if (q < n - 1) l += coef(a.c, a.nM, m, (int)a.M[i + st], AXIS) * ((hi[i + st] - u[i + st]) - vi);
  }
  lo[i] = hi[i] - a.dt / 2 * l;
}

// One step's contributions to dJ/dc, summed per (a, b, d) in LDS (one FP64
// LDS atomic per wavefront where all its lanes hit the same coefficient,
// the usual case away from interfaces) and added to the global sums; a
// grid-stride loop keeps the number of global atomics per step small.
constexpr int kCoefBins = 192;  // LDS bins: tables of up to 8 media
template <bool LDS_BINS>
__global__ void __launch_bounds__(kHeatTPB) heat_adj_coef(HeatArgs<double> a, const double* __restrict__ mu1, const double* __restrict__ mu2,
                                                         const double* __restrict__ mu3, const double* __restrict__ u,
                                                         const double* __restrict__ T1, const double* __restrict__ T2,
                                                         const double* __restrict__ T3, double* dJdc) {
  __shared__ double sB[LDS_BINS ? kCoefBins : 1];
  const int nM = a.nM, nB = nM * nM * 3;
  if (LDS_BINS) {
    for (int k = threadIdx.x; k < nB; k += blockDim.x) sB[k] = 0;
    __syncthreads();
  }
  const int nx = a.nx, ny = a.ny, nz = a.nz, nxy = nx * ny;
  const int64_t L = (int64_t)nxy * nz;
  const double dt = a.dt;
  const int lane = threadIdx.x & 63;
  const int64_t span = (int64_t)gridDim.x * blockDim.x;
  // whole wavefronts run the loop together (shuffles below need every lane)
  const int64_t iters = (L + span - 1) / span;
  for (int64_t it = 0; it < iters; ++it) {
    const int64_t i = it * span + (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool live = i < L;
    int x = 0, y = 0, z = 0, m = 0;
    bool act = false;
    if (live) {
      z = (int)(i / nxy);
      const int p = (int)(i - (int64_t)z * nxy);
      x = p % nx, y = p / nx;
      m = a.M[i];
      act = !heat_frozen(a, x, y, z);
    }
    for (int d = 0; d < 3; ++d) {
      for (int s = -1; s <= 1; s += 2) {
        double g = 0;
        int k = -1;
        if (act) {
          const int q = (d == 0 ? x : d == 1 ? y : z) + s, n = d == 0 ? nx : d == 1 ? ny : nz;
          if (q >= 0 && q < n) {
            const int64_t st = d == 0 ? 1 : d == 1 ? nx : nxy;
            const int64_t j = i + s * st;
            const int mn = a.M[j];
            k = m + mn * nM + d * nM * nM;
            if (d == 0) {
              g = dt / 2 * mu1[i] * ((u[j] + T1[j]) - (u[i] + T1[i]));
            } else {
              const double* W = d == 1 ? mu2 : mu3;
              const double* V = d == 1 ? T2 : T3;
              g = dt * mu1[i] * (u[j] - u[i]) + dt / 2 * W[i] * ((V[j] - u[j]) - (V[i] - u[i]));
            }
          }
        }
        if (LDS_BINS) {
          const int k0 = __shfl(k, 0);
          if (__all(k == k0) && k0 >= 0) {
            for (int off = 32; off > 0; off >>= 1) g += __shfl_xor(g, off);
            if (lane == 0) atomicAdd(&sB[k0], g);
          } else if (k >= 0) {
            atomicAdd(&sB[k], g);
          }
        } else if (k >= 0 && g != 0) {
          atomicAdd(&dJdc[k], g);
        }
      }
    }
  }
  if (LDS_BINS) {
    __syncthreads();
    for (int k = threadIdx.x; k < nB; k += blockDim.x)
      if (sB[k] != 0) atomicAdd(&dJdc[k], sB[k]);
  }
}

}  // namespace mcm

using namespace mcm;

struct HeatBuf {
  void* p = nullptr;
  void release() {
    if (p) (void)hipFree(p);
    p = nullptr;
  }
  ~HeatBuf() { release(); }
};

// An instantiated graph of `steps` time steps at one (dt, lights) setting,
// valid while the state and sensor buffers it captured stay in place.
struct HeatGraph {
  hipGraphExec_t exec = nullptr;
  int64_t steps = 0;
  double dt = 0;
  int lightsOn = 0;
  const void *T1 = nullptr, *sensors = nullptr;
  bool factored = false;  // the captured FP32 sweeps read the line factors
};

struct mcm_heat_plan {
  int device = 0;
  hipStream_t stream = nullptr;
  int fp32 = 0, explicitScheme = 0;
  int explicitZRun = 16;  // z planes per workgroup of the explicit stencil
  int nx = 0, ny = 0, nz = 0, nM = 0;
  int64_t L = 0;
  int sinked = 0, calcDamage = 0;
  int64_t nS = 0;
  int64_t stepsDone = 0;
  int64_t sensorsRecorded = 0;  // sensor columns 0 .. sensorsRecorded-1 are in `sensors`
  int64_t sensorCap = 0;      // columns allocated in `sensors`
  bool interrupted = false;
  int (*interrupt)(void) = nullptr;
  HeatBuf M, Q, c, logA, E, T1, T2, B, Om, maxKey, sIdx, sW, sensors, stage32, stage64, stepDev;
  HeatBuf fac[3];             // FP32 line factors (ensure_factors) for facDt
  bool facReady = false;
  double facDt = 0;
  bool factored(double dt) const { return facReady && facDt == dt; }
  double constR = 0, constC = 0;
  HostStage hostStage;
  int64_t graphSteps = 32;    // steps per captured graph (0: launch every step)
  std::vector<HeatGraph> graphs;
  void drop_graphs() {
    for (HeatGraph& g : graphs)
      if (g.exec) (void)hipGraphExecDestroy(g.exec);
    graphs.clear();
  }
  ~mcm_heat_plan() {
    drop_graphs();
    if (stream) (void)hipStreamDestroy(stream);
  }
};

// Plans advanced together: one graph holds K steps of every plan, each plan
// a branch on its own stream, so the small kernels of different grids run
// concurrently.
struct mcm_heat_group {
  int device = 0;
  std::vector<mcm_heat_plan*> plans;
  std::vector<hipEvent_t> events;  // [0] fork, [1 + i] join of plan i
  struct Graph {
    hipGraphExec_t exec = nullptr;
    int64_t steps = 0;
    std::vector<double> dt;
    std::vector<int> lightsOn;
    std::vector<const void*> T1, sensors;
    std::vector<bool> factored;
  };
  std::vector<Graph> graphs;
  void drop_graphs() {
    for (Graph& g : graphs)
      if (g.exec) (void)hipGraphExecDestroy(g.exec);
    graphs.clear();
  }
  ~mcm_heat_group() {
    drop_graphs();
    for (hipEvent_t e : events) (void)hipEventDestroy(e);
  }
};

namespace {

size_t rt_size(const mcm_heat_plan* p) { return p->fp32 ? sizeof(float) : sizeof(double); }

int halloc(HeatBuf& b, size_t bytes) {
  MCM_HIP(hipMalloc(&b.p, std::max<size_t>(bytes, 8)));
  return MCM_OK;
}

template <typename RT>
void launch_explicit(mcm_heat_plan* P, const HeatArgs<RT>& a, int zr) {
  const int64_t nxy = (int64_t)P->nx * P->ny;
  const unsigned ge = (unsigned)((nxy + kHeatTPB - 1) / kHeatTPB * ((P->nz + zr - 1) / zr));
  auto go = [&](auto off) {
    using OFF = decltype(off);
    if (P->nM * P->nM * 3 <= kLdsCoef) hipLaunchKernelGGL((heat_explicit_march<RT, true, OFF>), dim3(ge), dim3(kHeatTPB), 0, P->stream, a, zr);
    else hipLaunchKernelGGL((heat_explicit_march<RT, false, OFF>), dim3(ge), dim3(kHeatTPB), 0, P->stream, a, zr);
  };
  if (nxy < ((int64_t)1 << 28)) go(uint32_t());
  else go(uint64_t());
}

template <typename RT>
HeatArgs<RT> make_args(mcm_heat_plan* P, double dt, int lightsOn) {
  HeatArgs<RT> a{};
  a.nx = P->nx;
  a.ny = P->ny;
  a.nz = P->nz;
  a.nM = P->nM;
  a.sinked = P->sinked;
  a.lightsOn = lightsOn;
  a.calcDamage = P->calcDamage;
  a.dt = (RT)dt;
  a.Rgas = (RT)P->constR;
  a.czero = (RT)P->constC;
  a.M = (const uint8_t*)P->M.p;
  a.Q = (const float*)P->Q.p;
  a.c = (const RT*)P->c.p;
  a.logA = (const RT*)P->logA.p;
  a.E = (const RT*)P->E.p;
  a.T1 = (const RT*)P->T1.p;
  a.T2 = (RT*)P->T2.p;
  a.B = (RT*)P->B.p;
  a.Om = (RT*)P->Om.p;
  a.maxKey = (unsigned long long*)P->maxKey.p;
  if (P->factored(dt))
    for (int d = 0; d < 3; ++d) a.fac[d] = (float*)P->fac[d].p;
  return a;
}

// The explicit stencil's best run of z planes per workgroup depends on how
// the workgroup count fills the GPU (measured, us/step at 100^3 / 200^3 /
// 225x190x171 / 256x256x120: 8 planes 11.7 / 43.8 / 40.7 / 41.3, 12 planes
// 13.7 / 43.1 / 37.6 / 39.7, 16 planes 16.6 / 41.1 / 40.5 / 41.3, 24 planes
// 21.2 / 50.1 / 48.8 / 37.6, 32 planes 27.8 / 42.8 / 39.2 / 38.7), so each
// explicit plan times a few candidate runs once at
// creation.  The trial steps read the initial state and write only the
// other state buffer (overwritten by the first real step), a scratch damage
// field (the DG-ADI work buffer, unused by this scheme) and scratch maxima;
// no sensor is recorded.
// The choice is kept per grid shape, precision and device for the process,
// so later plans of the same shape (a schedule cut into many calls) do not
// time again; a plan created for fewer than kTuneMinSteps steps does not
// time at all and takes kDefaultZRun, unless the shape is known.
constexpr int kDefaultZRun = 16;
constexpr int64_t kTuneMinSteps = 64;
std::mutex g_zrunMutex;
std::map<std::array<int, 6>, int> g_zrunCache;

bool valid_zrun(int zr) { return zr == 8 || zr == 12 || zr == 16 || zr == 24 || zr == 32; }

template <typename RT>
int tune_explicit(mcm_heat_plan* P, int64_t steps) {
  const std::array<int, 6> key = {P->device, P->nx, P->ny, P->nz, P->fp32, P->nM * P->nM * 3 <= kLdsCoef};
  if (const char* e = std::getenv("MCM_HEAT_ZRUN")) {
    const int zr = std::atoi(e);
    if (valid_zrun(zr)) {
      P->explicitZRun = zr;
      return MCM_OK;
    }
  }
  {
    std::lock_guard<std::mutex> lk(g_zrunMutex);
    auto it = g_zrunCache.find(key);
    if (it != g_zrunCache.end()) {
      P->explicitZRun = it->second;
      return MCM_OK;
    }
  }
  if (steps < kTuneMinSteps) {
    P->explicitZRun = kDefaultZRun;
    return MCM_OK;
  }
  HeatArgs<RT> a = make_args<RT>(P, 1e-9, 1);
  a.Om = (RT*)P->B.p;
  HeatBuf keys;
  if (int rc = halloc(keys, (size_t)P->nM * 8)) return rc;
  a.maxKey = (unsigned long long*)keys.p;
  hipEvent_t e0, e1;
  MCM_HIP(hipEventCreate(&e0));
  MCM_HIP(hipEventCreate(&e1));
  float best = 0.f;
  int bestZ = 16;
  for (int zr : {8, 12, 16, 24, 32}) {
    if (zr > 8 && zr >= P->nz + 8) break;  // longer runs than the grid change nothing
    launch_explicit<RT>(P, a, zr);
    (void)hipEventRecord(e0, P->stream);
    for (int r = 0; r < 3; ++r) launch_explicit<RT>(P, a, zr);
    (void)hipEventRecord(e1, P->stream);
    float ms = 0.f;
    if (hipEventSynchronize(e1) != hipSuccess || hipEventElapsedTime(&ms, e0, e1) != hipSuccess) break;
    if (best == 0.f || ms < best) best = ms, bestZ = zr;
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  MCM_HIP(hipGetLastError());
  MCM_HIP(hipStreamSynchronize(P->stream));
  P->explicitZRun = bestZ;
  std::lock_guard<std::mutex> lk(g_zrunMutex);
  g_zrunCache[key] = bestZ;
  return MCM_OK;
}

int ensure_sensor_capacity(mcm_heat_plan* P, int64_t cols) {
  if (P->nS == 0 || cols <= P->sensorCap) return MCM_OK;
  int64_t cap = std::max<int64_t>(cols, 2 * P->sensorCap);
  void* np = nullptr;
  MCM_HIP(hipMalloc(&np, (size_t)(cap * P->nS) * sizeof(double)));
  if (P->sensors.p) {
    MCM_HIP(hipMemcpyAsync(np, P->sensors.p, (size_t)(P->sensorCap * P->nS) * sizeof(double), hipMemcpyDeviceToDevice, P->stream));
    MCM_HIP(hipStreamSynchronize(P->stream));
    MCM_HIP(hipFree(P->sensors.p));
  }
  P->sensors.p = np;
  P->sensorCap = cap;
  return MCM_OK;
}

template <typename RT>
int record_sensors(mcm_heat_plan* P, int64_t col) {
  if (P->nS == 0) return MCM_OK;
  hipLaunchKernelGGL(heat_sensors<RT>, dim3(1), dim3(256), 0, P->stream, (const RT*)P->T1.p, P->nx, P->nx * P->ny,
                     (const long long*)P->sIdx.p, (const RT*)P->sW.p, (int)P->nS, (double*)P->sensors.p, (long long)col);
  MCM_HIP(hipGetLastError());
  return MCM_OK;
}

// FP32 sweep along axis KIND through LDS (build: its factors); false when the
// line is too long.
template <int KIND>
bool launch_lines32(mcm_heat_plan* P, const HeatArgs<float>& a, bool build = false) {
  const int n = KIND == SWEEP_X ? P->nx : KIND == SWEEP_Y ? P->ny : P->nz, tl = line32_lines(n);
  if (!tl) return false;
  const size_t lds = (size_t)tl * (n | 1) * 16;
  auto go = [&](auto TL) {
    constexpr int T = decltype(TL)::value;
    const dim3 g(KIND == SWEEP_X ? (unsigned)((P->ny * P->nz + T - 1) / T)
                                 : (unsigned)(((P->nx + T - 1) / T) * (KIND == SWEEP_Y ? P->nz : P->ny)));
    const dim3 b(kLine32TPB);
    if (build) hipLaunchKernelGGL((heat_sweep_lines32<KIND, T, LINES_BUILD, true>), g, b, lds, P->stream, a);
    else if (a.fac[KIND]) hipLaunchKernelGGL((heat_sweep_lines32<KIND, T, LINES_FACTORED, true>), g, b, lds, P->stream, a);
    else if (P->nM * P->nM * 3 <= kLdsCoef) hipLaunchKernelGGL((heat_sweep_lines32<KIND, T, LINES_PLAIN, true>), g, b, lds, P->stream, a);
    else hipLaunchKernelGGL((heat_sweep_lines32<KIND, T, LINES_PLAIN, false>), g, b, lds, P->stream, a);
  };
  if (tl == 32) go(std::integral_constant<int, 32>());
  else if (tl == 16) go(std::integral_constant<int, 16>());
  else go(std::integral_constant<int, 8>());
  return true;
}

// The FP32 line factors for dt, built when a run of at least kFactorSteps steps
// starts with another dt than the last such run's (building them costs about
// what one step gains three times over).  Runs without them compute them row
// by row.  Not called while a stream captures: captured steps read the
// buffers, which every run refills for its own dt before its replays.
constexpr int64_t kFactorSteps = 4;
int ensure_factors(mcm_heat_plan* P, int64_t steps, double dt) {
  if (!P->fp32 || P->explicitScheme) return MCM_OK;
  if (P->factored(dt)) return MCM_OK;
  if (steps < kFactorSteps || P->nM * P->nM * 3 > kLdsCoef) {
    P->facReady = false;
    return MCM_OK;
  }
  const int n[3] = {P->nx, P->ny, P->nz};
  for (int d = 0; d < 3; ++d)
    if (line32_lines(n[d]) && !P->fac[d].p && hipMalloc(&P->fac[d].p, (size_t)P->L * 4) != hipSuccess) {
      (void)hipGetLastError();
      P->fac[d].p = nullptr;
      for (HeatBuf& f : P->fac) f.release();  // (all or none: nothing captured reads them)
      P->facReady = false;
      return MCM_OK;
    }
  P->facReady = true;
  P->facDt = dt;
  const HeatArgs<float> a = make_args<float>(P, dt, 0);
  launch_lines32<SWEEP_X>(P, a, true);
  launch_lines32<SWEEP_Y>(P, a, true);
  launch_lines32<SWEEP_Z>(P, a, true);
  MCM_HIP(hipGetLastError());
  return MCM_OK;
}

// Lane-per-line y (AXIS 1) or z (AXIS 2) sweep, coefficients in LDS when
// they fit.
template <typename RT, int AXIS>
void launch_lane_sweep(mcm_heat_plan* P, const HeatArgs<RT>& a, unsigned g) {
  const bool lc = P->nM * P->nM * 3 <= kLdsCoef;
  if (AXIS == 1) {
    if (lc) hipLaunchKernelGGL((heat_sweep_y<RT, true>), dim3(g), dim3(kHeatTPB), 0, P->stream, a);
    else hipLaunchKernelGGL((heat_sweep_y<RT, false>), dim3(g), dim3(kHeatTPB), 0, P->stream, a);
  } else {
    if (lc) hipLaunchKernelGGL((heat_sweep_z<RT, true>), dim3(g), dim3(kHeatTPB), 0, P->stream, a);
    else hipLaunchKernelGGL((heat_sweep_z<RT, false>), dim3(g), dim3(kHeatTPB), 0, P->stream, a);
  }
}

// x-sweep launch: the wavefront solver for FP64 lines of up to 512 voxels,
// else the sequential lane-per-line kernel (FP32 keeps the reference's
// sequential recurrence).
template <typename RT>
void launch_sweep_x(mcm_heat_plan* P, const HeatArgs<RT>& a, unsigned gx) {
  if constexpr (std::is_same<RT, double>::value) {
    if (wave_line(P->nx)) {
      const bool lc = P->nM * P->nM * 3 <= kLdsCoef;
      with_x_shape(P->nx, [&](auto sTag, auto wTag) {
        constexpr int SS = decltype(sTag)::value, WW = decltype(wTag)::value;
        const int64_t lines = (int64_t)P->ny * P->nz, perBlock = kHeatTPB / WW;
        const unsigned gw = (unsigned)((lines + perBlock - 1) / perBlock);
        if (lc) hipLaunchKernelGGL((heat_sweep_x_wave<SS, WW, true>), dim3(gw), dim3(kHeatTPB), 0, P->stream, a);
        else hipLaunchKernelGGL((heat_sweep_x_wave<SS, WW, false>), dim3(gw), dim3(kHeatTPB), 0, P->stream, a);
      });
      return;
    }
  } else if (launch_lines32<SWEEP_X>(P, a)) {
    return;
  }
  if (P->nM * P->nM * 3 <= kLdsCoef) hipLaunchKernelGGL((heat_sweep_x<RT, true>), dim3(gx), dim3(kHeatTPB), 0, P->stream, a);
  else hipLaunchKernelGGL((heat_sweep_x<RT, false>), dim3(gx), dim3(kHeatTPB), 0, P->stream, a);
}

// y and z sweeps: the wavefront solver for FP64 lines of up to 512 voxels,
// else the sequential lane-per-line kernels.
template <int KIND>
void launch_yz_wave(mcm_heat_plan* P, const HeatArgs<double>& a, int n) {
  with_yz_shape(n, [&](auto sTag, auto cTag) {
    constexpr int S = decltype(sTag)::value, NC = decltype(cTag)::value;
    const unsigned g = (unsigned)(((P->nx + 15) / 16) * (KIND == SWEEP_Y ? P->nz : P->ny));
    if (P->nM * P->nM <= kAxisCoef) hipLaunchKernelGGL((heat_sweep_yz<S, NC, KIND, true>), dim3(g), dim3(NC * 16), 0, P->stream, a);
    else hipLaunchKernelGGL((heat_sweep_yz<S, NC, KIND, false>), dim3(g), dim3(NC * 16), 0, P->stream, a);
  });
}

template <typename RT>
void launch_sweep_yz(mcm_heat_plan* P, const HeatArgs<RT>& a, unsigned gy, unsigned gz) {
  if constexpr (std::is_same<RT, double>::value) {
    if (wave_line(P->ny)) launch_yz_wave<SWEEP_Y>(P, a, P->ny);
    else launch_lane_sweep<RT, 1>(P, a, gy);
    if (wave_line(P->nz)) launch_yz_wave<SWEEP_Z>(P, a, P->nz);
    else launch_lane_sweep<RT, 2>(P, a, gz);
  } else {
    if (!launch_lines32<SWEEP_Y>(P, a)) launch_lane_sweep<RT, 1>(P, a, gy);
    if (!launch_lines32<SWEEP_Z>(P, a)) launch_lane_sweep<RT, 2>(P, a, gz);
  }
}

// The kernels of one time step on the plan's stream; swaps the state buffers.
template <typename RT>
void enqueue_step(mcm_heat_plan* P, double dt, int lightsOn, const long long* colBase, long long col) {
  const int tpb = kHeatTPB;
  HeatArgs<RT> a = make_args<RT>(P, dt, lightsOn);
  if (P->nS) {
    // the step's first kernel records the state it starts from
    a.nS = (int)P->nS;
    a.sIdx = (const long long*)P->sIdx.p;
    a.sW = (const RT*)P->sW.p;
    a.sOut = (double*)P->sensors.p;
    a.sColBase = colBase;
    a.sCol = col;
  }
  if (P->explicitScheme) {
    launch_explicit<RT>(P, a, P->explicitZRun);
    (void)tpb;
  } else {
    launch_sweep_x<RT>(P, a, (unsigned)((P->ny * P->nz + tpb - 1) / tpb));
    launch_sweep_yz<RT>(P, a, (unsigned)((P->nx * P->nz + tpb - 1) / tpb), (unsigned)((P->nx * P->ny + tpb - 1) / tpb));
  }
  std::swap(P->T1.p, P->T2.p);
}

// K (even) steps as graph nodes on the plan's stream, which is capturing:
// step k records sensor column (device step counter) + k, and the last node
// advances the counter by K.  An even K leaves T1/T2 where they were.
template <typename RT>
void enqueue_graph_steps(mcm_heat_plan* P, int64_t K, double dt, int lightsOn) {
  for (int64_t k = 0; k < K; ++k) enqueue_step<RT>(P, dt, lightsOn, (const long long*)P->stepDev.p, (long long)k);
  if (P->nS) hipLaunchKernelGGL(heat_step_counter, dim3(1), dim3(64), 0, P->stream, (long long*)P->stepDev.p, (long long)K, 1);
}

// The cached graph of K steps at (dt, lightsOn) for the current buffers, or
// a new capture (at most four are kept).
template <typename RT>
int step_graph(mcm_heat_plan* P, int64_t K, double dt, int lightsOn, hipGraphExec_t* out) {
  for (HeatGraph& g : P->graphs)
    if (g.steps == K && g.dt == dt && g.lightsOn == lightsOn && g.T1 == P->T1.p && g.sensors == P->sensors.p && g.factored == P->factored(dt)) {
      *out = g.exec;
      return MCM_OK;
    }
  if (P->nS && !P->stepDev.p) MCM_HIP(hipMalloc(&P->stepDev.p, sizeof(long long)));
  MCM_HIP(hipStreamBeginCapture(P->stream, hipStreamCaptureModeThreadLocal));
  enqueue_graph_steps<RT>(P, K, dt, lightsOn);
  hipGraph_t graph = nullptr;
  const hipError_t launchErr = hipGetLastError();
  const hipError_t endErr = hipStreamEndCapture(P->stream, &graph);
  if (launchErr != hipSuccess || endErr != hipSuccess) {
    if (graph) (void)hipGraphDestroy(graph);
    return fail(MCM_ERR_DEVICE, "capturing %lld heat steps: %s", (long long)K, hipGetErrorString(launchErr != hipSuccess ? launchErr : endErr));
  }
  hipGraphExec_t exec = nullptr;
  const hipError_t instErr = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
  (void)hipGraphDestroy(graph);
  if (instErr != hipSuccess) return fail(MCM_ERR_DEVICE, "instantiating the heat step graph: %s", hipGetErrorString(instErr));
  if (P->graphs.size() >= 4) {
    // the oldest graph may still be queued or running on the stream: an
    // executable graph is destroyed only once its launches have finished
    MCM_HIP(hipStreamSynchronize(P->stream));
    (void)hipGraphExecDestroy(P->graphs.front().exec);
    P->graphs.erase(P->graphs.begin());
  }
  HeatGraph g;
  g.exec = exec;
  g.steps = K;
  g.dt = dt;
  g.lightsOn = lightsOn;
  g.T1 = P->T1.p;
  g.sensors = P->sensors.p;
  g.factored = P->factored(dt);
  P->graphs.push_back(g);
  *out = exec;
  return MCM_OK;
}

template <typename RT>
int advance(mcm_heat_plan* P, int64_t steps, double dt, int lightsOn) {
  int rc = ensure_sensor_capacity(P, P->stepsDone + steps + 1);
  if (rc) return rc;
  if ((rc = ensure_factors(P, steps, dt))) return rc;
  int64_t n = 0;
  // runs of K steps replay one captured graph (one launch instead of 2-4
  // per step); the interrupt is polled between replays
  const int64_t K = P->graphSteps & ~(int64_t)1;
  if (K >= 2 && steps >= 2 * K) {
    hipGraphExec_t g = nullptr;
    if ((rc = step_graph<RT>(P, K, dt, lightsOn, &g))) return rc;
    if (P->nS) hipLaunchKernelGGL(heat_step_counter, dim3(1), dim3(64), 0, P->stream, (long long*)P->stepDev.p, (long long)P->stepsDone, 0);
    for (; steps - n >= K; n += K) {
      if (P->interrupt && P->interrupt()) {
        P->interrupted = true;
        return MCM_OK;
      }
      MCM_HIP(hipGraphLaunch(g, P->stream));
      P->stepsDone += K;
      P->sensorsRecorded = P->stepsDone;
    }
  }
  for (; n < steps; ++n) {
    if (P->interrupt && P->interrupt()) {
      P->interrupted = true;
      break;
    }
    enqueue_step<RT>(P, dt, lightsOn, nullptr, P->stepsDone);
    MCM_HIP(hipGetLastError());
    ++P->stepsDone;
    P->sensorsRecorded = P->stepsDone;
  }
  return MCM_OK;
}

// The conduction coefficients.  Those of media that never meet along an axis
// (none do along an axis of one voxel) may have any value, but some kernels read
// one for a neighbour outside the grid, as a factor of a zero difference: where
// such a coefficient is infinite or no number it is 0 here.
std::vector<float> used_coefficients(const mcm_heat_input* in) {
  const int64_t nM = in->nM, n[3] = {in->nx, in->ny, in->nz}, st[3] = {1, in->nx, in->nx * in->ny}, L = n[0] * n[1] * n[2];
  std::vector<float> c(in->dTdtperdeltaT, in->dTdtperdeltaT + nM * nM * 3);
  if (std::all_of(c.begin(), c.end(), [](float v) { return std::isfinite(v); })) return c;
  std::vector<uint8_t> meet(c.size(), 0);
  for (int d = 0; d < 3; ++d)
    for (int64_t i = 0; i < L; ++i) {
      if (i / st[d] % n[d] == n[d] - 1) continue;
      const int64_t a = in->M[i], b = in->M[i + st[d]];
      meet[a + b * nM + d * nM * nM] = meet[b + a * nM + d * nM * nM] = 1;
    }
  for (size_t k = 0; k < c.size(); ++k)
    if (!meet[k] && !std::isfinite(c[k])) c[k] = 0.f;
  return c;
}

template <typename RT>
int upload_state(mcm_heat_plan* P, const mcm_heat_input* in) {
  const int tpb = 256;
  const unsigned nb = (unsigned)((P->L + tpb - 1) / tpb);
  // stage the host arrays through device buffers, then convert on the device
  if (in->T_f64) {
    MCM_HIP(hipMemcpyAsync(P->stage64.p, in->T_f64, (size_t)P->L * 8, hipMemcpyHostToDevice, P->stream));
    hipLaunchKernelGGL(heat_load<RT>, dim3(nb), dim3(tpb), 0, P->stream, (RT*)P->T1.p, nullptr, (const double*)P->stage64.p, P->L);
  } else {
    MCM_HIP(hipMemcpyAsync(P->stage32.p, in->T, (size_t)P->L * 4, hipMemcpyHostToDevice, P->stream));
    hipLaunchKernelGGL(heat_load<RT>, dim3(nb), dim3(tpb), 0, P->stream, (RT*)P->T1.p, (const float*)P->stage32.p, nullptr, P->L);
  }
  MCM_HIP(hipStreamSynchronize(P->stream));
  if (P->calcDamage) {
    if (in->Omega_f64) {
      MCM_HIP(hipMemcpyAsync(P->stage64.p, in->Omega_f64, (size_t)P->L * 8, hipMemcpyHostToDevice, P->stream));
      hipLaunchKernelGGL(heat_load<RT>, dim3(nb), dim3(tpb), 0, P->stream, (RT*)P->Om.p, nullptr, (const double*)P->stage64.p, P->L);
    } else {
      MCM_HIP(hipMemcpyAsync(P->stage32.p, in->Omega, (size_t)P->L * 4, hipMemcpyHostToDevice, P->stream));
      hipLaunchKernelGGL(heat_load<RT>, dim3(nb), dim3(tpb), 0, P->stream, (RT*)P->Om.p, (const float*)P->stage32.p, nullptr, P->L);
    }
  }
  MCM_HIP(hipGetLastError());
  MCM_HIP(hipStreamSynchronize(P->stream));
  return MCM_OK;
}

template <typename RT>
int download(mcm_heat_plan* P, mcm_heat_output* out) {
  const int tpb = 256;
  const unsigned nb = (unsigned)((P->L + tpb - 1) / tpb);
  int rc = MCM_OK;
  MCM_HIP(hipStreamSynchronize(P->stream));
  if (out->T || out->T_f64) {
    hipLaunchKernelGGL(heat_store<RT>, dim3(nb), dim3(tpb), 0, P->stream, (const RT*)P->T1.p, (float*)P->stage32.p,
                       (double*)(out->T_f64 ? P->stage64.p : nullptr), P->L);
    MCM_HIP(hipGetLastError());
    if (out->T && (rc = P->hostStage.download(out->T, P->stage32.p, (size_t)P->L * 4, P->device, P->stream))) return rc;
    if (out->T_f64 && (rc = P->hostStage.download(out->T_f64, P->stage64.p, (size_t)P->L * 8, P->device, P->stream))) return rc;
  }
  if (P->calcDamage && (out->Omega || out->Omega_f64)) {
    hipLaunchKernelGGL(heat_store<RT>, dim3(nb), dim3(tpb), 0, P->stream, (const RT*)P->Om.p, (float*)P->stage32.p,
                       (double*)(out->Omega_f64 ? P->stage64.p : nullptr), P->L);
    MCM_HIP(hipGetLastError());
    if (out->Omega && (rc = P->hostStage.download(out->Omega, P->stage32.p, (size_t)P->L * 4, P->device, P->stream))) return rc;
    if (out->Omega_f64 && (rc = P->hostStage.download(out->Omega_f64, P->stage64.p, (size_t)P->L * 8, P->device, P->stream))) return rc;
  } else if (!P->calcDamage && out->Omega) {
    out->Omega[0] = NAN;
  }
  if (P->nS && P->sensorsRecorded <= P->stepsDone) {
    // the current state's column (steps record the state they start from)
    rc = ensure_sensor_capacity(P, P->stepsDone + 1);
    if (rc) return rc;
    if ((rc = record_sensors<RT>(P, P->stepsDone))) return rc;
    P->sensorsRecorded = P->stepsDone + 1;
  }
  if (out->sensorTemps && P->nS) {
    MCM_HIP(hipMemcpyAsync(out->sensorTemps, P->sensors.p, (size_t)((P->stepsDone + 1) * P->nS) * sizeof(double), hipMemcpyDeviceToHost,
                           P->stream));
  }
  if (out->maxMediaTemps) {
    std::vector<unsigned long long> keys((size_t)P->nM);
    MCM_HIP(hipMemcpyAsync(keys.data(), P->maxKey.p, keys.size() * 8, hipMemcpyDeviceToHost, P->stream));
    MCM_HIP(hipStreamSynchronize(P->stream));
    for (int m = 0; m < P->nM; ++m) out->maxMediaTemps[m] = (float)key_value(keys[m]);
  }
  MCM_HIP(hipStreamSynchronize(P->stream));
  out->stepsDone = P->stepsDone;
  return MCM_OK;
}

// A_d^T solve along axis AXIS: the wavefront solver for lines of up to 512
// voxels, else the lane-per-line recurrence.
template <int AXIS>
void adj_solve(mcm_heat_plan* P, const HeatArgs<double>& a, const double* r, double* y, double* beta, unsigned gLane) {
  const int n = AXIS == 0 ? P->nx : AXIS == 1 ? P->ny : P->nz;
  const int64_t lines = AXIS == 0 ? (int64_t)P->ny * P->nz : AXIS == 1 ? (int64_t)P->nx * P->nz : (int64_t)P->nx * P->ny;
  if (!wave_line(n)) {
    hipLaunchKernelGGL(heat_adj_solve<AXIS>, dim3(gLane), dim3(kHeatTPB), 0, P->stream, a, r, y, beta);
    return;
  }
  if constexpr (AXIS != 0) {
    with_yz_shape(n, [&](auto sTag, auto cTag) {
      constexpr int S = decltype(sTag)::value, NC = decltype(cTag)::value;
      const unsigned g = (unsigned)(((P->nx + 15) / 16) * (AXIS == 1 ? P->nz : P->ny));
      if (P->nM * P->nM <= kAxisCoef) hipLaunchKernelGGL((heat_adj_solve_yz<S, NC, AXIS, true>), dim3(g), dim3(NC * 16), 0, P->stream, a, r, y);
      else hipLaunchKernelGGL((heat_adj_solve_yz<S, NC, AXIS, false>), dim3(g), dim3(NC * 16), 0, P->stream, a, r, y);
    });
  } else {
    with_x_shape(n, [&](auto sTag, auto wTag) {
      constexpr int S = decltype(sTag)::value, W = decltype(wTag)::value;
      const unsigned gw = (unsigned)((lines + kHeatTPB / W - 1) / (kHeatTPB / W));
      if (P->nM * P->nM <= kAxisCoef) hipLaunchKernelGGL((heat_adj_solve_x<S, W, true>), dim3(gw), dim3(kHeatTPB), 0, P->stream, a, r, y);
      else hipLaunchKernelGGL((heat_adj_solve_x<S, W, false>), dim3(gw), dim3(kHeatTPB), 0, P->stream, a, r, y);
    });
  }
}

}  // namespace

extern "C" {

int mcm_heat_plan_create(const mcm_heat_input* in, mcm_heat_plan** out) {
  if (!in || !out) return fail(MCM_ERR_INVALID_ARGUMENT, "null argument");
  *out = nullptr;
  if (in->nx < 1 || in->ny < 1 || in->nz < 1) return fail(MCM_ERR_INVALID_ARGUMENT, "grid dimensions must be positive");
  if (in->nx * in->ny * in->nz >= ((int64_t)1 << 31)) return fail(MCM_ERR_INVALID_ARGUMENT, "grid too large for 32-bit voxel indices");
  if (in->nM < 1 || in->nM > 256) return fail(MCM_ERR_INVALID_ARGUMENT, "number of media must be 1..256");
  if (!in->T || !in->M || !in->dTdtperdeltaT || !in->dTdt_abs || !in->A || !in->E)
    return fail(MCM_ERR_INVALID_ARGUMENT, "missing T, M, dTdtperdeltaT, dTdt_abs, A or E");
  if (in->steps < 0) return fail(MCM_ERR_INVALID_ARGUMENT, "steps must be non-negative");
  if (in->precision != MCM_HEAT_FP64 && in->precision != MCM_HEAT_FP32) return fail(MCM_ERR_INVALID_ARGUMENT, "unknown precision");
  if (in->scheme != MCM_HEAT_DGADI && in->scheme != MCM_HEAT_EXPLICIT) return fail(MCM_ERR_INVALID_ARGUMENT, "unknown scheme");
  if (in->nSensors < 0 || (in->nSensors > 0 && (!in->tempSensorCornerIdxs || !in->tempSensorInterpWeights)))
    return fail(MCM_ERR_INVALID_ARGUMENT, "sensor arrays missing");
  const int64_t L = in->nx * in->ny * in->nz;
  for (int64_t k = 0; k < L; ++k)
    if (in->M[k] >= in->nM) return fail(MCM_ERR_INVALID_ARGUMENT, "P.M holds a medium index outside 0..nM-1");
  std::vector<long long> sidx((size_t)in->nSensors);
  for (int64_t s = 0; s < in->nSensors; ++s) {
    const double v = in->tempSensorCornerIdxs[s];
    const long long k = (long long)v;
    // the 8 interpolation corners must lie in the grid
    if (!(v >= 0) || k + 1 + in->nx + in->nx * in->ny >= L) return fail(MCM_ERR_INVALID_ARGUMENT, "sensor corner index out of range");
    sidx[s] = k;
  }
  int rc = use_device(in->GPUdevice);
  if (rc) return rc;
  std::unique_ptr<mcm_heat_plan> P(new mcm_heat_plan());
  P->device = in->GPUdevice;
  P->fp32 = in->precision == MCM_HEAT_FP32;
  P->explicitScheme = in->scheme == MCM_HEAT_EXPLICIT;
  P->nx = (int)in->nx;
  P->ny = (int)in->ny;
  P->nz = (int)in->nz;
  P->nM = (int)in->nM;
  P->L = L;
  P->sinked = in->heatBoundaryType != 0;
  P->calcDamage = in->Omega != nullptr || in->Omega_f64 != nullptr;
  P->nS = in->nSensors;
  P->interrupt = in->isInterruptPending;
  MCM_HIP(hipStreamCreate(&P->stream));
  // default steps per captured graph (0: launch every step, e.g. under a
  // kernel tracer that does not follow graph launches)
  if (const char* e = std::getenv("MCM_HEAT_GRAPH_STEPS")) P->graphSteps = std::max<int64_t>(0, std::atoll(e));
  const size_t rs = rt_size(P.get());
  if ((rc = halloc(P->M, (size_t)L)) || (rc = halloc(P->Q, (size_t)L * 4)) || (rc = halloc(P->c, (size_t)P->nM * P->nM * 3 * rs)) ||
      (rc = halloc(P->logA, (size_t)P->nM * rs)) || (rc = halloc(P->E, (size_t)P->nM * rs)) || (rc = halloc(P->T1, (size_t)L * rs)) ||
      (rc = halloc(P->T2, (size_t)L * rs)) || (rc = halloc(P->B, (size_t)L * rs)) ||
      (rc = halloc(P->Om, (size_t)(P->calcDamage ? L : 1) * rs)) || (rc = halloc(P->maxKey, (size_t)P->nM * 8)) ||
      (rc = halloc(P->sIdx, (size_t)std::max<int64_t>(P->nS, 1) * 8)) || (rc = halloc(P->sW, (size_t)std::max<int64_t>(P->nS, 1) * 3 * rs)) ||
      (rc = halloc(P->stage32, (size_t)L * 4)) || (rc = halloc(P->stage64, (size_t)L * 8)))
    return rc;
  hipStream_t s = P->stream;
  MCM_HIP(hipMemcpyAsync(P->M.p, in->M, (size_t)L, hipMemcpyHostToDevice, s));
  MCM_HIP(hipMemcpyAsync(P->Q.p, in->dTdt_abs, (size_t)L * 4, hipMemcpyHostToDevice, s));
  // per-medium constants in the working precision (the reference casts
  // log(A) and E to float, :711-718)
  const int nM = P->nM;
  std::vector<double> c64((size_t)nM * nM * 3), la64(nM), e64(nM), w64((size_t)std::max<int64_t>(P->nS, 1) * 3);
  std::vector<float> c32(c64.size()), la32(nM), e32(nM), w32(w64.size());
  const std::vector<float> coefs = used_coefficients(in);
  for (size_t k = 0; k < c64.size(); ++k) {
    c64[k] = (double)coefs[k];
    c32[k] = coefs[k];
  }
  for (int m = 0; m < nM; ++m) {
    la64[m] = std::log(in->A[m]);
    la32[m] = (float)std::log(in->A[m]);
    e64[m] = in->E[m];
    e32[m] = (float)in->E[m];
  }
  for (int64_t k = 0; k < P->nS * 3; ++k) {
    w64[k] = in->tempSensorInterpWeights[k];
    w32[k] = (float)in->tempSensorInterpWeights[k];
  }
  if (P->fp32) {
    MCM_HIP(hipMemcpyAsync(P->c.p, c32.data(), c32.size() * 4, hipMemcpyHostToDevice, s));
    MCM_HIP(hipMemcpyAsync(P->logA.p, la32.data(), nM * 4, hipMemcpyHostToDevice, s));
    MCM_HIP(hipMemcpyAsync(P->E.p, e32.data(), nM * 4, hipMemcpyHostToDevice, s));
    MCM_HIP(hipMemcpyAsync(P->sW.p, w32.data(), w32.size() * 4, hipMemcpyHostToDevice, s));
    P->constR = (double)8.3144598f;   // finiteElementHeatPropagator.c:86-87
    P->constC = (double)273.15f;
  } else {
    MCM_HIP(hipMemcpyAsync(P->c.p, c64.data(), c64.size() * 8, hipMemcpyHostToDevice, s));
    MCM_HIP(hipMemcpyAsync(P->logA.p, la64.data(), nM * 8, hipMemcpyHostToDevice, s));
    MCM_HIP(hipMemcpyAsync(P->E.p, e64.data(), nM * 8, hipMemcpyHostToDevice, s));
    MCM_HIP(hipMemcpyAsync(P->sW.p, w64.data(), w64.size() * 8, hipMemcpyHostToDevice, s));
    P->constR = 8.3144598;
    P->constC = 273.15;
  }
  if (P->nS) MCM_HIP(hipMemcpyAsync(P->sIdx.p, sidx.data(), sidx.size() * 8, hipMemcpyHostToDevice, s));
  hipLaunchKernelGGL(heat_init_keys, dim3(1), dim3(256), 0, s, (unsigned long long*)P->maxKey.p, nM);
  MCM_HIP(hipGetLastError());
  MCM_HIP(hipStreamSynchronize(s));
  rc = P->fp32 ? upload_state<float>(P.get(), in) : upload_state<double>(P.get(), in);
  if (rc) return rc;
  if ((rc = ensure_sensor_capacity(P.get(), std::max<int64_t>(in->steps, 1) + 1))) return rc;
  if (P->explicitScheme && (rc = P->fp32 ? tune_explicit<float>(P.get(), in->steps) : tune_explicit<double>(P.get(), in->steps))) return rc;
  MCM_HIP(hipStreamSynchronize(s));
  *out = P.release();
  return MCM_OK;
}

int mcm_heat_plan_advance(mcm_heat_plan* P, int64_t steps, double dt, int32_t lightsOn) {
  if (!P) return fail(MCM_ERR_INVALID_ARGUMENT, "null plan");
  if (steps < 0) return fail(MCM_ERR_INVALID_ARGUMENT, "steps must be non-negative");
  MCM_HIP(hipSetDevice(P->device));
  return P->fp32 ? advance<float>(P, steps, dt, lightsOn) : advance<double>(P, steps, dt, lightsOn);
}

int mcm_heat_group_create(mcm_heat_plan* const* plans, int64_t nPlans, mcm_heat_group** out) {
  if (!plans || !out || nPlans < 1) return fail(MCM_ERR_INVALID_ARGUMENT, "a group needs at least one plan");
  *out = nullptr;
  for (int64_t i = 0; i < nPlans; ++i) {
    if (!plans[i]) return fail(MCM_ERR_INVALID_ARGUMENT, "plan %lld is null", (long long)i);
    if (plans[i]->device != plans[0]->device) return fail(MCM_ERR_INVALID_ARGUMENT, "the plans of a group share one device");
    for (int64_t j = 0; j < i; ++j)
      if (plans[j] == plans[i]) return fail(MCM_ERR_INVALID_ARGUMENT, "plan %lld appears twice", (long long)i);
  }
  MCM_HIP(hipSetDevice(plans[0]->device));
  std::unique_ptr<mcm_heat_group> G(new mcm_heat_group);
  G->device = plans[0]->device;
  G->plans.assign(plans, plans + nPlans);
  G->events.assign((size_t)nPlans + 1, nullptr);
  for (hipEvent_t& e : G->events) MCM_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  *out = G.release();
  return MCM_OK;
}

int mcm_heat_group_advance(mcm_heat_group* G, int64_t steps, const double* dt, const int32_t* lightsOn, int64_t stepsPerGraph) {
  if (!G || !dt || !lightsOn) return fail(MCM_ERR_INVALID_ARGUMENT, "null argument");
  if (steps < 0 || stepsPerGraph < 0) return fail(MCM_ERR_INVALID_ARGUMENT, "steps must be non-negative");
  const size_t n = G->plans.size();
  mcm_heat_plan* P0 = G->plans[0];
  MCM_HIP(hipSetDevice(P0->device));
  for (size_t i = 0; i < n; ++i) {
    int rc = ensure_sensor_capacity(G->plans[i], G->plans[i]->stepsDone + steps + 1);
    if (rc) return rc;
    if (G->plans[i]->nS && !G->plans[i]->stepDev.p) MCM_HIP(hipMalloc(&G->plans[i]->stepDev.p, sizeof(long long)));
    if ((rc = ensure_factors(G->plans[i], steps, dt[i]))) return rc;
  }
  const int64_t K = stepsPerGraph & ~(int64_t)1;
  int64_t done = 0;
  if (K >= 2 && steps >= K) {
    mcm_heat_group::Graph* g = nullptr;
    for (mcm_heat_group::Graph& c : G->graphs) {
      bool same = c.steps == K;
      for (size_t i = 0; same && i < n; ++i)
        same = c.dt[i] == dt[i] && c.lightsOn[i] == (lightsOn[i] != 0) && c.T1[i] == G->plans[i]->T1.p && c.sensors[i] == G->plans[i]->sensors.p &&
               c.factored[i] == G->plans[i]->factored(dt[i]);
      if (same) g = &c;
    }
    if (!g) {
      // fork from P0's stream into every plan's stream, K steps per plan, join
      MCM_HIP(hipStreamBeginCapture(P0->stream, hipStreamCaptureModeThreadLocal));
      hipError_t err = hipEventRecord(G->events[0], P0->stream);
      for (size_t i = 1; i < n && err == hipSuccess; ++i) err = hipStreamWaitEvent(G->plans[i]->stream, G->events[0], 0);
      for (size_t i = 0; i < n && err == hipSuccess; ++i) {
        mcm_heat_plan* P = G->plans[i];
        if (P->fp32) enqueue_graph_steps<float>(P, K, dt[i], lightsOn[i] != 0);
        else enqueue_graph_steps<double>(P, K, dt[i], lightsOn[i] != 0);
        err = hipGetLastError();
      }
      for (size_t i = 1; i < n && err == hipSuccess; ++i) {
        err = hipEventRecord(G->events[i + 1], G->plans[i]->stream);
        if (err == hipSuccess) err = hipStreamWaitEvent(P0->stream, G->events[i + 1], 0);
      }
      hipGraph_t graph = nullptr;
      const hipError_t endErr = hipStreamEndCapture(P0->stream, &graph);
      if (err != hipSuccess || endErr != hipSuccess) {
        if (graph) (void)hipGraphDestroy(graph);
        return fail(MCM_ERR_DEVICE, "capturing the group's steps: %s", hipGetErrorString(err != hipSuccess ? err : endErr));
      }
      hipGraphExec_t exec = nullptr;
      err = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
      (void)hipGraphDestroy(graph);
      if (err != hipSuccess) return fail(MCM_ERR_DEVICE, "instantiating the group's step graph: %s", hipGetErrorString(err));
      if (G->graphs.size() >= 4) {
        // replays of the oldest graph end on P0's stream (every branch joins
        // it there): wait for them before the executable graph is destroyed
        MCM_HIP(hipStreamSynchronize(P0->stream));
        (void)hipGraphExecDestroy(G->graphs.front().exec);
        G->graphs.erase(G->graphs.begin());
      }
      mcm_heat_group::Graph c;
      c.exec = exec;
      c.steps = K;
      for (size_t i = 0; i < n; ++i) {
        c.dt.push_back(dt[i]);
        c.lightsOn.push_back(lightsOn[i] != 0);
        c.T1.push_back(G->plans[i]->T1.p);
        c.sensors.push_back(G->plans[i]->sensors.p);
        c.factored.push_back(G->plans[i]->factored(dt[i]));
      }
      G->graphs.push_back(std::move(c));
      g = &G->graphs.back();
    }
    // order the replays after every plan's earlier work; set the step counters
    for (size_t i = 1; i < n; ++i) {
      MCM_HIP(hipEventRecord(G->events[i + 1], G->plans[i]->stream));
      MCM_HIP(hipStreamWaitEvent(P0->stream, G->events[i + 1], 0));
    }
    for (size_t i = 0; i < n; ++i)
      if (G->plans[i]->nS)
        hipLaunchKernelGGL(heat_step_counter, dim3(1), dim3(64), 0, P0->stream, (long long*)G->plans[i]->stepDev.p,
                           (long long)G->plans[i]->stepsDone, 0);
    for (; steps - done >= K; done += K) {
      if (P0->interrupt && P0->interrupt()) {
        P0->interrupted = true;
        break;
      }
      MCM_HIP(hipGraphLaunch(g->exec, P0->stream));
      for (size_t i = 0; i < n; ++i) {
        G->plans[i]->stepsDone += K;
        G->plans[i]->sensorsRecorded = G->plans[i]->stepsDone;
      }
    }
    // later work on any plan's stream follows the replays
    MCM_HIP(hipEventRecord(G->events[0], P0->stream));
    for (size_t i = 1; i < n; ++i) MCM_HIP(hipStreamWaitEvent(G->plans[i]->stream, G->events[0], 0));
    if (P0->interrupted) return MCM_OK;
  }
  for (size_t i = 0; i < n && done < steps; ++i) {
    mcm_heat_plan* P = G->plans[i];
    const int rc = P->fp32 ? advance<float>(P, steps - done, dt[i], lightsOn[i] != 0) : advance<double>(P, steps - done, dt[i], lightsOn[i] != 0);
    if (rc) return rc;
  }
  return MCM_OK;
}

int mcm_heat_group_destroy(mcm_heat_group* G) {
  if (!G) return MCM_OK;
  // the plans may already be gone: wait for the device, not their streams
  (void)hipSetDevice(G->device);
  (void)hipDeviceSynchronize();
  delete G;
  return MCM_OK;
}

int mcm_heat_plan_set_explicit_zrun(mcm_heat_plan* P, int32_t zPlanes) {
  if (!P) return fail(MCM_ERR_INVALID_ARGUMENT, "null plan");
  if (!P->explicitScheme) return fail(MCM_ERR_INVALID_ARGUMENT, "the plan does not use the explicit scheme");
  if (!valid_zrun(zPlanes)) return fail(MCM_ERR_INVALID_ARGUMENT, "z planes per workgroup must be 8, 12, 16, 24 or 32");
  MCM_HIP(hipSetDevice(P->device));
  MCM_HIP(hipStreamSynchronize(P->stream));
  P->drop_graphs();  // captured steps hold the old launch shape
  P->explicitZRun = zPlanes;
  return MCM_OK;
}

int32_t mcm_heat_plan_explicit_zrun(const mcm_heat_plan* P) { return P ? P->explicitZRun : 0; }

int mcm_heat_plan_set_graph_steps(mcm_heat_plan* P, int64_t steps) {
  if (!P) return fail(MCM_ERR_INVALID_ARGUMENT, "null plan");
  if (steps < 0) return fail(MCM_ERR_INVALID_ARGUMENT, "steps per graph must be non-negative");
  MCM_HIP(hipSetDevice(P->device));
  MCM_HIP(hipStreamSynchronize(P->stream));
  P->drop_graphs();
  P->graphSteps = steps;
  return MCM_OK;
}

int mcm_heat_plan_download(mcm_heat_plan* P, mcm_heat_output* out) {
  if (!P || !out) return fail(MCM_ERR_INVALID_ARGUMENT, "null argument");
  MCM_HIP(hipSetDevice(P->device));
  return P->fp32 ? download<float>(P, out) : download<double>(P, out);
}

int mcm_heat_plan_destroy(mcm_heat_plan* P) {
  if (!P) return MCM_OK;
  (void)hipSetDevice(P->device);
  (void)hipStreamSynchronize(P->stream);
  delete P;
  return MCM_OK;
}


int mcm_heat_adjoint_run(const mcm_heat_input* in, const mcm_heat_segment* segments, int64_t nSegments, const uint8_t* targetMask,
                         int64_t checkpointEvery, mcm_heat_adjoint_output* out) {
  return mcm_heat_adjoint_run_within(in, segments, nSegments, targetMask, checkpointEvery,
                                     checkpointEvery > 0 ? MCM_HEAT_ADJOINT_STATES_PERIOD : MCM_HEAT_ADJOINT_STATES, out);
}

int mcm_heat_adjoint_run_within(const mcm_heat_input* in, const mcm_heat_segment* segments, int64_t nSegments, const uint8_t* targetMask,
                                int64_t checkpointEvery, int64_t maxStateBytes, mcm_heat_adjoint_output* out) {
  if (!in || !out) return fail(MCM_ERR_INVALID_ARGUMENT, "null argument");
  if (maxStateBytes < 0) return fail(MCM_ERR_INVALID_ARGUMENT, "maxStateBytes must be non-negative");
  if (in->precision != MCM_HEAT_FP64 || in->scheme != MCM_HEAT_DGADI)
    return fail(MCM_ERR_UNSUPPORTED, "the adjoint is implemented for the FP64 DG-ADI scheme");
  if (!in->Omega && !in->Omega_f64) return fail(MCM_ERR_INVALID_ARGUMENT, "the objective is the damage integral: Omega is required");
  if (nSegments < 0 || (nSegments > 0 && !segments)) return fail(MCM_ERR_INVALID_ARGUMENT, "segments missing");
  std::vector<double> dts;
  std::vector<int> lights;
  if (nSegments == 0) {
    dts.assign((size_t)std::max<int64_t>(in->steps, 0), in->dt);
    lights.assign(dts.size(), in->lightsOn != 0);
  }
  for (int64_t k = 0; k < nSegments; ++k) {
    if (segments[k].steps < 0) return fail(MCM_ERR_INVALID_ARGUMENT, "segment steps must be non-negative");
    dts.insert(dts.end(), (size_t)segments[k].steps, segments[k].dt);
    lights.insert(lights.end(), (size_t)segments[k].steps, segments[k].lightsOn != 0);
  }
  const int64_t N = (int64_t)dts.size();
  mcm_heat_plan* raw = nullptr;
  int rc = mcm_heat_plan_create(in, &raw);
  if (rc) return rc;
  std::unique_ptr<mcm_heat_plan, int (*)(mcm_heat_plan*)> PP(raw, mcm_heat_plan_destroy);
  mcm_heat_plan* P = PP.get();
  const int64_t L = P->L;
  const size_t bytes = (size_t)L * sizeof(double);
  hipStream_t s = P->stream;
  // target voxels: the mask, or every voxel whose medium has E != 0
  std::vector<uint8_t> mask((size_t)L);
  for (int64_t i = 0; i < L; ++i) mask[i] = targetMask ? (targetMask[i] != 0) : (in->E[in->M[i]] != 0);
  HeatBuf dMask, chk, seg, lam, lamN, mu1, mu2, mu3, dQ, s1, s2, dC;
  if ((rc = halloc(dMask, (size_t)L))) return rc;
  MCM_HIP(hipMemcpyAsync(dMask.p, mask.data(), (size_t)L, hipMemcpyHostToDevice, s));
  // The reverse sweep needs the state at every step.  Where all of them fit in
  // maxStateBytes, or are no more than the checkpoints and a segment, they are
  // kept (one segment, no checkpoint), else the steps of one segment at a time
  // are run again from its checkpoint (96 x 80 x 72, 120 steps: 10.7 ms a call
  // kept, 14.8 with three segments of 40 and copies).  What the sweep cannot do
  // without is allocated first.
  const bool gradients = out->dJ_dQ || out->dJ_dT0 || out->dJ_dc;
  const int nBins = P->nM * P->nM * 3;
  if (gradients && ((rc = halloc(lam, bytes)) || (rc = halloc(lamN, bytes)) || (rc = halloc(mu1, bytes)) || (rc = halloc(mu2, bytes)) ||
                    (rc = halloc(mu3, bytes)) || (rc = halloc(dQ, bytes))))
    return rc;
  // the step's intermediate states and the coefficient sums
  if (out->dJ_dc && ((rc = halloc(s1, bytes)) || (rc = halloc(s2, bytes)) || (rc = halloc(dC, (size_t)nBins * sizeof(double))))) return rc;
  int64_t C = std::min<int64_t>(checkpointEvery > 0 ? checkpointEvery : 100, std::max<int64_t>(N, 1));
  int64_t nChk = std::max<int64_t>(1, (N + C - 1) / C);
  bool keep = gradients && ((size_t)(N + 1) <= (size_t)maxStateBytes / bytes || N + 1 <= nChk + C + 1);
  if (keep && hipMalloc(&seg.p, (size_t)(N + 1) * bytes) != hipSuccess) {
    (void)hipGetLastError();
    seg.p = nullptr;
    keep = false;
  }
  if (keep) C = std::max<int64_t>(N, 1), nChk = 0;
  else if ((rc = halloc(chk, (size_t)nChk * bytes)) || (gradients && (rc = halloc(seg, (size_t)(C + 1) * bytes)))) return rc;
  auto chkp = [&](int64_t k) { return (double*)chk.p + (size_t)k * L; };
  auto segp = [&](int64_t k) { return (double*)seg.p + (size_t)k * L; };
  // steps n0 .. n1 - 1 from the state in segp(0) into segp(1), segp(2), ...: each
  // step reads and writes the segment in place of the plan's state buffers
  auto run_segment = [&](int64_t n0, int64_t n1) -> int {
    struct Restore {
      mcm_heat_plan* P;
      void *T1, *T2;
      ~Restore() { P->T1.p = T1, P->T2.p = T2; }
    } restore{P, P->T1.p, P->T2.p};
    P->T1.p = segp(0);
    for (int64_t n = n0; n < n1; ++n) {
      double* const to = segp(n - n0 + 1);
      P->T2.p = to;
      if (int e = advance<double>(P, 1, dts[(size_t)n], lights[(size_t)n])) return e;
      if (P->T1.p != to) {  // interrupted: the state stays
        MCM_HIP(hipMemcpyAsync(to, P->T1.p, bytes, hipMemcpyDeviceToDevice, s));
        P->T1.p = to;
      }
    }
    return MCM_OK;
  };
  if (keep) {
    MCM_HIP(hipMemcpyAsync(segp(0), P->T1.p, bytes, hipMemcpyDeviceToDevice, s));
    if ((rc = run_segment(0, N))) return rc;
  } else {
    // forward pass with checkpoints every C steps
    for (int64_t n = 0; n < N; ++n) {
      if (n % C == 0) MCM_HIP(hipMemcpyAsync(chkp(n / C), P->T1.p, bytes, hipMemcpyDeviceToDevice, s));
      if ((rc = advance<double>(P, 1, dts[(size_t)n], lights[(size_t)n]))) return rc;
    }
    if (N == 0) MCM_HIP(hipMemcpyAsync(chkp(0), P->T1.p, bytes, hipMemcpyDeviceToDevice, s));
  }
  std::vector<double> om((size_t)L);
  MCM_HIP(hipMemcpyAsync(om.data(), P->Om.p, bytes, hipMemcpyDeviceToHost, s));
  MCM_HIP(hipStreamSynchronize(s));
  double J = 0;
  for (int64_t i = 0; i < L; ++i)
    if (mask[i]) J += om[i];
  out->J = J;
  if (out->Omega_f64) std::memcpy(out->Omega_f64, om.data(), bytes);
  if (!gradients) return MCM_OK;
  if (P->nz > 65535) return fail(MCM_ERR_UNSUPPORTED, "heat adjoint: nz > 65535 z planes");
  // reverse sweep, one checkpoint segment at a time
  if (out->dJ_dc) MCM_HIP(hipMemsetAsync(dC.p, 0, (size_t)nBins * sizeof(double), s));
  MCM_HIP(hipMemsetAsync(lam.p, 0, bytes, s));
  MCM_HIP(hipMemsetAsync(dQ.p, 0, bytes, s));
  const int tpb = kHeatTPB;
  const unsigned gv = (unsigned)((L + tpb - 1) / tpb);
  const unsigned gx = (unsigned)(((int64_t)P->ny * P->nz + tpb - 1) / tpb);
  const unsigned gy = (unsigned)(((int64_t)P->nx * P->nz + tpb - 1) / tpb);
  const unsigned gz = (unsigned)(((int64_t)P->nx * P->ny + tpb - 1) / tpb);
  for (int64_t k = (N + C - 1) / C - 1; k >= 0; --k) {
    const int64_t s0 = k * C, e0 = std::min(N, s0 + C);
    if (!keep) {
      MCM_HIP(hipMemcpyAsync(segp(0), chkp(k), bytes, hipMemcpyDeviceToDevice, s));
      if ((rc = run_segment(s0, e0))) return rc;
    }
    for (int64_t n = e0 - 1; n >= s0; --n) {
      HeatArgs<double> a = make_args<double>(P, dts[(size_t)n], lights[(size_t)n]);
      const double* x0 = segp(n - s0);
      const double* x1 = segp(n - s0 + 1);
      double* B = (double*)P->B.p;
      // (the others' damage is added by the combine of the step after them)
      if (n == e0 - 1)
        hipLaunchKernelGGL(heat_adj_damage, dim3(gv), dim3(tpb), 0, s, a, x0, x1, (const uint8_t*)dMask.p, (double*)lam.p, L);
      const double* xm = n > s0 ? segp(n - s0 - 1) : nullptr;
      const double dtm = n > s0 ? dts[(size_t)n - 1] : 0.0;
      adj_solve<2>(P, a, (const double*)lam.p, (double*)mu3.p, B, gz);
      adj_solve<1>(P, a, (const double*)mu3.p, (double*)mu2.p, B, gy);
      adj_solve<0>(P, a, (const double*)mu2.p, (double*)mu1.p, B, gx);
      const dim3 gc((unsigned)((P->nx * P->ny + tpb - 1) / tpb) * (unsigned)P->nz);
      if (P->nM * P->nM * 3 <= kLdsCoef)
        hipLaunchKernelGGL(heat_adj_combine<true>, gc, dim3(tpb), 0, s, a, (const double*)mu1.p, (const double*)mu2.p,
                           (const double*)mu3.p, x0, x1, (const uint8_t*)dMask.p, (double*)lamN.p, (double*)dQ.p, lights[(size_t)n], xm, dtm);
      else
        hipLaunchKernelGGL(heat_adj_combine<false>, gc, dim3(tpb), 0, s, a, (const double*)mu1.p, (const double*)mu2.p,
                           (const double*)mu3.p, x0, x1, (const uint8_t*)dMask.p, (double*)lamN.p, (double*)dQ.p, lights[(size_t)n], xm, dtm);
      MCM_HIP(hipGetLastError());
      if (out->dJ_dc) {
        const dim3 gp((unsigned)((P->nx * P->ny + tpb - 1) / tpb), (unsigned)P->nz);
        hipLaunchKernelGGL(heat_adj_undo<2>, gp, dim3(tpb), 0, s, a, x1, x0, (double*)s2.p);
        hipLaunchKernelGGL(heat_adj_undo<1>, gp, dim3(tpb), 0, s, a, (const double*)s2.p, x0, (double*)s1.p);
        const unsigned gcoef = (unsigned)std::min<int64_t>((L + tpb - 1) / tpb, 2048);
        if (nBins <= kCoefBins)
          hipLaunchKernelGGL(heat_adj_coef<true>, dim3(gcoef), dim3(tpb), 0, s, a, (const double*)mu1.p, (const double*)mu2.p,
                             (const double*)mu3.p, x0, (const double*)s1.p, (const double*)s2.p, x1, (double*)dC.p);
        else
          hipLaunchKernelGGL(heat_adj_coef<false>, dim3(gcoef), dim3(tpb), 0, s, a, (const double*)mu1.p, (const double*)mu2.p,
                             (const double*)mu3.p, x0, (const double*)s1.p, (const double*)s2.p, x1, (double*)dC.p);
        MCM_HIP(hipGetLastError());
      }
      std::swap(lam.p, lamN.p);
    }
  }
  if (out->dJ_dc) MCM_HIP(hipMemcpyAsync(out->dJ_dc, dC.p, (size_t)nBins * sizeof(double), hipMemcpyDeviceToHost, s));
  if (out->dJ_dQ) MCM_HIP(hipMemcpyAsync(out->dJ_dQ, dQ.p, bytes, hipMemcpyDeviceToHost, s));
  if (out->dJ_dT0) MCM_HIP(hipMemcpyAsync(out->dJ_dT0, lam.p, bytes, hipMemcpyDeviceToHost, s));
  MCM_HIP(hipStreamSynchronize(s));
  return MCM_OK;
}

// The whole MEX call (:688-821).  With steps == 0 the reference returns a
// zero-filled T (the step loop never writes its output array); here the input
// state is returned unchanged.
int mcm_heat_run(const mcm_heat_input* in, mcm_heat_output* out) {
  if (!in || !out) return fail(MCM_ERR_INVALID_ARGUMENT, "null argument");
  mcm_heat_plan* raw = nullptr;
  int rc = mcm_heat_plan_create(in, &raw);
  if (rc) return rc;
  std::unique_ptr<mcm_heat_plan, int (*)(mcm_heat_plan*)> P(raw, mcm_heat_plan_destroy);
  if ((rc = mcm_heat_plan_advance(P.get(), in->steps, in->dt, in->lightsOn))) return rc;
  return mcm_heat_plan_download(P.get(), out);
}

}  // extern "C"
