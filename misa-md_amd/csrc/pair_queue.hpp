// Pairs set aside by the LDS force passes, and the sums they go to.
//
// A persistent block holds the spline segments of the majority species' pairs
// in LDS.  The other pairs (a Cu or Ni atom on either side, or a distance
// below the first knot held) are a few per cent in a dilute alloy, but nearly
// every offset of a wavefront meets one, and a masked gather of their segments
// costs a load slot of the texture units whether one lane or 64 take part
// (FP64: 320 of the pass's 445 loads per 64 sites; now 190).  So
// a wavefront only notes such a pair (offset and lane, one LDS word) and works
// the noted pairs off 64 at a time with full wavefronts: each lane gathers the
// records and segments of one noted pair and adds its terms to the sums of the
// pair's own site in LDS.
//
// Which pairs are set aside depends on the species and on the knot alone, and
// every force pass (with LDS or without, alone or in a batch) keeps their sum
// apart and adds it to the site's force in the same way, so that all passes
// give the same bits.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace misa {
namespace site {

__device__ __forceinline__ int laneRank(uint64_t lanes) {  // set bits of `lanes` below this lane
  return static_cast<int>(__builtin_amdgcn_mbcnt_hi(
      static_cast<uint32_t>(lanes >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(lanes), 0u)));
}
__device__ __forceinline__ int laneGet(int v, int src) { return __builtin_amdgcn_ds_bpermute(src << 2, v); }
__device__ __forceinline__ float laneGet(float v, int src) {
  return __int_as_float(laneGet(__float_as_int(v), src));
}
__device__ __forceinline__ double laneGet(double v, int src) {
  return __hiloint2double(laneGet(__double2hiint(v), src), laneGet(__double2loint(v), src));
}
// Orders a wavefront's LDS writes before its own later reads by other lanes.
__device__ __forceinline__ void waveLdsFence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}
__device__ __forceinline__ void ldsAdd(double* p, double v) {
  __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Mixed precision: the terms of the pairs set aside, as FP64 products of the
// FP32 factors rounded to multiples of 2^-36 eV/A (1.5e-11, far below the
// FP32 factors' own rounding), so that their FP64 sums are exact (up to
// 2^17 eV/A) and do not depend on the order they are added in.
constexpr double kTermGrid = 1.5 * 65536.0;
__device__ __forceinline__ double gridTerm(float d, float fp) {
#pragma clang fp contract(off)
  const double t = static_cast<double>(d) * static_cast<double>(fp);
  return (t + kTermGrid) - kTermGrid;
}
struct OtherM {
  double x = 0, y = 0, z = 0;
  __device__ __forceinline__ void add(float d0, float d1, float d2, float fp) {
    x += gridTerm(d0, fp);
    y += gridTerm(d1, fp);
    z += gridTerm(d2, fp);
  }
};

// The queue of one wavefront: pairs as offset << 6 | lane.  Two groups of four
// offsets can add 8 x 64 pairs to the at most 63 left waiting.
constexpr int kQueueM = 576;
struct WaveQueueM {
  uint16_t q[kQueueM];
};
// Sums of the pairs set aside, per component and lane of the wavefront.
struct WaveSums {
  double s[3][64];
};

// FP64: the sums of the pairs set aside run over the offsets in order, one
// range of 32 offsets after the other, so the queue is worked off in order
// and at the end of each range.  A pair carries its rank among its site's
// pairs in the range: the pairs of one rank belong to different sites and are
// added together, rank after rank.
template <int U>  // offsets a group: U x 64 pairs on top of at most 63 waiting
struct WaveQueueD {
  uint16_t q[64 * (U + 1)];  // rank << 11 | offset in its range << 6 | lane
};
// The pairs still waiting after the first 64 were worked off move to the
// front, in order.
template <int U>
__device__ __forceinline__ void shiftQueueD(WaveQueueD<U>& wq, int lane) {
  uint16_t e[U];
#pragma unroll
  for (int u = 0; u < U; ++u) e[u] = wq.q[64 * (u + 1) + lane];
  waveLdsFence();
#pragma unroll
  for (int u = 0; u < U; ++u) wq.q[64 * u + lane] = e[u];
  waveLdsFence();
}

}  // namespace site
}  // namespace misa
