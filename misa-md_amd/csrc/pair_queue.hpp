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
template <typename T>
__device__ __forceinline__ void ldsAdd(T* p, T v) {
  __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Mixed precision: the sum of the pairs set aside does not depend on the order
// they are added in.  A term, the exact FP64 product t of two FP32 factors, is
// taken apart into a multiple of 2^-32 eV/A and the rest in whole units of
// 2^-56; an FP64 and an integer sum of those parts over a site's 128 offsets
// are exact (for sums below 2^19 eV/A), and the two meet in one rounding at the
// end.  A term loses at most 2^-57 eV/A, less than FP64 additions in order lose
// once a partial sum is above 0.1 eV/A, and keeps the bits of its FP32 factor
// down to 1e-10 eV/A.  (In order instead, each lane over the noted pairs of its
// site, kForceL took 370 to 410 us at 2M atoms against 300: the 58 pairs of one
// atom of another species are then a chain that the other lanes wait for.)
constexpr double kTermHi = 1.5 * 1048576.0;  // 1.5 x 2^20: the last bit of a sum with it is 2^-32
constexpr double kTermLo = 0.09375;          // 1.5 x 2^-4: 2^-56
constexpr double kLoUnit = 1.0 / 72057594037927936.0;
struct Term2 {
  double hi;
  int lo;
};
__device__ __forceinline__ Term2 splitTerm(float d, float fp) {
#pragma clang fp contract(off)
  const double x = static_cast<double>(d), f = static_cast<double>(fp);
  Term2 s;
  s.hi = __fma_rn(x, f, kTermHi) - kTermHi;
  s.lo = __double2loint(__fma_rn(x, f, kTermLo - s.hi));  // the low word of 1.5 x 2^52 + the units
  return s;
}
// A lane's sum.  The FP64 part starts at kTermHi and so rounds every term to
// the grid as it is added (a tie may go the other way than in splitTerm; the
// rest makes up for it).
struct OtherM {
  double a[3] = {kTermHi, kTermHi, kTermHi};
  int lo[3] = {0, 0, 0};
  __device__ __forceinline__ void add(float d0, float d1, float d2, float fp) {
#pragma clang fp contract(off)
    const float d[3] = {d0, d1, d2};
    const double f = static_cast<double>(fp);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const double x = static_cast<double>(d[c]), v = __fma_rn(x, f, a[c]), h = v - a[c];
      a[c] = v;
      lo[c] += __double2loint(__fma_rn(x, f, kTermLo - h));
    }
  }
  __device__ __forceinline__ double hi(int c) const { return a[c] - kTermHi; }
  __device__ __forceinline__ void join(int c, double h, int l) {
    a[c] += h;
    lo[c] += l;
  }
  __device__ __forceinline__ double sum(int c) const { return __fma_rn(static_cast<double>(lo[c]), kLoUnit, hi(c)); }
};

// The queue of one wavefront: pairs as offset << 6 | lane.  Two groups of four
// offsets can add 8 x 64 pairs to the at most 63 left waiting.
constexpr int kQueueM = 576;
struct WaveQueueM {
  uint16_t q[kQueueM];
};
// Sums of the pairs set aside, per component and lane of the wavefront; in
// mixed precision of either part of their terms.
struct WaveSums {
  double s[3][64];
};
struct WaveSumsM {
  double hi[3][64];
  int lo[3][64];
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
