// What a step does per inter atom: density and F', force and the half kicks,
// the first half step.  Shared by the site passes, whose launches carry this
// work along, and by the kernels of a batch.
#pragma once
#include <hip/hip_runtime.h>

#include "device_common.hpp"
#include "inter_common.hpp"
#include "resident.hpp"
#include "site_common.hpp"

namespace misa {
namespace site {

// Per inter atom one wavefront: lane l takes the sites of full-list items
// l - 1, l + 63, l + 127, ... (item -1 is the nearest site itself) and the
// inter atoms in their buckets; the lanes' partial sums then meet in a fixed
// shuffle tree, so the result does not depend on the launch.
__device__ __forceinline__ double waveSum(double v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// atom::interRho (atom.cpp:194-284): lattice (nearest site, full list), same
// bucket without itself, then the buckets of the full list; F' at once.
template <typename T>
__device__ __forceinline__ void interRhoBody(const Geom& G, const Tables<T>& tb, const InterView& iv, CXPtr lx,
                                             const int8_t* __restrict__ ltype, const InterDev& in, int w0,
                                             int wstride) {
  const int nl = static_cast<int>(iv.ctl->n_inter);
  const int ne = nl + static_cast<int>(iv.ctl->n_ghost);
  const FullPlaneOffsets& full = *iv.full;
  const int lane = threadIdx.x & 63;
  for (int i = w0; i < nl; i += wstride) {
    const int64_t n = in.e_slot[i];
    if (!isSubBoxSlot(G, n)) continue;
    const double xi0 = in.x[0][i], xi1 = in.x[1][i], xi2 = in.x[2][i];
    const uint64_t myid = in.id[i];
    const int par = n >= G.plane ? 1 : 0;
    double rho = 0.0;
    for (int k = lane - 1; k < full.n[par]; k += 64) {
      const int64_t j = k < 0 ? n : n + full.off[par][k];
      const int8_t tj = ltype[j];
      if (!isVacant(tj)) {
        const double d0 = xi0 - lx.c[0][j], d1 = xi1 - lx.c[1][j], d2 = xi2 - lx.c[2][j];
        const double r2 = d0 * d0 + d1 * d1 + d2 * d2;
        if (r2 < G.rc2) rho += rhoPair(tb, species(tj), r2);
      }
      forBucket(iv, j, ne, [&](int e) {
        const int src = iv.e_src[e];
        if (k < 0 && e < nl && iv.id[src] == myid) return;  // itself (ghost images carry no id)
        const double d0 = xi0 - iv.e_x[0][e], d1 = xi1 - iv.e_x[1][e], d2 = xi2 - iv.e_x[2][e];
        const double r2 = d0 * d0 + d1 * d1 + d2 * d2;
        if (r2 < G.rc2) rho += rhoPair(tb, species(iv.type[src]), r2);
      });
    }
    rho = waveSum(rho);
    if (lane == 0) {
      in.rho[i] = rho;
      checkRho(iv.ctl, rho, static_cast<double>(tb.rhomax));
      const T dfi = dEmbed(tb, species(in.type[i]), static_cast<T>(rho));
      if constexpr (sizeof(T) == 8)
        in.df64[i] = dfi;
      else
        in.df32[i] = dfi;
    }
  }
}
// atom::interForce (atom.cpp:360-473) for the inter list, then
//   MODE 0: f stored, v += c f                    (secondstep)
//   MODE 1: f stored, v += c f; v += c f; x += dt v (secondstep + next firststep)
//   MODE 2: f stored only                         (first force evaluation)
// An inter atom's position is read here by its own wavefront alone; the others
// see it through the entries (e_x), which the decide rebuilds.
template <typename T, int MODE>
__device__ __forceinline__ void interForceBody(const Geom& G, const Tables<T>& tb, const InterView& iv, CXPtr lx,
                                               const int8_t* __restrict__ ltype, const T* __restrict__ ldf,
                                               int ldfStride, const InterDev& in, const VerletParams& vp, int w0,
                                               int wstride) {
  const int nl = static_cast<int>(iv.ctl->n_inter);
  const int ne = nl + static_cast<int>(iv.ctl->n_ghost);
  const FullPlaneOffsets& full = *iv.full;
  const int lane = threadIdx.x & 63;
  for (int i = w0; i < nl; i += wstride) {
    const int64_t n = in.e_slot[i];
    double f0 = 0, f1 = 0, f2 = 0;
    const int ei = species(in.type[i]);
    if (isSubBoxSlot(G, n)) {
      const double xi0 = in.x[0][i], xi1 = in.x[1][i], xi2 = in.x[2][i];
      const uint64_t myid = in.id[i];
      const T dfi = dfOf<T>(iv, i);
      const int par = n >= G.plane ? 1 : 0;
      for (int k = lane - 1; k < full.n[par]; k += 64) {
        const int64_t j = k < 0 ? n : n + full.off[par][k];
        const int8_t tj = ltype[j];
        {
          const double d0 = xi0 - lx.c[0][j], d1 = xi1 - lx.c[1][j], d2 = xi2 - lx.c[2][j];
          const double r2 = d0 * d0 + d1 * d1 + d2 * d2;
          if (r2 < G.rc2 && !isVacant(tj)) {
            const double fp = static_cast<double>(pairForce(tb, ei, species(tj), r2, dfi, ldf[j * ldfStride]));
            f0 += d0 * fp;
            f1 += d1 * fp;
            f2 += d2 * fp;
          }
        }
        forBucket(iv, j, ne, [&](int e) {
          const int src = iv.e_src[e];
          if (k < 0 && e < nl && iv.id[src] == myid) return;
          const double d0 = xi0 - iv.e_x[0][e], d1 = xi1 - iv.e_x[1][e], d2 = xi2 - iv.e_x[2][e];
          const double r2 = d0 * d0 + d1 * d1 + d2 * d2;
          if (r2 < G.rc2) {
            const double fp =
                static_cast<double>(pairForce(tb, ei, species(iv.type[src]), r2, dfi, dfOf<T>(iv, src)));
            f0 += d0 * fp;
            f1 += d1 * fp;
            f2 += d2 * fp;
          }
        });
      }
      f0 = waveSum(f0);
      f1 = waveSum(f1);
      f2 = waveSum(f2);
    }
    if (lane == 0) {
      checkFinite(iv.ctl, f0, f1, f2);
      in.f[0][i] = f0;
      in.f[1][i] = f1;
      in.f[2][i] = f2;
      if (MODE != 2) {  // each product and sum rounded separately (newton_motion.cpp:46-77)
#pragma clang fp contract(off)
        const StepDt sd = stepDt(vp, ei);
        const double f[3] = {f0, f1, f2};
#pragma unroll
        for (int d = 0; d < 3; d++) {
          double v = in.v[d][i] + sd.c * f[d];
          if (MODE == 1) {
            v = v + sd.c * f[d];
            in.x[d][i] += sd.dt * v;
          }
          in.v[d][i] = v;
        }
      }
    }
  }
}
// NewtonMotion::firststep for the inter list (newton_motion.cpp:46-54).
__device__ __forceinline__ void interFirstBody(const InterDev& in, const Ctl* ctl, const VerletParams& vp, int i0,
                                               int istride) {
#pragma clang fp contract(off)  // the half kick and drift round as newton_motion.cpp does
  const int nl = static_cast<int>(ctl->n_inter);
  for (int i = i0; i < nl; i += istride) {
    const StepDt sd = stepDt(vp, species(in.type[i]));
    const double c = sd.c;
    for (int d = 0; d < 3; d++) {
      const double v = in.v[d][i] + c * in.f[d][i];
      in.v[d][i] = v;
      in.x[d][i] += sd.dt * v;
    }
  }
}
}  // namespace site
}  // namespace misa
