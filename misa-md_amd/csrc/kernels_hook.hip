// Hook-mode kernels: the reference's accelerator hooks hip_eam_rho_calc,
// hip_eam_df_calc and hip_eam_force_calc (src/arch/arch_imp.h:27-31) on a
// device copy of the host AtomList array (104-byte AtomElement slots,
// ghost-extended, doubled x index).
//
// A site's neighbours sit 104 bytes and more apart in that array, so that a
// wavefront's read of one field touches a cache line a lane.  kHookPack first
// takes what a sum needs out of it into 16-byte halves {x, y} and {z, w} per
// parity-plane slot (handle scratch), and the sums read those: 64 neighbours
// in two coalesced loads (54 000 cells: density 217 -> 37 us, force 188 -> 54,
// packing 7 each).  The w holds the species for the density sum; for the force
// sum it holds the caller's F' whole, and the species come as a byte each.
// Four wavefronts share 64 sites, each with a quarter of the
// reference's full offset list (NeighbourIndex even/odd,
// neighbour_index.inl:13-76), since a hook's boxes have too few sites to hide
// the round trips of 228 offsets behind other wavefronts; the quarters' sums
// join in list order.  Every lane's sum is complete: rho and f of the sub-box
// slots come out final and the ghost slots keep the zeros atom::clearForce
// left, so the reference's reverse halos (rho_packer.cpp, force_packer.cpp)
// that follow the hooks add nothing.
#include <hip/hip_runtime.h>

#include "buffer_load.hpp"
#include "device_common.hpp"
#include "hook.hpp"
#include "inter_common.hpp"
#include "site_common.hpp"

namespace misa {

namespace {

using namespace site;

constexpr int kHookBlock = 256;
constexpr int kHookParts = kHookBlock / 64;  // wavefronts that share 64 sites
// Neighbours in flight in a wavefront: with four the force sums need 160
// registers and three wavefronts a SIMD (56 us against 52).
constexpr int kHookRhoGroup = 4, kHookForceGroup = 2;

struct HookGeom {
  int n0, n1, n2, g;
  int64_t sx, sy, slots;
  int64_t NX, plane;
  double rc2;
};

// Reference slot r of the doubled-x array -> parity-plane slot.
__device__ __forceinline__ int64_t hookPlaneSlot(const HookGeom& G, int64_t r) {
  const int64_t X = r % G.sx, row = r / G.sx;
  return (X & 1) * G.plane + row * G.NX + (X >> 1);
}

template <bool FORCE>
__global__ __launch_bounds__(kHookBlock) void kHookPack(HookGeom G, const AtomElement* __restrict__ a, Rec64 rec,
                                                        uint8_t* __restrict__ sp) {
  const int64_t r = static_cast<int64_t>(blockIdx.x) * kHookBlock + threadIdx.x;
  if (r >= G.slots) return;
  const AtomElement& e = a[r];
  const int64_t s = hookPlaneSlot(G, r);
  if (e.type < 0) {
    rec.xy[s] = make_double2(kVacantPos64, kVacantPos64);
    rec.zw[s] = make_double2(kVacantPos64, 0.0);
    if (FORCE) sp[s] = 0;
  } else {
    rec.xy[s] = make_double2(e.x[0], e.x[1]);
    rec.zw[s] = make_double2(e.x[2], FORCE ? e.df : packW64(0.0, e.type));
    if (FORCE) sp[s] = static_cast<uint8_t>(e.type);
  }
}

// Sub-box site t of parity p: reference slot r and plane slot s.
__device__ __forceinline__ void hookSite(const HookGeom& G, int p, int64_t t, int64_t& r, int64_t& s) {
  const int64_t cx = t % G.n0, rest = t / G.n0;
  const int64_t row = (rest / G.n1 + G.g) * G.sy + rest % G.n1 + G.g;
  r = row * G.sx + (2 * (cx + G.g) + p);
  s = p * G.plane + row * G.NX + cx + G.g;
}

// Calls group(deltas, nv) for the wavefront's part of the offset list of
// parity p, U at a time (the last group padded with the list's last entry; nv
// counts the real ones).
template <int U, typename Group>
__device__ __forceinline__ void forHookPart(const FullPlaneOffsets& full, int p, int part, Group group) {
  const int n = scalarRead(&full.n[p]);
  const int k0 = n * part / kHookParts, k1 = n * (part + 1) / kHookParts;
  for (int k = k0; k < k1; k += U) {
    int32_t o[U];
#pragma unroll
    for (int u = 0; u < U; ++u) o[u] = scalarRead(&full.off[p][min(k + u, n - 1)]);
    group(o, min(U, k1 - k));
  }
}

__global__ __launch_bounds__(kHookBlock) void kHookRho(HookGeom G, const FullPlaneOffsets* __restrict__ full,
                                                       Tables<double> tb, Rec64 rec, AtomElement* __restrict__ a) {
  __shared__ double sums[kHookParts][64];
  const int p = blockIdx.y;
  const int part = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int64_t nsub = static_cast<int64_t>(G.n0) * G.n1 * G.n2;
  const int64_t t = static_cast<int64_t>(blockIdx.x) * 64 + lane;
  int64_t r, s;
  hookSite(G, p, t < nsub ? t : nsub - 1, r, s);
  double2 xy = rec.xy[s], zw = rec.zw[s];
  if (a[r].type < 0) xy.x = xy.y = zw.x = kNoAtom;  // out of reach of the vacancies' records too
  double rho = 0.0;
  forHookPart<kHookRhoGroup>(*full, p, part, [&](const int32_t (&o)[kHookRhoGroup], int nv) {
    double2 nxy[kHookRhoGroup], nzw[kHookRhoGroup];
#pragma unroll
    for (int u = 0; u < kHookRhoGroup; ++u) {
      nxy[u] = rec.xy[s + o[u]];
      nzw[u] = rec.zw[s + o[u]];
    }
    bool in[kHookRhoGroup];
    double q[kHookRhoGroup], c[kHookRhoGroup][kRhoRec];
#pragma unroll
    for (int u = 0; u < kHookRhoGroup; ++u) {
      const double d0 = xy.x - nxy[u].x, d1 = xy.y - nxy[u].y, d2 = zw.x - nzw[u].x;
      const double r2 = d0 * d0 + d1 * d1 + d2 * d2;
      in[u] = u < nv && r2 < G.rc2;
      if (in[u]) {
        const double rr = r2 > 0.0 ? r2 * rsqrtRefined(r2) : 0.0;
        const int m = knotOf(rr, tb.rdr, tb.nr, false, q[u]);
        const double2* k = reinterpret_cast<const double2*>(
            tb.rhoV + (static_cast<int64_t>(recSpecies64(nzw[u].y)) * tb.nr + m) * kRhoRec);
        const double2 k0 = k[0], k1 = k[1];
        c[u][0] = k0.x;
        c[u][1] = k0.y;
        c[u][2] = k1.x;
        c[u][3] = k1.y;
      }
    }
#pragma unroll
    for (int u = 0; u < kHookRhoGroup; ++u)
      if (in[u]) rho += ((c[u][0] * q[u] + c[u][1]) * q[u] + c[u][2]) * q[u] + c[u][3];
  });
  sums[part][lane] = rho;
  __syncthreads();
  if (part != 0 || t >= nsub || a[r].type < 0) return;
  double sum = 0.0;
#pragma unroll
  for (int w = 0; w < kHookParts; ++w) sum += sums[w][lane];
  a[r].rho += sum;
}

__global__ __launch_bounds__(kHookBlock) void kHookDf(HookGeom G, Tables<double> tb, AtomElement* __restrict__ a) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * kHookBlock + threadIdx.x;
  if (t >= static_cast<int64_t>(G.n0) * G.n1 * G.n2) return;
  int64_t r, s;
  hookSite(G, blockIdx.y, t, r, s);
  if (a[r].type < 0) return;
  a[r].df = dEmbed(tb, a[r].type, a[r].rho);
}

__global__ __launch_bounds__(kHookBlock) void kHookForce(HookGeom G, const FullPlaneOffsets* __restrict__ full,
                                                         Tables<double> tb, Rec64 rec,
                                                         const uint8_t* __restrict__ sp,
                                                         AtomElement* __restrict__ a) {
  __shared__ double sums[kHookParts][3][64];
  const int p = blockIdx.y;
  const int part = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int64_t nsub = static_cast<int64_t>(G.n0) * G.n1 * G.n2;
  const int64_t t = static_cast<int64_t>(blockIdx.x) * 64 + lane;
  int64_t r, s;
  hookSite(G, p, t < nsub ? t : nsub - 1, r, s);
  double2 xy = rec.xy[s], zw = rec.zw[s];
  if (a[r].type < 0) xy.x = xy.y = zw.x = kNoAtom;  // out of reach of the vacancies' records too
  const int ei = sp[s];
  const double dfi = a[r].df;
  double f0 = 0, f1 = 0, f2 = 0;
  forHookPart<kHookForceGroup>(*full, p, part, [&](const int32_t (&o)[kHookForceGroup], int nv) {
    double2 nxy[kHookForceGroup], nzw[kHookForceGroup];
    int nsp[kHookForceGroup];
#pragma unroll
    for (int u = 0; u < kHookForceGroup; ++u) {
      nxy[u] = rec.xy[s + o[u]];
      nzw[u] = rec.zw[s + o[u]];
      nsp[u] = sp[s + o[u]];
    }
    bool in[kHookForceGroup];
    double q[kHookForceGroup], ri[kHookForceGroup];
    double2 c[kHookForceGroup][4], ci[kHookForceGroup][2];  // r*phi c3..c6, rho_j c3..c6; rho_i c3..c6
#pragma unroll
    for (int u = 0; u < kHookForceGroup; ++u) {
      nxy[u].x = xy.x - nxy[u].x;
      nxy[u].y = xy.y - nxy[u].y;
      nzw[u].x = zw.x - nzw[u].x;
      const double r2 = nxy[u].x * nxy[u].x + nxy[u].y * nxy[u].y + nzw[u].x * nzw[u].x;
      in[u] = u < nv && r2 < G.rc2;
      if (in[u]) {
        ri[u] = rsqrtRefined(r2);
        const int m = knotOf(r2 > 0.0 ? r2 * ri[u] : 0.0, tb.rdr, tb.nr, false, q[u]);
        const int ej = nsp[u];
        const double2* k = reinterpret_cast<const double2*>(
            tb.pairF + (static_cast<int64_t>(ei * 3 + ej) * tb.nr + m) * kPairRec);
#pragma unroll
        for (int w = 0; w < 4; ++w) c[u][w] = k[w];
        ci[u][0] = c[u][2];
        ci[u][1] = c[u][3];
        if (ej != ei) {
          const double2* ki =
              reinterpret_cast<const double2*>(tb.rhoV + (static_cast<int64_t>(ei) * tb.nr + m) * kRhoRec);
          ci[u][0] = ki[0];
          ci[u][1] = ki[1];
        }
      }
    }
#pragma unroll
    for (int u = 0; u < kHookForceGroup; ++u)
      if (in[u]) {
        const double fp = pairFpD(q[u], ri[u], c[u][0].x, c[u][0].y, c[u][1].x, c[u][1].y, c[u][2].x, c[u][2].y,
                                  c[u][3].x, ci[u][0].x, ci[u][0].y, ci[u][1].x, dfi, nzw[u].y, tb.rdr);
        f0 = fma(nxy[u].x, fp, f0);
        f1 = fma(nxy[u].y, fp, f1);
        f2 = fma(nzw[u].x, fp, f2);
      }
  });
  sums[part][0][lane] = f0;
  sums[part][1][lane] = f1;
  sums[part][2][lane] = f2;
  __syncthreads();
  if (part != 0 || t >= nsub || a[r].type < 0) return;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    double sum = 0.0;
#pragma unroll
    for (int w = 0; w < kHookParts; ++w) sum += sums[w][k][lane];
    a[r].f[k] += sum;
  }
}

HookGeom hookGeom(const Box& b, double rc) {
  HookGeom G;
  G.n0 = static_cast<int>(b.n[0]);
  G.n1 = static_cast<int>(b.n[1]);
  G.n2 = static_cast<int>(b.n[2]);
  G.g = b.g;
  G.sx = b.sx;
  G.sy = b.sy;
  G.slots = b.slots();
  G.NX = b.n[0] + 2 * b.g;
  G.plane = G.slots / 2;
  G.rc2 = rc * rc;
  return G;
}

}  // namespace

void launchHook(int which, const Box& b, double rc, const FullPlaneOffsets* o, const Tables<double>& tb, Rec64 rec,
                uint8_t* sp, AtomElement* a, hipStream_t st) {
  const HookGeom G = hookGeom(b, rc);
  const int64_t nsub = b.n[0] * b.n[1] * b.n[2];
  if (which == 1) {
    kHookDf<<<dim3(static_cast<unsigned>((nsub + kHookBlock - 1) / kHookBlock), 2, 1), kHookBlock, 0, st>>>(G, tb, a);
    return;
  }
  const dim3 grid(static_cast<unsigned>((nsub + 63) / 64), 2, 1);
  const unsigned packs = static_cast<unsigned>((G.slots + kHookBlock - 1) / kHookBlock);
  if (which == 0) {
    kHookPack<false><<<packs, kHookBlock, 0, st>>>(G, a, rec, sp);
    kHookRho<<<grid, kHookBlock, 0, st>>>(G, o, tb, rec, a);
  } else {
    kHookPack<true><<<packs, kHookBlock, 0, st>>>(G, a, rec, sp);
    kHookForce<<<grid, kHookBlock, 0, st>>>(G, o, tb, rec, sp, a);
  }
}

}  // namespace misa
