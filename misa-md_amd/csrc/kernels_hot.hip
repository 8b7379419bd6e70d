// The two hot passes of the resident EAM step on MI355X (gfx950).
//
//   kRhoDf : rho_i = sum_j rho_{t_j}(r_ij) over the pruned full neighbour list,
//            F'(rho_i) -> df (+ ghost images)   (atom::latRho + latDf + the F'
//            forward halo, atom.cpp:102-149)
//   kForce : f_i = sum_j (x_i - x_j) fpair_ij, then the second half kick and,
//            in the fused mode, the next step's half kick, drift, the lattice
//            part of atom::decide and the position halo (atom::latForce,
//            NewtonMotion, atom::decide; simulation.cpp:164-194)
//
// Each in three forms that give the same bits: four wavefronts to 64 sites in
// boxes of few sites (kRhoDfP, kForceP), a wavefront each (kRhoDf, kForce), and
// persistent blocks with the majority species' segments in LDS (kRhoDL,
// kForceDL); the mixed ones carry an M (kForceL is the mixed LDS pass).  The
// inter atoms' density and force ride in the same launches.
//
// One thread per site.  A full list (each lane owns its site's sums) replaces
// the reference's half list with ghost partials and reverse halos: no atomics,
// deterministic sums.  The list keeps the reference offsets whose ideal
// separation is below rc + 0.4a (+0.01a): a lattice atom normally stays within
// 0.2a of its site (decide() turns it into an inter atom otherwise), so every
// dropped offset is beyond the cutoff for such pairs.  The exception is an
// inter atom that has just refilled a vacancy anywhere in its Wigner-Seitz
// cell: the sites within its full neighbourhood carry kWide and also visit
// the dropped offsets, so the visited pair set is always the reference's.
//
// Memory access: every lane of a wavefront reads neighbour k at the same slot
// delta, so x, type and F' are fetched with buffer loads whose per-lane
// offset (site * size) is fixed for the whole loop and whose scalar offset is
// the (shifted, non-negative) delta: no per-neighbour address arithmetic.
// Neighbours are taken in groups of U: the group's position and type loads
// are all issued before the first distance test, and the spline records of
// the in-cutoff pairs are all issued before the first pair term, so a wave
// keeps U gathers in flight instead of waiting on each neighbour in turn.
// Spline records are packed per knot: the density value cubic (4 values) per
// species for the rho pass, and per ordered species pair the value cubics of
// r*phi and of the neighbour's density (8 values) for the force pass; the
// derivatives are taken from the value cubics, and the centre's density
// cubic is fetched separately only for unlike pairs.
#include <hip/hip_runtime.h>

#include <cmath>
#include <vector>

#include "device_common.hpp"
#include "inter_common.hpp"
#include "inter_step.hpp"
#include "resident.hpp"
#include "site_common.hpp"
#include "buffer_load.hpp"
#include "mixed_site.hpp"

namespace misa {

namespace {

using namespace site;

__device__ __forceinline__ double rsqT(double x) { return rsqrtRefined(x); }

// |x_i - x_j|^2 in FP64 with one fixed rounding, so that the density and
// force passes agree on which pairs are within the cutoff.
__device__ __forceinline__ double dist2D(double d0, double d1, double d2) {
  return __fma_rn(d2, d2, __fma_rn(d1, d1, __dmul_rn(d0, d0)));
}

// Index of the wavefront among those of block b and its predecessors, in a
// scalar register (threadIdx.x >> 6 is the same in every lane of a wavefront).
__device__ __forceinline__ uint32_t waveId(uint32_t b) {
  return b * (kBlock / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
}

// The site passes carry the inter atoms' work of the same pass along, in their
// first blocks (a multiple of 8, so that the others keep their XCD): neither
// part reads what the other writes, and a launch of its own for a list that is
// mostly empty costs 2 to 5 us.  A wavefront works one atom off after the
// other, and a cascade's inter atoms grow with the box: as many blocks as the
// site grid has, 64 to 256.  64 everywhere are too few wavefronts for thousands
// (93 000 atoms FP64: 4 000 inter atoms 766 -> 603 us a step with 256, 12 000 3174
// -> 2481; 755 and 2689 in launches of their own); 256 everywhere cost 2 000 atoms
// at rest 0.5 us a pass.
__host__ __device__ inline uint32_t frontBlocks(const Geom& G) {
  const uint32_t n = static_cast<uint32_t>(16 * G.W.bpx);
  return n < 64u ? 64u : n > 256u ? 256u : n;
}
__device__ __forceinline__ int frontWave() {
  return static_cast<int>(blockIdx.x * (kBlock / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6));
}
__device__ __forceinline__ int frontWaves(const Geom& G) { return static_cast<int>(frontBlocks(G) * (kBlock / 64)); }
// A wavefront-uniform 64-bit value moved to scalar registers.
__device__ __forceinline__ uint64_t uniform64(uint64_t v) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v));
  const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v >> 32));
  return (static_cast<uint64_t>(hi) << 32) | lo;
}

// The lane's record address, or for a lane without an atom that of the
// wavefront's first atom (same parity), from where every offset is readable.
// Called by whole wavefronts.
__device__ __forceinline__ uint32_t addressOfLives(uint32_t o16, bool live, uint64_t lives) {
  const uint32_t first = static_cast<uint32_t>(
      __builtin_amdgcn_readlane(static_cast<int>(o16), __builtin_ctzll(lives)));
  return live ? o16 : first;
}

// Calls visit(ks, nv) for the set bits of (b0, b1) in increasing order, U at
// a time, then one at a time (nv = U or 1; ks holds the offsets).
template <int U, typename Visit>
__device__ __forceinline__ void forMaskGroups(uint64_t b0, uint64_t b1, Visit visit) {
  int left = __builtin_popcountll(b0) + __builtin_popcountll(b1);
  for (; left > 0;) {
    const int V = left >= U ? U : 1;
    int ks[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (u < V) {
        if (b0) {
          ks[u] = __builtin_ctzll(b0);
          b0 &= b0 - 1;
        } else {
          ks[u] = 64 + __builtin_ctzll(b1);
          b1 &= b1 - 1;
        }
      } else {
        ks[u] = 0;
      }
    }
    visit(ks, V);
    left -= V;
  }
}

// Calls visit(ks, act) for the set bits of (b0, b1) in increasing order,
// always U at a time: in the last group the entries past the last bit
// (act[u] false) repeat the last offset, and the caller makes them add
// nothing.  One shape of group keeps the gathers of a group in flight
// together.
template <int U, typename Visit>
__device__ __forceinline__ void forMaskGroupsFull(uint64_t b0, uint64_t b1, Visit visit) {
  int k = 0;
  while (b0 | b1) {
    int ks[U];
    bool act[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      act[u] = (b0 | b1) != 0;
      if (b0) {
        k = __builtin_ctzll(b0);
        b0 &= b0 - 1;
      } else if (b1) {
        k = 64 + __builtin_ctzll(b1);
        b1 &= b1 - 1;
      }
      ks[u] = k;
    }
    visit(ks, act);
  }
}

// Set bit k of the 128-bit offset mask (m0, m1).
__device__ __forceinline__ void setBit(uint64_t& m0, uint64_t& m1, int k) {
  if (k < 64) m0 |= 1ull << k;
  else m1 |= 1ull << (k - 64);
}

// The leader (first gathering lane) writes the wavefront's masks.
__device__ __forceinline__ void writeMasks(bool gathers, uint32_t wv, uint64_t w0, uint64_t w1, uint64_t* wmask,
                                           bool full, uint64_t s0, uint64_t s1, uint64_t* smask) {
  const uint64_t gathered = __ballot(gathers);
  if (!gathered) return;
  const int leader = __builtin_ctzll(gathered);
  const uint64_t a0 = __shfl(w0, leader, 64), a1 = __shfl(w1, leader, 64);
  const uint64_t c0 = __shfl(s0, leader, 64), c1 = __shfl(s1, leader, 64);
  if (static_cast<int>(threadIdx.x & 63) == leader) {
    wmask[2 * wv] = a0;
    wmask[2 * wv + 1] = a1;
    if (full) {
      smask[2 * wv] = c0;
      smask[2 * wv + 1] = c1;
    }
  }
}

// ---------------------------------------------------------------------------
// pass 1: rho and F'
// FP64 and mixed density passes record, per wavefront, the pruned offsets
// within the cutoff for some lane (wmask) for the force pass, which visits
// only those.  A full scan also records the offsets within cutoff + skin
// (smask); while decide finds that no atom can have crossed the skin
// (Ctl::skin_mode) the density pass visits only those: the same pairs in the
// same order, so the sums do not change.
// ---------------------------------------------------------------------------
// What a lane's site needs for the FP64 density sum.
struct RhoSiteD {
  double x0, x1, x2;
  Rsrc rxy, rzw, rtab;  // neighbours' FP64 site records (a vacancy sits far out); the density cubics
  uint32_t o16;
  const uint32_t* sh;
  double rc2, rcs2;
  int mlo;
};
__device__ __forceinline__ double cubicD(double c3, double c4, double c5, double c6, double q) {
  return __fma_rn(__fma_rn(__fma_rn(c3, q, c4), q, c5), q, c6);
}
__device__ __forceinline__ RhoSiteD rhoSiteD(const Geom& G, const LatOffsets& O, const Tables<double>& tb, CXPtr x,
                                             const Rec64& r64, double rcs2, int mlo, int64_t s, int p) {
  return RhoSiteD{x.c[0][s], x.c[1][s], x.c[2][s], rsrcBelow(r64.xy, O.lo), rsrcBelow(r64.zw, O.lo),
                  rsrcAt(reinterpret_cast<uintptr_t>(tb.rhoV)), static_cast<uint32_t>(s) * 16u, O.sh[p], G.rc2, rcs2, mlo};
}
// The densities of V neighbours at offsets ks; sets the bits of the offsets
// within the cutoff for some lane (w) and, on a full scan, within cutoff +
// skin (s).
template <int V>
__device__ __forceinline__ void rhoGroupD(const RhoSiteD& c, const Tables<double>& tb, const int* ks, bool skin,
                                          RangeSum<0>& acc, RangeSum<0>& oacc, uint64_t& w0, uint64_t& w1,
                                          uint64_t& s0, uint64_t& s1) {
  double2 xy[V], zw[V];
#pragma unroll
  for (int u = 0; u < V; ++u) {
    const uint32_t so = c.sh[ks[u]] * 16u;
    xy[u] = ldRec64(c.rxy, c.o16, so);
    zw[u] = ldRec64(c.rzw, c.o16, so);
  }
  bool in[V], held[V];
  double pp[V], rec[V][kRhoRec];
#pragma unroll
  for (int u = 0; u < V; ++u) {
    const double r2 = dist2D(c.x0 - xy[u].x, c.x1 - xy[u].y, c.x2 - zw[u].x);
    in[u] = r2 < c.rc2;
    if (!skin && __ballot(r2 < c.rcs2)) setBit(s0, s1, ks[u]);
    if (__ballot(in[u])) setBit(w0, w1, ks[u]);
    if (in[u]) {
      const int m = knotM(r2 * rsqT(r2), tb.rdr, tb.nr, pp[u]);
      const int ej = recSpecies64(zw[u].y);
      held[u] = heldPair(0, static_cast<uint32_t>(ej), m, c.mlo);
      ldRec<double, kRhoRec>(c.rtab, static_cast<uint32_t>(ej * tb.nr + m) * (kRhoRec * 8u), rec[u]);
    }
  }
#pragma unroll
  for (int u = 0; u < V; ++u) {
    acc.at(ks[u]);
    oacc.at(ks[u]);
    if (in[u]) {
      const double v = cubicD(rec[u][0], rec[u][1], rec[u][2], rec[u][3], pp[u]);
      if (held[u]) acc.part.add(v);
      else oacc.part.add(v);
    }
  }
}
// Calls group(ks, V) over the offsets [k0, k1), or over the set bits of
// (b0, b1) when skin is set, U at a time and then one at a time.
template <int U, typename Group>
__device__ __forceinline__ void forRhoGroups(bool skin, int k0, int k1, uint64_t b0, uint64_t b1, Group group) {
  if (!skin) {
    int ks[U];
    int k = k0;
    for (; k + U <= k1; k += U) {
#pragma unroll
      for (int u = 0; u < U; ++u) ks[u] = k + u;
      group(std::integral_constant<int, U>{}, ks);
    }
    for (; k < k1; ++k) {
      ks[0] = k;
      group(std::integral_constant<int, 1>{}, ks);
    }
  } else {
    forMaskGroups<U>(b0, b1, [&](const int* ks, int nv) {
      if (nv == U) group(std::integral_constant<int, U>{}, ks);
      else group(std::integral_constant<int, 1>{}, ks);
    });
  }
}
// After the lattice sum: the inter atoms and, near a far lattice atom, the
// rest of the full list; then F'(rho), into df and the w of the site's record
// (and of its images' records).
__device__ __forceinline__ void rhoTailD(const Geom& G, int64_t s, int p, int cx, int cy, int cz, int8_t ti,
                                         Sum1<0>& acc, CXPtr x, const int8_t* __restrict__ type,
                                         const Tables<double>& tb, double* __restrict__ df,
                                         double* __restrict__ rho_out, const InterView& iv, const Rec64& r64,
                                         const TailHits* hits = nullptr) {
  double dfi = 0.0, rho = 0.0;
  if (!isVacant(ti)) {
    const double xi0 = x.c[0][s], xi1 = x.c[1][s], xi2 = x.c[2][s];
    if (ti & kNearInter) {  // inter atoms whose nearest site is within the full list (atom.cpp:224-240)
      const int ne = static_cast<int>(iv.ctl->n_inter + iv.ctl->n_ghost);
      const FullPlaneOffsets& full = *iv.full;
      forNearBuckets(iv, full, p, s, ne, hits, [&](int e) {
        const double d0 = xi0 - iv.e_x[0][e], d1 = xi1 - iv.e_x[1][e], d2 = xi2 - iv.e_x[2][e];
        const double r2 = d0 * d0 + d1 * d1 + d2 * d2;
        if (r2 < G.rc2) acc.add(rhoPair(tb, species(iv.type[iv.e_src[e]]), r2));
      });
    }
    if (ti & kWide) {  // full-list offsets beyond the pruned list, near a far lattice atom
      forWideTargets(*iv.full, x.c, type, G.rc2, p, s, ti, xi0, xi1, xi2, hits, [&](int64_t j, int8_t tj) {
        const double d0 = xi0 - x.c[0][j], d1 = xi1 - x.c[1][j], d2 = xi2 - x.c[2][j];
        const double r2 = d0 * d0 + d1 * d1 + d2 * d2;
        if (r2 < G.rc2) acc.add(rhoPair(tb, species(tj), r2));
      });
    }
    rho = acc.value();
    checkRho(iv.ctl, rho, tb.rhomax);
    dfi = dEmbed(tb, species(ti), rho);
  }
  df[s] = dfi;
  double* w64 = reinterpret_cast<double*>(r64.zw) + 1;
  const double wi = packW64(dfi, species(ti));
  if (!isVacant(ti)) w64[2 * s] = wi;
  if (rho_out) rho_out[s] = rho;
  forEachImage(G, p, cx, cy, cz, [&](int64_t q, int, int, int) {
    df[q] = dfi;
    if (rho_out) rho_out[q] = rho;
    if (!isVacant(ti)) w64[2 * q] = wi;
  });
}

// (Two sums, for the neighbours held in LDS elsewhere and for the others, need
// more registers than one: bound to seven wavefronts a SIMD it spills, 580 us
// at 108^3 cells; to five 554, with one sum 538.)
template <int U>
__global__ __launch_bounds__(kBlock, 5) void kRhoDf(Geom G, LatOffsets O, Tables<double> tb, CXPtr x,
                                                 const int8_t* __restrict__ type, double* __restrict__ df,
                                                 double* __restrict__ rho_out, uint64_t* __restrict__ wmask,
                                                 uint64_t* __restrict__ smask, double rcs2, InterView iv,
                                                 InterDev in, Rec64 r64, int mlo) {
  if (blockIdx.x < frontBlocks(G)) {
    interRhoBody<double>(G, tb, iv, x, type, in, frontWave(), frontWaves(G));
    return;
  }
  const uint32_t b = blockIdx.x - frontBlocks(G);
  int64_t s;
  int p, cx, cy, cz;
  if (!siteOfBlock(G, b, threadIdx.x, s, p, cx, cy, cz)) return;
  const int8_t ti = type[s];
  // a wavefront next to a far lattice atom (kWide) scans in full and records its masks afresh
  const bool skin =
      __builtin_amdgcn_readfirstlane(iv.ctl->skin_mode) != 0 && !__ballot(!isVacant(ti) && (ti & kWide));
  const uint32_t wv = waveId(b);
  RangeSum<0> acc, oacc;
  uint64_t w0 = 0, w1 = 0, s0 = 0, s1 = 0;
  if (!isVacant(ti)) {
    const RhoSiteD c = rhoSiteD(G, O, tb, x, r64, rcs2, mlo, s, p);
    forRhoGroups<U>(skin, 0, O.n[p], skin ? uniform64(smask[2 * wv]) : 0, skin ? uniform64(smask[2 * wv + 1]) : 0,
                    [&](auto UC, const int* ks) {
                      rhoGroupD<decltype(UC)::value>(c, tb, ks, skin, acc, oacc, w0, w1, s0, s1);
                    });
  }
  acc.close();
  oacc.close();
  acc.tot.join(oacc.tot);
  writeMasks(!isVacant(ti), wv, w0, w1, wmask, !skin, s0, s1, smask);
  rhoTailD(G, s, p, cx, cy, cz, ti, acc.tot, x, type, tb, df, rho_out, iv, r64);
}

// ---------------------------------------------------------------------------
// Boxes with few sites.  One wavefront's walk over its offsets is a chain of
// some sixteen to thirty groups, each a round trip to the records and one to
// the tables, about 1.5 us a group; when the sites fill only a few wavefronts
// per SIMD nothing hides it (2,000 atoms: kRhoDf 28 us and kForce 40-50 us,
// the same as at 16,000).  There the four wavefronts of a block share 64
// sites, each takes one range of 32 offsets (one word of the mask), and the
// first of them joins the four sums in the order the one-wavefront passes use
// and does what follows the lattice sum.  Same bits, a quarter of the chain.
// ---------------------------------------------------------------------------

// The offsets of range rg of a list of n: [32 rg, min(32 rg + 32, n)), and the
// mask bits of that range.
struct Range {
  int k0, k1;
};
__device__ __forceinline__ Range rangeOf(int rg, int n) { return Range{32 * rg, min(32 * rg + 32, n)}; }
__device__ __forceinline__ void rangeBits(const uint64_t* mask, uint32_t wv, int rg, uint64_t& b0, uint64_t& b1) {
  const uint32_t w = __builtin_amdgcn_readfirstlane(reinterpret_cast<const uint32_t*>(mask)[4 * wv + rg]);
  const uint64_t b = static_cast<uint64_t>(w) << (32 * (rg & 1));
  b0 = rg < 2 ? b : 0;
  b1 = rg < 2 ? 0 : b;
}
// writeMasks for one word of the masks.
__device__ __forceinline__ void writeMaskWord(bool gathers, uint32_t wv, int rg, uint64_t w0, uint64_t w1,
                                              uint64_t* wmask, bool full, uint64_t s0, uint64_t s1,
                                              uint64_t* smask) {
  const uint64_t gathered = __ballot(gathers);
  if (!gathered) return;
  const int leader = __builtin_ctzll(gathered);
  if (static_cast<int>(threadIdx.x & 63) == leader) {
    reinterpret_cast<uint32_t*>(wmask)[4 * wv + rg] = static_cast<uint32_t>((rg < 2 ? w0 : w1) >> (32 * (rg & 1)));
    if (full)
      reinterpret_cast<uint32_t*>(smask)[4 * wv + rg] = static_cast<uint32_t>((rg < 2 ? s0 : s1) >> (32 * (rg & 1)));
  }
}

// The shared site of this thread's wavefront (four wavefronts, the same site a
// lane): block b of a siteGrid launch, thread tl of it.  False without a site;
// ti is then a vacancy's type.
struct SharedSite {
  int64_t s = 0;
  int p = 0, cx = 0, cy = 0, cz = 0;
  uint32_t wv = 0;  // index of the masks
  int rg = 0;       // this wavefront's range
  int8_t ti = kVacant;
  bool site = false;
};
__device__ __forceinline__ SharedSite sharedSite(const Geom& G, const int8_t* __restrict__ type, uint32_t id) {
  SharedSite q;
  uint32_t b, sub;
  sharedUnit(id, b, sub);
  q.rg = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  q.wv = b * (kBlock / 64) + sub;
  q.p = static_cast<int>((b >> 3) & 1u);
  q.site = siteOfBlock(G, b, sub * 64u + (threadIdx.x & 63u), q.s, q.p, q.cx, q.cy, q.cz);
  if (q.site) q.ti = type[q.s];
  return q;
}

// Sums of the four ranges in LDS: what the later three wavefronts hand over.
struct RangeParts {
  double v[3][2][64];
};
template <int ACC>
__device__ __forceinline__ void putPart(RangeParts& r, int rg, const Sum1<ACC>& a) {
  const int lane = static_cast<int>(threadIdx.x & 63u);
  r.v[rg - 1][0][lane] = static_cast<double>(a.s);
  if constexpr (ACC == 1) r.v[rg - 1][1][lane] = static_cast<double>(a.c);
}
template <int ACC>
__device__ __forceinline__ void joinParts(const RangeParts& r, Sum1<ACC>& tot) {
  const int lane = static_cast<int>(threadIdx.x & 63u);
#pragma unroll
  for (int rg = 1; rg < 4; ++rg) {
    Sum1<ACC> a;
    a.s = static_cast<decltype(a.s)>(r.v[rg - 1][0][lane]);
    if constexpr (ACC == 1) a.c = static_cast<float>(r.v[rg - 1][1][lane]);
    tot.join(a);
  }
}

template <int U>
__global__ __launch_bounds__(kBlock) void kRhoDfP(Geom G, LatOffsets O, Tables<double> tb, CXPtr x,
                                                  const int8_t* __restrict__ type, double* __restrict__ df,
                                                  double* __restrict__ rho_out, uint64_t* __restrict__ wmask,
                                                  uint64_t* __restrict__ smask, double rcs2, InterView iv,
                                                  InterDev in, Rec64 r64, int mlo) {
  __shared__ RangeParts parts, oparts;
  __shared__ TailHits hits;
  if (blockIdx.x < frontBlocks(G)) {
    interRhoBody<double>(G, tb, iv, x, type, in, frontWave(), frontWaves(G));
    return;
  }
  const SharedSite q = sharedSite(G, type, blockIdx.x - frontBlocks(G));
  const bool live = !isVacant(q.ti);
  const bool skin = __builtin_amdgcn_readfirstlane(iv.ctl->skin_mode) != 0 && !__ballot(live && (q.ti & kWide));
  RangeSum<0> acc, oacc;
  acc.range = oacc.range = q.rg;
  uint64_t w0 = 0, w1 = 0, s0 = 0, s1 = 0, b0 = 0, b1 = 0;
  if (live) {
    const RhoSiteD c = rhoSiteD(G, O, tb, x, r64, rcs2, mlo, q.s, q.p);
    const Range r = rangeOf(q.rg, O.n[q.p]);
    if (skin) rangeBits(smask, q.wv, q.rg, b0, b1);
    forRhoGroups<U>(skin, r.k0, r.k1, b0, b1, [&](auto UC, const int* ks) {
      rhoGroupD<decltype(UC)::value>(c, tb, ks, skin, acc, oacc, w0, w1, s0, s1);
    });
  }
  writeMaskWord(live, q.wv, q.rg, w0, w1, wmask, !skin, s0, s1, smask);
  if (q.rg > 0) {
    putPart(parts, q.rg, acc.part);
    putPart(oparts, q.rg, oacc.part);
  }
  findTailHits(hits, q.rg, iv, x.c, type, G.rc2, q.p, q.s, q.ti);
  __syncthreads();
  if (q.rg > 0 || !q.site) return;
  acc.close();
  oacc.close();
  joinParts(parts, acc.tot);
  joinParts(oparts, oacc.tot);
  acc.tot.join(oacc.tot);
  rhoTailD(G, q.s, q.p, q.cx, q.cy, q.cz, q.ti, acc.tot, x, type, tb, df, rho_out, iv, r64, &hits);
}

// secondstep (and, fused, the next firststep and decide) of a lattice atom,
// newton_motion.cpp:46-77, with every product and sum rounded separately.
template <int MODE>
__device__ __forceinline__ void verletTail(const Geom& G, int64_t s, int p, int cx, int cy, int cz, int8_t ti,
                                           int ei, double xi0, double xi1, double xi2, double f0, double f1,
                                           double f2, XPtr xn, XPtr v, XPtr f, const uint64_t* __restrict__ id,
                                           const VerletParams& vp, const StageArgs& st, Ctl* ctl,
                                           const Rec64& rn64, unsigned long long& vb, unsigned long long& db) {
#pragma clang fp contract(off)
  const StepDt sd = stepDt(vp, ei);
  const double c = sd.c;
  double v0 = v.c[0][s] + c * f0;
  double v1 = v.c[1][s] + c * f1;
  double v2 = v.c[2][s] + c * f2;
  if (MODE == 2) {
    f.c[0][s] = f0;
    f.c[1][s] = f1;
    f.c[2][s] = f2;
    return;
  }
  if (MODE == 0) {
    f.c[0][s] = f0;
    f.c[1][s] = f1;
    f.c[2][s] = f2;
    v.c[0][s] = v0;
    v.c[1][s] = v1;
    v.c[2][s] = v2;
    vb = speed2Bits(v0, v1, v2);
    return;
  }
  v0 = v0 + c * f0;
  v1 = v1 + c * f1;
  v2 = v2 + c * f2;
  const double y0 = xi0 + sd.dt * v0;
  const double y1 = xi1 + sd.dt * v1;
  const double y2 = xi2 + sd.dt * v2;
  db = speed2Bits(y0 - xi0, y1 - xi1, y2 - xi2);
  if (leftSite(G, p, cx, cy, cz, y0, y1, y2)) {
    stageInter(st, ctl, refIndex(G, p, cx, cy, cz), s, id[s], ti, y0, y1, y2, v0, v1, v2);
    v0 = v1 = v2 = 0.0;
  }
  v.c[0][s] = v0;
  v.c[1][s] = v1;
  v.c[2][s] = v2;
  xn.c[0][s] = y0;
  xn.c[1][s] = y1;
  xn.c[2][s] = y2;
  putRec64(rn64, s, ti, y0, y1, y2);
  forEachImageLoop(G, p, cx, cy, cz, [&](int64_t q, int sx, int sy, int sz) {
    const double q0 = y0 + sx * G.L0, q1 = y1 + sy * G.L1, q2 = y2 + sz * G.L2;
    xn.c[0][q] = q0;
    xn.c[1][q] = q1;
    xn.c[2][q] = q2;
    putRec64(rn64, q, ti, q0, q1, q2);
  });
}

// ---------------------------------------------------------------------------
// pass 2: force and velocity Verlet
//   MODE 0: f stored, v += c f                        (secondstep)
//   MODE 1: v += c f; v += c f; x' = x + dt v; decide  (secondstep + next firststep)
//   MODE 2: f stored only                             (first force evaluation)
// ---------------------------------------------------------------------------
// The FP64 segments of a pair at knot m: rec = the r*phi value cubic c3..c6
// and the neighbour's density cubic c3..c6, reci = the centre's density
// cubic (rec's for a like pair).  With LDS a pair of Fe atoms at a knot from
// mlo on reads them from knD (7 doubles a knot, the density's c6 left out:
// no force or energy term uses it), every other pair from the tables in
// global memory; the values are the same.
template <bool LDS>
__device__ __forceinline__ void pairSegD(Rsrc rtab, Rsrc rtabR, const double* knD, int mlo, uint32_t pairBase,
                                         int nr, int ei, int ej, int m, double (&rec)[kPairRec],
                                         double (&reci)[kRhoRec]) {
  if (LDS && (ei | ej) == 0 && m >= mlo) {
    const double* k = knD + 7 * (m - mlo);
#pragma unroll
    for (int q = 0; q < 7; q++) rec[q] = k[q];
    rec[7] = 0.0;
#pragma unroll
    for (int q = 0; q < kRhoRec; q++) reci[q] = rec[4 + q];
    return;
  }
  ldRec<double, kPairRec>(rtab, (pairBase + static_cast<uint32_t>(ej * nr + m)) * (kPairRec * 8u), rec);
  if (ej != ei) {  // rho_ei differs from rho_ej only for unlike pairs
    ldRec<double, kRhoRec>(rtabR, static_cast<uint32_t>(ei * nr + m) * (kRhoRec * 8u), reci);
  } else {
#pragma unroll
    for (int q = 0; q < kRhoRec; q++) reci[q] = rec[4 + q];
  }
}

// The sums of the FP64 force passes run over four ranges of 32 offsets (the
// 32-bit words of the wavefront's mask): in each range the pairs that the LDS
// pass holds segments for and the others apart (heldPair), each in offset
// order, and the ranges' sums one after the other.
__device__ __forceinline__ uint32_t maskWord(uint64_t m0, uint64_t m1, int r) {
  return static_cast<uint32_t>((r < 2 ? m0 : m1) >> (32 * (r & 1)));
}

struct Force3 {
  double x = 0, y = 0, z = 0;
  __device__ __forceinline__ void add(double d0, double d1, double d2, double fp) {
    x = __fma_rn(d0, fp, x);
    y = __fma_rn(d1, fp, y);
    z = __fma_rn(d2, fp, z);
  }
  __device__ __forceinline__ void add(const Force3& o) {
    x += o.x;
    y += o.y;
    z += o.z;
  }
};

// A vacancy in the FP64 force pass: f = 0 (clearForce, and latForce skips it),
// or in the fused pass its stale position into the next buffers.
template <int MODE>
__device__ __forceinline__ void vacancyForceD(const Geom& G, int64_t s, int p, int cx, int cy, int cz, int8_t ti,
                                              CXPtr x, XPtr xn, XPtr f, const Rec64& rn64) {
  if (MODE != 1) {  // clearForce left 0 there and latForce skips it (atom.cpp:86-100, 311-358)
    f.c[0][s] = 0.0;
    f.c[1][s] = 0.0;
    f.c[2][s] = 0.0;
    return;
  }
  const double xi0 = x.c[0][s], xi1 = x.c[1][s], xi2 = x.c[2][s];
  xn.c[0][s] = xi0;
  xn.c[1][s] = xi1;
  xn.c[2][s] = xi2;
  putRec64(rn64, s, ti, xi0, xi1, xi2);
  forEachImage(G, p, cx, cy, cz, [&](int64_t q, int sx, int sy, int sz) {
    xn.c[0][q] = xi0 + sx * G.L0;
    xn.c[1][q] = xi1 + sy * G.L1;
    xn.c[2][q] = xi2 + sz * G.L2;
    putRec64(rn64, q, ti, xn.c[0][q], xn.c[1][q], xn.c[2][q]);
  });
}

// After the lattice sum of an occupied site: the inter atoms, the full-list
// remainder near far lattice atoms, then the Verlet step.
template <int MODE>
__device__ __forceinline__ void forceTailD(const Geom& G, int64_t s, int p, int cx, int cy, int cz, int8_t ti,
                                           int ei, double dfi, const Force3& lat, double xi0, double xi1, double xi2,
                                           const Tables<double>& tb, CXPtr x, XPtr xn,
                                           const int8_t* __restrict__ type, const double* __restrict__ df, XPtr v,
                                           XPtr f, const uint64_t* __restrict__ id, const VerletParams& vp,
                                           const StageArgs& st, Ctl* ctl, const InterView& iv, const Rec64& rn64,
                                           unsigned long long& vb, unsigned long long& db,
                                           const TailHits* hits = nullptr) {
  Force3 acc = lat;
  if (ti & kNearInter) {  // forces from inter atoms on lattice neighbours (atom.cpp:397-422)
    const int ne = static_cast<int>(iv.ctl->n_inter + iv.ctl->n_ghost);
    const FullPlaneOffsets& full = *iv.full;
    forNearBuckets(iv, full, p, s, ne, hits, [&](int e) {
      const int src = iv.e_src[e];
      const double d0 = xi0 - iv.e_x[0][e], d1 = xi1 - iv.e_x[1][e], d2 = xi2 - iv.e_x[2][e];
      const double r2 = d0 * d0 + d1 * d1 + d2 * d2;
      if (r2 < G.rc2) acc.add(d0, d1, d2, pairForce(tb, ei, species(iv.type[src]), r2, dfi, iv.df64[src]));
    });
  }
  if (ti & kWide) {  // full-list offsets beyond the pruned list, near a far lattice atom
    forWideTargets(*iv.full, x.c, type, G.rc2, p, s, ti, xi0, xi1, xi2, hits, [&](int64_t j, int8_t tj) {
      const double e0 = xi0 - x.c[0][j], e1 = xi1 - x.c[1][j], e2 = xi2 - x.c[2][j];
      const double r2 = e0 * e0 + e1 * e1 + e2 * e2;
      if (r2 < G.rc2) acc.add(e0, e1, e2, pairForce(tb, ei, species(tj), r2, dfi, df[j]));
    });
  }
  checkFinite(ctl, acc.x, acc.y, acc.z);
  verletTail<MODE>(G, s, p, cx, cy, cz, ti, ei, xi0, xi1, xi2, acc.x, acc.y, acc.z, xn, v, f, id, vp, st, ctl, rn64,
                   vb, db);
}

// What a lane's site needs for the FP64 force sum with the segments from the
// tables in global memory.
struct ForceSiteD {
  double x0, x1, x2, dfi;
  int ei;
  Rsrc rxy, rzw, rtab, rtabR;
  uint32_t o16, pairBase;
  const uint32_t* sh;
  double rc2;
  int mlo;
};
__device__ __forceinline__ ForceSiteD forceSiteOf(const Geom& G, const LatOffsets& O, const Tables<double>& tb,
                                                  CXPtr x, const double* __restrict__ df, const Rec64& r64, int mlo,
                                                  int64_t s, int p, int8_t ti) {
  const int ei = species(ti);
  // neighbours from the FP64 site records: position and, in w, F' with the
  // species (a vacancy sits far out, so the distance test drops it)
  return ForceSiteD{x.c[0][s],
                    x.c[1][s],
                    x.c[2][s],
                    df[s],
                    ei,
                    rsrcBelow(r64.xy, O.lo),
                    rsrcBelow(r64.zw, O.lo),
                    rsrcAt(reinterpret_cast<uintptr_t>(tb.pairF)),
                    rsrcAt(reinterpret_cast<uintptr_t>(tb.rhoV)),
                    static_cast<uint32_t>(s) * 16u,
                    static_cast<uint32_t>(ei * 3) * static_cast<uint32_t>(tb.nr),
                    O.sh[p],
                    G.rc2,
                    mlo};
}
// The pairs of range rg (mask word w) of a site: the held ones into part, the
// others into opart, in offset order.  With LDS the Fe-Fe segments from knot
// first on come from knD (pairSegD).
template <int U, bool LDS = false>
__device__ __forceinline__ void forceRangeD(const ForceSiteD& c, const Tables<double>& tb, uint32_t w, int rg,
                                            Force3& part, Force3& opart, const double* knD = nullptr,
                                            int first = 0) {
  auto group = [&](auto UC, const int* ks) {
    constexpr int V = decltype(UC)::value;
    double d0[V], d1[V], d2[V], wj[V];
#pragma unroll
    for (int u = 0; u < V; ++u) {
      const uint32_t so = c.sh[ks[u]] * 16u;
      const double2 xy = ldRec64(c.rxy, c.o16, so), zw = ldRec64(c.rzw, c.o16, so);
      d0[u] = xy.x;
      d1[u] = xy.y;
      d2[u] = zw.x;
      wj[u] = zw.y;
    }
    bool in[V], held[V];
    double pp[V], ri[V], rec[V][kPairRec], reci[V][kRhoRec];
#pragma unroll
    for (int u = 0; u < V; ++u) {
      d0[u] = c.x0 - d0[u];
      d1[u] = c.x1 - d1[u];
      d2[u] = c.x2 - d2[u];
      const double r2 = dist2D(d0[u], d1[u], d2[u]);
      in[u] = r2 < c.rc2;
      if (in[u]) {
        ri[u] = rsqT(r2);
        const int m = knotM(r2 * ri[u], tb.rdr, tb.nr, pp[u]);
        const int ej = recSpecies64(wj[u]);
        held[u] = heldPair(c.ei, static_cast<uint32_t>(ej), m, c.mlo);
        pairSegD<LDS>(c.rtab, c.rtabR, knD, first, c.pairBase, tb.nr, c.ei, ej, m, rec[u], reci[u]);
      }
    }
#pragma unroll
    for (int u = 0; u < V; ++u) {
      if (!in[u]) continue;
      const double* z = rec[u];
      const double fp = pairFpD(pp[u], ri[u], z[0], z[1], z[2], z[3], z[4], z[5], z[6], reci[u][0], reci[u][1],
                                reci[u][2], c.dfi, wj[u], tb.rdr);
      if (held[u]) part.add(d0[u], d1[u], d2[u], fp);
      else opart.add(d0[u], d1[u], d2[u], fp);
    }
  };
  forMaskGroups<U>(static_cast<uint64_t>(w), 0ull, [&](const int* k32, int nv) {
    int ks[U];
#pragma unroll
    for (int u = 0; u < U; ++u) ks[u] = k32[u] + 32 * rg;
    if (nv == U) group(std::integral_constant<int, U>{}, ks);
    else group(std::integral_constant<int, 1>{}, ks);
  });
}

// One site of the FP64 force pass, one wavefront over all its offsets.
template <int MODE, int U, bool LDS = false>
__device__ __forceinline__ void forceSiteD(const Geom& G, const LatOffsets& O, const Tables<double>& tb, CXPtr x,
                                           XPtr xn, const int8_t* __restrict__ type, const double* __restrict__ df,
                                           const uint64_t* __restrict__ wmask, XPtr v, XPtr f,
                                           const uint64_t* __restrict__ id, const VerletParams& vp,
                                           const StageArgs& st, Ctl* ctl, const InterView& iv, const Rec64& r64,
                                           const Rec64& rn64, int mlo, uint32_t b, uint32_t tl,
                                           unsigned long long& vb, unsigned long long& db,
                                           const double* knD = nullptr, int first = 0) {
  int64_t s;
  int p, cx, cy, cz;
  if (!siteOfBlock(G, b, tl, s, p, cx, cy, cz)) return;
  const int8_t ti = type[s];
  if (isVacant(ti)) {  // vacancy: keeps its stale position (atom.cpp:43-47)
    vacancyForceD<MODE>(G, s, p, cx, cy, cz, ti, x, xn, f, rn64);
    return;
  }
  const ForceSiteD c = forceSiteOf(G, O, tb, x, df, r64, mlo, s, p, ti);
  Force3 tot, otot;
  // the offsets the density pass found in range for some lane of this wavefront
  const uint32_t wv = b * (kBlock / 64) + __builtin_amdgcn_readfirstlane(tl >> 6);
  const uint64_t m0 = uniform64(wmask[2 * wv]), m1 = uniform64(wmask[2 * wv + 1]);
  for (int rg = 0; rg < 4; ++rg) {
    Force3 part, opart;
    forceRangeD<U, LDS>(c, tb, maskWord(m0, m1, rg), rg, part, opart, knD, first);
    tot.add(part);
    otot.add(opart);
  }
  tot.add(otot);
  forceTailD<MODE>(G, s, p, cx, cy, cz, ti, c.ei, c.dfi, tot, c.x0, c.x1, c.x2, tb, x, xn, type, df, v, f, id, vp,
                   st, ctl, iv, rn64, vb, db);
}

// The FP64 force pass with four wavefronts to 64 sites (boxes with few sites).
template <int MODE, int U>
__global__ __launch_bounds__(kBlock) void kForceP(Geom G, LatOffsets O, Tables<double> tb, CXPtr x, XPtr xn,
                                                  const int8_t* __restrict__ type, const double* __restrict__ df,
                                                  const uint64_t* __restrict__ wmask, XPtr v, XPtr f,
                                                  const uint64_t* __restrict__ id, VerletParams vp, StageArgs st,
                                                  Ctl* ctl, InterView iv, InterDev in, Rec64 r64, Rec64 rn64,
                                                  int mlo) {
  __shared__ double parts[3][6][64];
  __shared__ TailHits hits;
  if (blockIdx.x < frontBlocks(G)) {
    interForceBody<double, MODE>(G, tb, iv, x, type, df, 1, in, vp, frontWave(), frontWaves(G));
    return;
  }
  const SharedSite q = sharedSite(G, type, blockIdx.x - frontBlocks(G));
  const int lane = static_cast<int>(threadIdx.x & 63u);
  ForceSiteD c{};
  Force3 part, opart;
  if (!isVacant(q.ti)) {
    c = forceSiteOf(G, O, tb, x, df, r64, mlo, q.s, q.p, q.ti);
    const uint32_t w =
        __builtin_amdgcn_readfirstlane(reinterpret_cast<const uint32_t*>(wmask)[4 * q.wv + q.rg]);
    forceRangeD<U>(c, tb, w, q.rg, part, opart);
  }
  if (q.rg > 0) {
    double(&o)[6][64] = parts[q.rg - 1];
    o[0][lane] = part.x;
    o[1][lane] = part.y;
    o[2][lane] = part.z;
    o[3][lane] = opart.x;
    o[4][lane] = opart.y;
    o[5][lane] = opart.z;
  }
  findTailHits(hits, q.rg, iv, x.c, type, G.rc2, q.p, q.s, q.ti);
  __syncthreads();
  if (q.rg > 0) return;
  unsigned long long vb = 0, db = 0;
  if (q.site && isVacant(q.ti)) {
    vacancyForceD<MODE>(G, q.s, q.p, q.cx, q.cy, q.cz, q.ti, x, xn, f, rn64);
  } else if (q.site) {
    Force3 tot, otot;
    tot.add(part);
    otot.add(opart);
#pragma unroll
    for (int rg = 1; rg < 4; ++rg) {
      const double(&o)[6][64] = parts[rg - 1];
      part.x = o[0][lane];
      part.y = o[1][lane];
      part.z = o[2][lane];
      opart.x = o[3][lane];
      opart.y = o[4][lane];
      opart.z = o[5][lane];
      tot.add(part);
      otot.add(opart);
    }
    tot.add(otot);
    forceTailD<MODE>(G, q.s, q.p, q.cx, q.cy, q.cz, q.ti, c.ei, c.dfi, tot, c.x0, c.x1, c.x2, tb, x, xn, type, df, v,
                     f, id, vp, st, ctl, iv, rn64, vb, db, &hits);
  }
  if (MODE == 0 && vp.vmax) waveMaxTo(vb, vp.vmax);
  if (MODE == 1) waveMaxTo(db, &ctl->dispmax2);
}

// The Fe-Fe segments of the FP64 LDS pass from knot mlo on, 40 bytes a knot:
// {slope of r*phi, slope of rho} and {value of r*phi, its step to the next
// knot} in 16-byte halves, and the density's step.  The cubics' two other
// coefficients come from the knot and its successor, with the operations and
// roundings that the tables were built with, so the segments are the tables'.
struct KnotsD {
  const double2* s;   // {s_z, s_rho} of knot m at s[m] (the arrays start at knot mlo)
  const double2* yd;  // {y_z, y_z(m+1) - y_z(m)}
  const double* dr;   // y_rho(m+1) - y_rho(m)
};
__device__ __forceinline__ double hermite4(double dy, double s0, double s1) {  // 3 dy - 2 s0 - s1
  return __dsub_rn(__fma_rn(-2.0, s0, __dmul_rn(3.0, dy)), s1);
}
__device__ __forceinline__ double hermite3(double dy, double s0, double s1) {  // s0 + s1 - 2 dy
  return __fma_rn(-2.0, dy, __dadd_rn(s0, s1));
}

// Works off the first n (at most 64) noted pairs, one a lane, as
// drainQueueM does; the pairs of one rank are added before those of the next,
// so every site's pairs join its sum in offset order.
__device__ __forceinline__ void drainQueueD(const uint16_t* q, int n, int rg, double xi0, double xi1, double xi2,
                                            int ei, double dfi, uint32_t o16, Rsrc rxy, Rsrc rzw, Rsrc rtab, Rsrc rtabR,
                                            const Tables<double>& tb, const uint32_t* __restrict__ sh, WaveSums& ws) {
  const int lane = static_cast<int>(threadIdx.x & 63u);
  const bool on = lane < n;
  const uint32_t e = q[on ? lane : 0];
  const int owner = static_cast<int>(e & 63u);
  const uint32_t rank = e >> 11;
  const uint32_t oo = static_cast<uint32_t>(laneGet(static_cast<int>(o16), owner)) + sh[32 * rg + ((e >> 6) & 31u)] * 16u;
  const double2 xy = ldRec64(rxy, oo, 0), zw = ldRec64(rzw, oo, 0);
  const double d0 = laneGet(xi0, owner) - xy.x, d1 = laneGet(xi1, owner) - xy.y, d2 = laneGet(xi2, owner) - zw.x;
  const int ti = laneGet(ei, owner), tj = recSpecies64(zw.y);
  const double r2 = dist2D(d0, d1, d2);
  const double ri = rsqT(r2);
  double pp, rec[kPairRec], reci[kRhoRec];
  const int m = knotM(r2 * ri, tb.rdr, tb.nr, pp);
  pairSegD<false>(rtab, rtabR, nullptr, 0, static_cast<uint32_t>(ti * 3) * static_cast<uint32_t>(tb.nr), tb.nr, ti,
                  tj, m, rec, reci);
  const double fp = pairFpD(pp, ri, rec[0], rec[1], rec[2], rec[3], rec[4], rec[5], rec[6], reci[0], reci[1],
                            reci[2], laneGet(dfi, owner), zw.y, tb.rdr);
  bool wait = on;
  for (uint32_t r = 0; __ballot(wait); ++r) {
    if (wait && rank == r) {
      ws.s[0][owner] = __fma_rn(d0, fp, ws.s[0][owner]);
      ws.s[1][owner] = __fma_rn(d1, fp, ws.s[1][owner]);
      ws.s[2][owner] = __fma_rn(d2, fp, ws.s[2][owner]);
      wait = false;
    }
    waveLdsFence();  // another lane's pair of this site reads what was just written
  }
}

// One virtual block of the FP64 LDS force pass: per site the same pairs and
// sums as kForce (forceSiteD), the segments of the held pairs from LDS and
// the other pairs worked off by the whole wavefront at the end of each range.
template <int MODE, int U>
__device__ __forceinline__ void forceVBlockD(const Geom& G, const LatOffsets& O, const Tables<double>& tb, CXPtr x,
                                             XPtr xn, const int8_t* __restrict__ type,
                                             const double* __restrict__ df, const uint64_t* __restrict__ wmask,
                                             XPtr v, XPtr f, const uint64_t* __restrict__ id, const VerletParams& vp,
                                             const StageArgs& st, Ctl* ctl, const InterView& iv, const Rec64& r64,
                                             const Rec64& rn64, const KnotsD& kn, int mlo, WaveQueueD<U>& wq,
                                             WaveSums& ws, uint32_t b, uint32_t tl, unsigned long long& vb,
                                             unsigned long long& db) {
  int64_t s = 0;
  int p = 0, cx = 0, cy = 0, cz = 0;
  const bool site = siteOfBlock(G, b, tl, s, p, cx, cy, cz);
  int8_t ti = kVacant;
  if (site) {
    ti = type[s];
    if (isVacant(ti)) vacancyForceD<MODE>(G, s, p, cx, cy, cz, ti, x, xn, f, rn64);
  }
  const bool live = !isVacant(ti);
  const uint64_t lives = __ballot(live);
  if (!lives) return;
  const int lane = static_cast<int>(threadIdx.x & 63u);
  const int ei = live ? species(ti) : 0;
  double xi0 = kNoAtom, xi1 = kNoAtom, xi2 = kNoAtom, dfi = 0.0;
  if (live) {
    xi0 = x.c[0][s];
    xi1 = x.c[1][s];
    xi2 = x.c[2][s];
    dfi = df[s];
  }
  const Rsrc rxy = rsrcBelow(r64.xy, O.lo), rzw = rsrcBelow(r64.zw, O.lo);
  const Rsrc rtab = rsrcAt(reinterpret_cast<uintptr_t>(tb.pairF));
  const Rsrc rtabR = rsrcAt(reinterpret_cast<uintptr_t>(tb.rhoV));
  const uint32_t o16 = addressOfLives(static_cast<uint32_t>(s) * 16u, live, lives);
  const uint32_t* sh = O.sh[__builtin_amdgcn_readfirstlane((b >> 3) & 1u)];
  const uint32_t wv = b * (kBlock / 64) + __builtin_amdgcn_readfirstlane(tl >> 6);
  const uint64_t m0 = uniform64(wmask[2 * wv]), m1 = uniform64(wmask[2 * wv + 1]);
  Force3 tot, otot;
  // The next U offsets of a range and their records' loads; an entry past the
  // range's last offset reads the site's own record and counts for no lane,
  // and so does a group past the last range (rg 4).
  struct Group {
    int rg;
    int ks[U];
    bool act[U];
    double2 xy[U], zw[U];
  } g, h;
  uint32_t w = maskWord(m0, m1, 0);
  int next = 0;  // the range w belongs to
  auto fetch = [&](Group& q) {
    while (w == 0 && next < 3) w = maskWord(m0, m1, ++next);
    q.rg = w ? next : 4;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      q.act[u] = w != 0;
      q.ks[u] = w ? 32 * next + __builtin_ctz(w) : kPadOffset;
      w &= w - 1;
      const uint32_t so = sh[q.ks[u]] * 16u;
      q.xy[u] = ldRec64(rxy, o16, so);
      q.zw[u] = ldRec64(rzw, o16, so);
    }
  };
  int rg = 0, qn = 0;  // the range being summed, the pairs noted in it
  uint32_t rank = 0;
  bool sums = false;
  Force3 part;
  auto pairs = [&](const Group& q) {
    bool held[U];
    uint64_t other[U];
    double d0[U], d1[U], d2[U], fp[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      d0[u] = xi0 - q.xy[u].x;
      d1[u] = xi1 - q.xy[u].y;
      d2[u] = xi2 - q.zw[u].x;
      const double r2 = dist2D(d0[u], d1[u], d2[u]);
      const double ri = rsqT(r2);
      double pp;
      const int m = knotM(r2 * ri, tb.rdr, tb.nr, pp);
      const uint64_t in = q.act[u] ? __ballot(r2 < G.rc2) : 0;
      const uint64_t hm =
          in & __ballot((static_cast<uint32_t>(ei) | static_cast<uint32_t>(recSpecies64(q.zw[u].y))) == 0u) &
          __ballot(m >= mlo);
      other[u] = in & ~hm;
      held[u] = __builtin_amdgcn_inverse_ballot_w64(hm);
      const int k = max(m, mlo);
      const double2 s0 = kn.s[k], s1 = kn.s[k + 1], yd = kn.yd[k];
      const double dr = kn.dr[k];
      const double z3 = hermite3(yd.y, s0.x, s1.x), z4 = hermite4(yd.y, s0.x, s1.x);
      const double j3 = hermite3(dr, s0.y, s1.y), j4 = hermite4(dr, s0.y, s1.y);
      fp[u] = pairFpD(pp, ri, z3, z4, s0.x, yd.x, j3, j4, s0.y, j3, j4, s0.y, dfi, q.zw[u].y, tb.rdr);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (other[u]) {
        if (__builtin_amdgcn_inverse_ballot_w64(other[u]))
          wq.q[qn + laneRank(other[u])] =
              static_cast<uint16_t>((rank++ << 11) | ((static_cast<uint32_t>(q.ks[u]) & 31u) << 6) |
                                    static_cast<uint32_t>(lane));
        qn += __builtin_popcountll(other[u]);
      }
      if (held[u]) part.add(d0[u], d1[u], d2[u], fp[u]);
    }
  };
  // Before a group of range `to`: works off full wavefronts of noted pairs
  // and, where a range ends, all of them, and closes its sums.
  auto settle = [&](int to) {
    while (qn >= (to != rg ? 1 : 64)) {
      if (!sums) {
        sums = true;
        for (int c = 0; c < 3; ++c) ws.s[c][lane] = 0.0;
      }
      waveLdsFence();
      const int n = qn < 64 ? qn : 64;
      drainQueueD(wq.q, n, rg, xi0, xi1, xi2, ei, dfi, o16, rxy, rzw, rtab, rtabR, tb, sh, ws);
      qn -= n;
      waveLdsFence();
      if (qn > 0) shiftQueueD(wq, lane);
    }
    if (to == rg) return;
    rg = to;
    rank = 0;
    tot.add(part);
    part = Force3();
    if (sums) {
      Force3 o;
      o.x = ws.s[0][lane];
      o.y = ws.s[1][lane];
      o.z = ws.s[2][lane];
      otot.add(o);
      sums = false;
    }
  };
  fetch(g);
  while (g.rg < 4) {
    fetch(h);
    if (g.rg != rg || qn >= 64) settle(g.rg);
    pairs(g);
    if (h.rg == 4) break;
    fetch(g);
    if (h.rg != rg || qn >= 64) settle(h.rg);
    pairs(h);
  }
  settle(4);
  if (!live) return;
  tot.add(otot);
  unsigned long long vbs = 0, dbs = 0;
  forceTailD<MODE>(G, s, p, cx, cy, cz, ti, ei, dfi, tot, xi0, xi1, xi2, tb, x, xn, type, df, v, f, id, vp, st, ctl,
                   iv, rn64, vbs, dbs);
  vb = vbs > vb ? vbs : vb;
  db = dbs > db ? dbs : db;
}

template <int MODE, int U>
__global__ __launch_bounds__(kBlock) void kForce(Geom G, LatOffsets O, Tables<double> tb, CXPtr x, XPtr xn,
                                                 const int8_t* __restrict__ type, const double* __restrict__ df,
                                                 const uint64_t* __restrict__ wmask, XPtr v, XPtr f,
                                                 const uint64_t* __restrict__ id, VerletParams vp, StageArgs st,
                                                 Ctl* ctl, InterView iv, InterDev in, Rec64 r64, Rec64 rn64,
                                                 int mlo) {
  unsigned long long vb = 0;  // |v|^2 bits after the secondstep (MODE 0)
  unsigned long long db = 0;  // |dx|^2 bits of the drift (MODE 1)
  if (blockIdx.x < frontBlocks(G)) {
    interForceBody<double, MODE>(G, tb, iv, x, type, df, 1, in, vp, frontWave(), frontWaves(G));
    return;
  }
  forceSiteD<MODE, U>(G, O, tb, x, xn, type, df, wmask, v, f, id, vp, st, ctl, iv, r64, rn64, mlo,
                      blockIdx.x - frontBlocks(G), threadIdx.x, vb, db);
  if (MODE == 0 && vp.vmax) waveMaxTo(vb, vp.vmax);
  if (MODE == 1) waveMaxTo(db, &ctl->dispmax2);
}

// Sums of the neighbours set aside by the FP64 LDS density pass, per lane.
struct WaveSum1 {
  double s[64];
};

// drainQueueD for the density: the noted neighbours' densities, rank after rank.
__device__ __forceinline__ void drainRhoD(const uint16_t* q, int n, int rg, double xi0, double xi1, double xi2,
                                          uint32_t o16, Rsrc rxy, Rsrc rzw, Rsrc rtab, const Tables<double>& tb,
                                          const uint32_t* __restrict__ sh, WaveSum1& ws) {
  const int lane = static_cast<int>(threadIdx.x & 63u);
  const bool on = lane < n;
  const uint32_t e = q[on ? lane : 0];
  const int owner = static_cast<int>(e & 63u);
  const uint32_t rank = e >> 11;
  const uint32_t oo = static_cast<uint32_t>(laneGet(static_cast<int>(o16), owner)) + sh[32 * rg + ((e >> 6) & 31u)] * 16u;
  const double2 xy = ldRec64(rxy, oo, 0), zw = ldRec64(rzw, oo, 0);
  const double r2 = dist2D(laneGet(xi0, owner) - xy.x, laneGet(xi1, owner) - xy.y, laneGet(xi2, owner) - zw.x);
  double pp, c[kRhoRec];
  const int m = knotM(r2 * rsqT(r2), tb.rdr, tb.nr, pp);
  ldRec<double, kRhoRec>(rtab, static_cast<uint32_t>(recSpecies64(zw.y) * tb.nr + m) * (kRhoRec * 8u), c);
  const double v = cubicD(c[0], c[1], c[2], c[3], pp);
  bool wait = on;
  for (uint32_t r = 0; __ballot(wait); ++r) {
    if (wait && rank == r) {
      ws.s[owner] += v;
      wait = false;
    }
    waveLdsFence();  // another lane's neighbour of this site reads what was just written
  }
}

// The Fe density cubics of the LDS density pass, knot m's {c3, c4} at a[m] and
// {c5, c6} at b[m], in arrays of their own: at 32 bytes a knot in one array
// the 16-byte reads of a wavefront would meet in half the banks.
struct KnotsRho {
  const double2* a;
  const double2* b;
};

// One virtual block of the FP64 LDS density pass: per site the same
// neighbours, sums and masks as kRhoDf; an Fe neighbour's cubic at a knot from
// mlo on from LDS, the others worked off by the whole wavefront as in
// forceVBlockD, with the next group's records in flight during a group.
template <int U>
__device__ __forceinline__ void rhoVBlockD(const Geom& G, const LatOffsets& O, const Tables<double>& tb, CXPtr x,
                                           const int8_t* __restrict__ type, double* __restrict__ df,
                                           double* __restrict__ rho_out, uint64_t* __restrict__ wmask,
                                           uint64_t* __restrict__ smask, double rcs2, const InterView& iv,
                                           const Rec64& r64, const KnotsRho& kn, int mlo, WaveQueueD<U>& wq,
                                           WaveSum1& ws, uint32_t b, uint32_t tl) {
  int64_t s = 0;
  int p = 0, cx = 0, cy = 0, cz = 0;
  const bool site = siteOfBlock(G, b, tl, s, p, cx, cy, cz);
  const int8_t ti = site ? type[s] : kVacant;
  const bool live = !isVacant(ti);
  const uint64_t lives = __ballot(live);
  Sum1<0> tot, otot;
  if (lives) {
    const bool skin = __builtin_amdgcn_readfirstlane(iv.ctl->skin_mode) != 0 && !__ballot(live && (ti & kWide));
    const int lane = static_cast<int>(threadIdx.x & 63u);
    double xi0 = kNoAtom, xi1 = kNoAtom, xi2 = kNoAtom;
    if (live) {
      xi0 = x.c[0][s];
      xi1 = x.c[1][s];
      xi2 = x.c[2][s];
    }
    const Rsrc rxy = rsrcBelow(r64.xy, O.lo), rzw = rsrcBelow(r64.zw, O.lo);
    const Rsrc rtab = rsrcAt(reinterpret_cast<uintptr_t>(tb.rhoV));
    const uint32_t o16 = addressOfLives(static_cast<uint32_t>(s) * 16u, live, lives);
    const int pu = __builtin_amdgcn_readfirstlane((b >> 3) & 1u);
    const uint32_t* sh = O.sh[pu];
    const uint32_t wv = b * (kBlock / 64) + __builtin_amdgcn_readfirstlane(tl >> 6);
    uint64_t m0, m1;
    if (skin) {
      m0 = uniform64(smask[2 * wv]);
      m1 = uniform64(smask[2 * wv + 1]);
    } else {
      const int nk = O.n[pu];
      m0 = nk >= 64 ? ~0ull : (1ull << nk) - 1;
      m1 = nk > 64 ? (1ull << (nk - 64)) - 1 : 0;  // nk < 128: kPadOffset is no offset
    }
    uint64_t w0 = 0, w1 = 0, s0 = 0, s1 = 0;
    struct Group {
      int rg;
      int ks[U];
      bool act[U];
      double2 xy[U], zw[U];
    } g, h;
    uint32_t w = maskWord(m0, m1, 0);
    int next = 0;  // the range w belongs to
    auto fetch = [&](Group& q) {
      while (w == 0 && next < 3) w = maskWord(m0, m1, ++next);
      q.rg = w ? next : 4;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        q.act[u] = w != 0;
        q.ks[u] = w ? 32 * next + __builtin_ctz(w) : kPadOffset;
        w &= w - 1;
        const uint32_t so = sh[q.ks[u]] * 16u;
        q.xy[u] = ldRec64(rxy, o16, so);
        q.zw[u] = ldRec64(rzw, o16, so);
      }
    };
    int rg = 0, qn = 0;  // the range being summed, the neighbours noted in it
    uint32_t rank = 0;
    bool sums = false;
    Sum1<0> part;
    auto pairs = [&](const Group& q) {
      double r2[U];
      uint64_t in[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        r2[u] = dist2D(xi0 - q.xy[u].x, xi1 - q.xy[u].y, xi2 - q.zw[u].x);
        in[u] = q.act[u] ? __ballot(r2[u] < G.rc2) : 0;
        if (!skin && q.act[u] && __ballot(r2[u] < rcs2)) setBit(s0, s1, q.ks[u]);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (!in[u]) continue;  // a third of the offsets of a full scan
        setBit(w0, w1, q.ks[u]);
        double pp;
        const int m = knotM(r2[u] * rsqT(r2[u]), tb.rdr, tb.nr, pp);
        const uint64_t hm = in[u] & __ballot(recSpecies64(q.zw[u].y) == 0) & __ballot(m >= mlo);
        const uint64_t other = in[u] & ~hm;
        const int k = max(m, mlo);
        const double2 c = kn.a[k], d = kn.b[k];
        if (other) {
          if (__builtin_amdgcn_inverse_ballot_w64(other))
            wq.q[qn + laneRank(other)] =
                static_cast<uint16_t>((rank++ << 11) | ((static_cast<uint32_t>(q.ks[u]) & 31u) << 6) |
                                      static_cast<uint32_t>(lane));
          qn += __builtin_popcountll(other);
        }
        if (__builtin_amdgcn_inverse_ballot_w64(hm)) part.add(cubicD(c.x, c.y, d.x, d.y, pp));
      }
    };
    // as in forceVBlockD: before a group of range `to`
    auto settle = [&](int to) {
      while (qn >= (to != rg ? 1 : 64)) {
        if (!sums) {
          sums = true;
          ws.s[lane] = 0.0;
        }
        waveLdsFence();
        const int n = qn < 64 ? qn : 64;
        drainRhoD(wq.q, n, rg, xi0, xi1, xi2, o16, rxy, rzw, rtab, tb, sh, ws);
        qn -= n;
        waveLdsFence();
        if (qn > 0) shiftQueueD(wq, lane);
      }
      if (to == rg) return;
      rg = to;
      rank = 0;
      tot.join(part);
      part = Sum1<0>();
      if (sums) {
        Sum1<0> o;
        o.s = ws.s[lane];
        otot.join(o);
        sums = false;
      }
    };
    fetch(g);
    while (g.rg < 4) {
      fetch(h);
      if (g.rg != rg || qn >= 64) settle(g.rg);
      pairs(g);
      if (h.rg == 4) break;
      fetch(g);
      if (h.rg != rg || qn >= 64) settle(h.rg);
      pairs(h);
    }
    settle(4);
    if (lane == __builtin_ctzll(lives)) {
      wmask[2 * wv] = w0;
      wmask[2 * wv + 1] = w1;
      if (!skin) {
        smask[2 * wv] = s0;
        smask[2 * wv + 1] = s1;
      }
    }
  }
  if (!site) return;
  tot.join(otot);
  rhoTailD(G, s, p, cx, cy, cz, ti, tot, x, type, tb, df, rho_out, iv, r64);
}

// The FP64 density pass in persistent blocks, one per compute unit, with the
// Fe density cubics from knot mlo on in LDS.  Half of kRhoDf's loads are the
// segments, scattered over 160 KB a species, and the texture units bound it;
// from LDS two 16-byte reads take their place (2M atoms: 483 -> 372 us).  Two
// offsets a group: four need 118 registers and leave more of a group idle at
// the end of a range (390 us).
template <int U>
__global__ __launch_bounds__(kBlockP) void kRhoDL(Geom G, LatOffsets O, Tables<double> tb, CXPtr x,
                                                  const int8_t* __restrict__ type, double* __restrict__ df,
                                                  double* __restrict__ rho_out, uint64_t* __restrict__ wmask,
                                                  uint64_t* __restrict__ smask, double rcs2, InterView iv, InterDev in,
                                                  Rec64 r64, int mlo, int nkn) {
  __shared__ WaveQueueD<U> queues[kBlockP / 64];
  __shared__ WaveSum1 sums[kBlockP / 64];
  extern __shared__ double2 knS[];  // nkn {c3, c4}, nkn {c5, c6}
  const double2* z = reinterpret_cast<const double2*>(tb.rhoV) + 2 * static_cast<size_t>(mlo);  // row Fe is the first
  for (int i = threadIdx.x; i < nkn; i += kBlockP) {
    knS[i] = z[2 * i];
    knS[nkn + i] = z[2 * i + 1];
  }
  __syncthreads();
  const KnotsRho kn{knS - mlo, knS + nkn - mlo};
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  interRhoBody<double>(G, tb, iv, x, type, in, static_cast<int>(wave * gridDim.x + blockIdx.x),
                       static_cast<int>(gridDim.x) * (kBlockP / 64));
  forVirtualBlocks(G, [&](uint32_t b, uint32_t tl) {
    rhoVBlockD<U>(G, O, tb, x, type, df, rho_out, wmask, smask, rcs2, iv, r64, kn, mlo, queues[wave], sums[wave], b,
                  tl);
  });
}

// Potential energy and virial of site s (FP64 tables, FP64 site records):
// F(rho_i) into vals[0], 1/2 sum_j phi(r_ij) into vals[1] and
// 1/2 sum_j r_ij^2 fpair_ij into vals[2], fpair as the force pass computes it
// and F'(rho_j) from the records' w.  The offsets are those of the
// wavefront's skin mask (within the cutoff plus the skin of every pair at the
// last full density scan, so a superset of the pairs within the cutoff), or
// all pruned offsets when all is set (no skin).  With LDS the Fe-Fe segments
// come from knD, 7 doubles a knot (pairSegD).  Near a far lattice atom the rest of the
// full list follows from x and df.
template <bool LDS>
__device__ __forceinline__ void energySiteD(const Geom& G, const LatOffsets& O, const FullPlaneOffsets* full,
                                           const Tables<double>& tb, CXPtr x, const int8_t* __restrict__ type,
                                           const double* __restrict__ rho, const double* __restrict__ df,
                                           const uint64_t* __restrict__ smask, bool all, const Rec64& r64,
                                           const double* knD, int mlo, uint32_t b, uint32_t tl,
                                           double (&vals)[3]) {
  int64_t s;
  int p, cx, cy, cz;
  if (!siteOfBlock(G, b, tl, s, p, cx, cy, cz)) return;
  const int8_t ti = type[s];
  if (isVacant(ti)) return;
  const int ei = species(ti);
  const double ri = rho[s];
  const double dfi = dEmbed(tb, ei, ri);
  vals[0] += embed(tb, ei, ri);
  const double xi0 = x.c[0][s], xi1 = x.c[1][s], xi2 = x.c[2][s];
  const Rsrc rxy = rsrcBelow(r64.xy, O.lo), rzw = rsrcBelow(r64.zw, O.lo);
  const Rsrc rtab = rsrcAt(reinterpret_cast<uintptr_t>(tb.pairF));
  const Rsrc rtabR = rsrcAt(reinterpret_cast<uintptr_t>(tb.rhoV));
  const uint32_t o16 = static_cast<uint32_t>(s) * 16u;
  const uint32_t pairBase = static_cast<uint32_t>(ei * 3) * static_cast<uint32_t>(tb.nr);
  const uint32_t* sh = O.sh[p];
  auto group = [&](auto UC, const int* ks) {
    constexpr int V = decltype(UC)::value;
    double d0[V], d1[V], d2[V], wj[V];
#pragma unroll
    for (int u = 0; u < V; ++u) {
      const uint32_t so = sh[ks[u]] * 16u;
      const double2 xy = ldRec64(rxy, o16, so), zw = ldRec64(rzw, o16, so);
      d0[u] = xi0 - xy.x;
      d1[u] = xi1 - xy.y;
      d2[u] = xi2 - zw.x;
      wj[u] = zw.y;
    }
    bool in[V];
    double r2[V], pp[V], rinv[V], rec[V][kPairRec], reci[V][kRhoRec];
#pragma unroll
    for (int u = 0; u < V; ++u) {
      r2[u] = dist2D(d0[u], d1[u], d2[u]);
      in[u] = r2[u] < G.rc2;
      if (in[u]) {
        rinv[u] = rsqT(r2[u]);
        const int m = knotOf(r2[u] * rinv[u], tb.rdr, tb.nr, false, pp[u]);
        pairSegD<LDS>(rtab, rtabR, knD, mlo, pairBase, tb.nr, ei, recSpecies64(wj[u]), m, rec[u], reci[u]);
      }
    }
#pragma unroll
    for (int u = 0; u < V; ++u) {
      if (!in[u]) continue;
      const double q = pp[u];
      const double* z = rec[u];
      const double* rj = rec[u] + 4;
      const double* rI = reci[u];
      const double z2 = ((z[0] * q + z[1]) * q + z[2]) * q + z[3];
      const double z2p = ((3.0 * z[0] * q + 2.0 * z[1]) * q + z[2]) * tb.rdr;
      const double rhojp = ((3.0 * rj[0] * q + 2.0 * rj[1]) * q + rj[2]) * tb.rdr;
      const double rhoip = ((3.0 * rI[0] * q + 2.0 * rI[1]) * q + rI[2]) * tb.rdr;
      const double phi = z2 * rinv[u];
      const double phip = z2p * rinv[u] - phi * rinv[u];
      const double psip = dfi * rhojp + wj[u] * rhoip + phip;
      vals[1] += 0.5 * phi;
      vals[2] += 0.5 * r2[u] * (-psip * rinv[u]);
    }
  };
  if (all) {
    const int nk = O.n[p];
    int ks[2];
    int k = 0;
    for (; k + 2 <= nk; k += 2) {
      ks[0] = k;
      ks[1] = k + 1;
      group(std::integral_constant<int, 2>{}, ks);
    }
    if (k < nk) {
      ks[0] = k;
      group(std::integral_constant<int, 1>{}, ks);
    }
  } else {
    const uint32_t wv = b * (kBlock / 64) + __builtin_amdgcn_readfirstlane(tl >> 6);
    forMaskGroups<2>(uniform64(smask[2 * wv]), uniform64(smask[2 * wv + 1]), [&](const int* ks, int nv) {
      if (nv == 2) group(std::integral_constant<int, 2>{}, ks);
      else group(std::integral_constant<int, 1>{}, ks);
    });
  }
  if (ti & kWide) {  // full-list offsets beyond the pruned list, near a far lattice atom
    forWideTargets(*full, x.c, type, G.rc2, p, s, ti, xi0, xi1, xi2, nullptr, [&](int64_t j, int8_t tj) {
      const double e0 = xi0 - x.c[0][j], e1 = xi1 - x.c[1][j], e2 = xi2 - x.c[2][j];
      const double q2 = e0 * e0 + e1 * e1 + e2 * e2;
      if (q2 < G.rc2) {
        const int ej = species(tj);
        const double r = sqrt(q2);
        double q;
        const int m = knotOf(r, tb.rdr, tb.nr, false, q);
        vals[1] += 0.5 * splineVal(tb.z2 + pairIdx(ei, ej) * tb.sR + static_cast<int64_t>(m) * kKnot, q) / r;
        vals[2] += 0.5 * q2 * pairForce(tb, ei, ej, q2, dfi, df[j]);
      }
    });
  }
}

// Sums of a block's threads (fixed order), one value each into out.
template <int N, int THREADS>
__device__ __forceinline__ void blockSumD(double (&vals)[N], double* out) {
  __shared__ double red[N][THREADS / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int q = 0; q < N; q++) {
    double v = vals[q];
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    if (lane == 0) red[q][w] = v;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int q = 0; q < N; q++) {
      double v = 0;
      for (int k = 0; k < THREADS / 64; k++) v += red[q][k];
      out[q] = v;
    }
  }
}

// Potential energy and virial, one block's partial sums each: energySiteD
// over the sites of a siteGrid launch, or in persistent blocks with the
// Fe-Fe segments in LDS.
__global__ __launch_bounds__(kBlock) void kEnergyD(Geom G, LatOffsets O, const FullPlaneOffsets* __restrict__ full,
                                                   Tables<double> tb, CXPtr x, const int8_t* __restrict__ type,
                                                   const double* __restrict__ rho, const double* __restrict__ df,
                                                   const uint64_t* __restrict__ smask, int all, Rec64 r64,
                                                   double* partials) {
  double vals[3] = {0, 0, 0};
  energySiteD<false>(G, O, full, tb, x, type, rho, df, smask, all != 0, r64, nullptr, 0, blockIdx.x, threadIdx.x,
                     vals);
  blockSumD<3, kBlock>(vals, partials + 3 * blockIdx.x);
}
// The Fe-Fe segments from knot mlo on, 7 doubles a knot (pairSegD).
__device__ __forceinline__ void fillKnots7(const Tables<double>& tb, double* knD, int mlo, int nkn) {
  const double* z = tb.pairF + static_cast<size_t>(mlo) * kPairRec;  // row (Fe, Fe) is the first
  for (int i = threadIdx.x; i < 7 * nkn; i += kBlockP) {
    const int k = i / 7, q = i - 7 * k;
    knD[i] = z[static_cast<size_t>(k) * kPairRec + q];
  }
}
__global__ __launch_bounds__(kBlockP) void kEnergyDL(Geom G, LatOffsets O, const FullPlaneOffsets* __restrict__ full,
                                                     Tables<double> tb, CXPtr x, const int8_t* __restrict__ type,
                                                     const double* __restrict__ rho, const double* __restrict__ df,
                                                     const uint64_t* __restrict__ smask, int all, Rec64 r64,
                                                     double* partials, int mlo, int nkn) {
  extern __shared__ double knD[];
  fillKnots7(tb, knD, mlo, nkn);
  __syncthreads();
  double vals[3] = {0, 0, 0};
  forVirtualBlocks(G, [&](uint32_t b, uint32_t tl) {
    energySiteD<true>(G, O, full, tb, x, type, rho, df, smask, all != 0, r64, knD, mlo, b, tl, vals);
  });
  blockSumD<3, kBlockP>(vals, partials + 3 * blockIdx.x);
}

// The FP64 force pass in persistent blocks, one per compute unit, with the
// Fe-Fe segments from knot mlo on in LDS (forceVBlockD).  2M atoms with the
// fused half steps: 546 us, against 657 with 7 doubles a knot, the other pairs
// re-read under a mask and one group in flight.  At 16M atoms (4.41 ms) the
// queued neighbours' records come from beyond the L2 a second time, 1189 bytes
// an atom in all, 4.3 TB/s or 90 % of what a copy reaches; the texture-data
// units are 90 % busy and VALU issue takes 64 % of the cycles.
template <int MODE, int U>
__global__ __launch_bounds__(kBlockP) void kForceDL(Geom G, LatOffsets O, Tables<double> tb, CXPtr x, XPtr xn,
                                                    const int8_t* __restrict__ type, const double* __restrict__ df,
                                                    const uint64_t* __restrict__ wmask, XPtr v, XPtr f,
                                                    const uint64_t* __restrict__ id, VerletParams vp, StageArgs st,
                                                    Ctl* ctl, InterView iv, InterDev in, Rec64 r64, Rec64 rn64,
                                                    int mlo, int nkn) {
  __shared__ WaveQueueD<U> queues[kBlockP / 64];
  __shared__ WaveSums sums[kBlockP / 64];
  extern __shared__ double2 knS[];  // nkn {s_z, s_rho}, nkn {y_z, dy_z}, nkn dy_rho
  double2* ks = knS;  // one knot more: the last one starts no segment, but a pair there reads two
  double2* kyd = knS + nkn + 1;
  double* kdr = reinterpret_cast<double*>(knS + 2 * nkn + 1);
  const double* z = tb.pairF + static_cast<size_t>(mlo) * kPairRec;  // row (Fe, Fe) is the first
  for (int i = threadIdx.x; i < nkn; i += kBlockP) {
    const double* c = z + static_cast<size_t>(i) * kPairRec;       // r*phi c3..c6, rho c3..c6
    const double* n = i + 1 < nkn ? c + kPairRec : c;              // the last knot starts no segment
    ks[i] = make_double2(c[2], c[6]);
    if (i + 1 == nkn) ks[nkn] = ks[i];
    kyd[i] = make_double2(c[3], __dsub_rn(n[3], c[3]));
    kdr[i] = __dsub_rn(n[7], c[7]);
  }
  __syncthreads();
  const KnotsD kn{ks - mlo, kyd - mlo, kdr - mlo};
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  interForceBody<double, MODE>(G, tb, iv, x, type, df, 1, in, vp, static_cast<int>(wave * gridDim.x + blockIdx.x),
                               static_cast<int>(gridDim.x) * (kBlockP / 64));
  unsigned long long vb = 0, db = 0;
  forVirtualBlocks(G, [&](uint32_t b, uint32_t tl) {
    forceVBlockD<MODE, U>(G, O, tb, x, xn, type, df, wmask, v, f, id, vp, st, ctl, iv, r64, rn64, kn, mlo,
                          queues[wave], sums[wave], b, tl, vb, db);
  });
  if (MODE == 0 && vp.vmax) waveMaxTo(vb, vp.vmax);
  if (MODE == 1) waveMaxTo(db, &ctl->dispmax2);
}

// The FP64 force pass in persistent blocks with the Fe-Fe segments from knot
// `first` on in LDS (7 doubles a knot) and the other pairs' gathered under a
// mask, a lane each (forceSiteD): the form where so many pairs are not held
// that their queue costs more than the load slots of the masked gathers.
template <int MODE, int U>
__global__ __launch_bounds__(kBlockP) void kForceDG(Geom G, LatOffsets O, Tables<double> tb, CXPtr x, XPtr xn,
                                                    const int8_t* __restrict__ type, const double* __restrict__ df,
                                                    const uint64_t* __restrict__ wmask, XPtr v, XPtr f,
                                                    const uint64_t* __restrict__ id, VerletParams vp, StageArgs st,
                                                    Ctl* ctl, InterView iv, InterDev in, Rec64 r64, Rec64 rn64,
                                                    int mlo, int first, int nkn) {
  extern __shared__ double knD[];
  fillKnots7(tb, knD, first, nkn);
  __syncthreads();
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  interForceBody<double, MODE>(G, tb, iv, x, type, df, 1, in, vp, static_cast<int>(wave * gridDim.x + blockIdx.x),
                               static_cast<int>(gridDim.x) * (kBlockP / 64));
  unsigned long long vb = 0, db = 0;
  forVirtualBlocks(G, [&](uint32_t b, uint32_t tl) {
    unsigned long long vbs = 0, dbs = 0;
    forceSiteD<MODE, U, true>(G, O, tb, x, xn, type, df, wmask, v, f, id, vp, st, ctl, iv, r64, rn64, mlo, b, tl, vbs,
                              dbs, knD, first);
    vb = vbs > vb ? vbs : vb;
    db = dbs > db ? dbs : db;
  });
  if (MODE == 0 && vp.vmax) waveMaxTo(vb, vp.vmax);
  if (MODE == 1) waveMaxTo(db, &ctl->dispmax2);
}

// ---------------------------------------------------------------------------
// Mixed precision on site records: one 16-byte load per neighbour.
//   x_i - x_j = (u_i - u_j) - (site_j - site_i), the lattice vector of the
//   offset coming from a per-offset table in scalar registers.  The FP32
//   displacement differs from the FP64 one by a few 1e-7 relative, far inside
//   the mixed path's error bar, and the pair set differs from FP64's only for
//   pairs within that distance of the cutoff, where the tabulated functions
//   and their slopes vanish.
// ---------------------------------------------------------------------------
// The masks of pass 1 work as in FP64: both passes see the same records and
// round the distances the same way (dist2M), so a skipped offset has no pair.
// Per lane: the density sum of site s over the offsets [k0, k1), or with skin
// set over the bits of (b0, b1) of the last full scan's mask, U at a time; the
// entries past the last repeat its offset with the padding entry's lattice
// vector: they add nothing.  Sets the mask bits as rhoGroupD does.
template <int ACC, int U>
__device__ __forceinline__ void rhoSumM(const LatOffsets& O, const Tables<float>& tb, const float4* rec,
                                        const float4* __restrict__ dl, float rc2, float rcs2, int64_t s, int p,
                                        bool skin, int k0, int k1, uint64_t b0, uint64_t b1, RangeSum<ACC>& acc,
                                        uint64_t& w0, uint64_t& w1, uint64_t& s0, uint64_t& s1) {
  const float4 me = rec[s];
  const Rsrc rr = rsrcBelow(rec, O.lo);
  const Rsrc rtab = rsrcAt(reinterpret_cast<uintptr_t>(tb.rhoH));
  const uint32_t o16 = static_cast<uint32_t>(s) * 16u;
  // per pruned offset: the lattice vector and, in w, the record shift * 16
  const float4* D = dl + (2 + p) * kMaxLatOffsets;
  auto group = [&](const int (&ks)[U], const bool (&act)[U]) {
    float4 nb[U], d[U];
    bool in[U], sk[U];
#pragma unroll
    for (int u = 0; u < U; ++u) d[u] = D[act[u] ? ks[u] : kPadOffset];
#pragma unroll
    for (int u = 0; u < U; ++u) nb[u] = ldRec4(rr, o16, __float_as_uint(d[u].w));
    rhoGroupM<ACC, U>(me, nb, d, rc2, rcs2, rtab, tb, ks, acc, in, sk);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (__ballot(in[u])) setBit(w0, w1, ks[u]);
      if (!skin && __ballot(sk[u])) setBit(s0, s1, ks[u]);
    }
  };
  int ks[U];
  bool act[U];
  if (!skin) {
    for (int k = k0; k < k1; k += U) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        act[u] = k + u < k1;
        ks[u] = act[u] ? k + u : k1 - 1;
      }
      group(ks, act);
    }
  } else {
    int k = 0;
    while (b0 | b1) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        act[u] = (b0 | b1) != 0;
        if (b0) {
          k = __builtin_ctzll(b0);
          b0 &= b0 - 1;
        } else if (b1) {
          k = 64 + __builtin_ctzll(b1);
          b1 &= b1 - 1;
        }
        ks[u] = k;
      }
      group(ks, act);
    }
  }
}

// The density pass of block `blk` of one box (the kernel's own block, or a
// block of one box of a batch).
template <int ACC, int U>
__device__ __forceinline__ void rhoPassM(const Geom& G, const LatOffsets& O, const Tables<float>& tb, CXPtr x,
                                         const int8_t* __restrict__ type, float4* rec,
                                         const float4* __restrict__ dl, double* __restrict__ rho_out,
                                         uint64_t* __restrict__ wmask, uint64_t* __restrict__ smask, float rcs2,
                                         const InterView& iv, uint32_t blk) {
  int64_t s;
  int p, cx, cy, cz;
  if (!siteOfBlock(G, blk, threadIdx.x, s, p, cx, cy, cz)) return;
  const int8_t ti = type[s];
  // a wavefront next to a far lattice atom (kWide) scans in full and records its masks afresh
  const bool skin =
      __builtin_amdgcn_readfirstlane(iv.ctl->skin_mode) != 0 && !__ballot(!isVacant(ti) && (ti & kWide));
  const uint32_t wv = blk * (kBlock / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  RangeSum<ACC> acc;
  uint64_t w0 = 0, w1 = 0;  // offsets in range for some lane (uniform among the lanes that gather)
  uint64_t s0 = 0, s1 = 0;  // offsets within cutoff + skin for some lane (full scan)
  if (!isVacant(ti)) {
    uint64_t b0 = 0, b1 = 0;
    if (skin) {  // the offsets of the last full scan's skin mask, in ascending order
      b0 = uniform64(smask[2 * wv]);
      b1 = uniform64(smask[2 * wv + 1]);
    }
    rhoSumM<ACC, U>(O, tb, rec, dl, static_cast<float>(G.rc2), rcs2, s, p, skin, 0, O.n[p], b0, b1, acc, w0, w1, s0,
                    s1);
  }
  acc.close();
  writeMasks(!isVacant(ti), wv, w0, w1, wmask, !skin, s0, s1, smask);
  rhoTailM<ACC>(G, s, p, cx, cy, cz, ti, acc.tot, x, type, tb, iv, rec, rho_out);
}

// The mixed density pass with four wavefronts to 64 sites (boxes with few sites).
template <int ACC, int U>
__global__ __launch_bounds__(kBlock) void kRhoDfMP(Geom G, LatOffsets O, Tables<float> tb, CXPtr x,
                                                   const int8_t* __restrict__ type, float4* rec,
                                                   const float4* __restrict__ dl, double* __restrict__ rho_out,
                                                   uint64_t* __restrict__ wmask, uint64_t* __restrict__ smask,
                                                   float rcs2, InterView iv, InterDev in) {
  __shared__ RangeParts parts;
  __shared__ TailHits hits;
  if (blockIdx.x < frontBlocks(G)) {
    interRhoBody<float>(G, tb, iv, x, type, in, frontWave(), frontWaves(G));
    return;
  }
  const SharedSite q = sharedSite(G, type, blockIdx.x - frontBlocks(G));
  const bool live = !isVacant(q.ti);
  const bool skin = __builtin_amdgcn_readfirstlane(iv.ctl->skin_mode) != 0 && !__ballot(live && (q.ti & kWide));
  RangeSum<ACC> acc;
  acc.range = q.rg;
  uint64_t w0 = 0, w1 = 0, s0 = 0, s1 = 0, b0 = 0, b1 = 0;
  if (live) {
    const Range r = rangeOf(q.rg, O.n[q.p]);
    if (skin) rangeBits(smask, q.wv, q.rg, b0, b1);
    rhoSumM<ACC, U>(O, tb, rec, dl, static_cast<float>(G.rc2), rcs2, q.s, q.p, skin, r.k0, r.k1, b0, b1, acc, w0, w1,
                    s0, s1);
  }
  writeMaskWord(live, q.wv, q.rg, w0, w1, wmask, !skin, s0, s1, smask);
  if (q.rg > 0) putPart(parts, q.rg, acc.part);
  findTailHits(hits, q.rg, iv, x.c, type, G.rc2, q.p, q.s, q.ti);
  __syncthreads();
  if (q.rg > 0 || !q.site) return;
  acc.close();
  joinParts(parts, acc.tot);
  rhoTailM<ACC>(G, q.s, q.p, q.cx, q.cy, q.cz, q.ti, acc.tot, x, type, tb, iv, rec, rho_out, &hits);
}

template <int ACC, int U>
__global__ __launch_bounds__(kBlock, U == 4 ? 8 : 6) void kRhoDfM(Geom G, LatOffsets O, Tables<float> tb, CXPtr x,
                                                  const int8_t* __restrict__ type, float4* rec,
                                                  const float4* __restrict__ dl, double* __restrict__ rho_out,
                                                  uint64_t* __restrict__ wmask, uint64_t* __restrict__ smask,
                                                  float rcs2, InterView iv, InterDev in) {
  if (blockIdx.x < frontBlocks(G)) {
    interRhoBody<float>(G, tb, iv, x, type, in, frontWave(), frontWaves(G));
    return;
  }
  rhoPassM<ACC, U>(G, O, tb, x, type, rec, dl, rho_out, wmask, smask, rcs2, iv, blockIdx.x - frontBlocks(G));
}

// The density pass of every box of a batch in one launch: the blocks of box
// b are [start[b], start[b+1]), in the box's own block order (the starts are
// multiples of 8, so a block keeps its XCD).
template <int ACC, int U>
__global__ __launch_bounds__(kBlock) void kRhoDfMB(const BatchBox* __restrict__ boxes, const uint32_t* start,
                                                   int nbox, int flip) {
  const int b = boxOfBlock(start, nbox, blockIdx.x);
  const BatchBox& B = boxes[b];
  const int c = B.cur ^ flip;
  rhoPassM<ACC, U>(B.G, B.O, B.t32, cxp(B.x[c]), B.type, B.rec[c], B.dl, nullptr, B.wmask, B.smask, B.rcs2, B.iv,
                   blockIdx.x - start[b]);
}

// Per lane: the force sum of the atom on site s (record me) over the offsets
// of the mask (b0, b1), the segments from the tables in global memory: the
// held pairs into acc, the others into oth.
template <int U, typename Acc>
__device__ __forceinline__ void forceSumM(const LatOffsets& O, const Tables<float>& tb, const float4* rec,
                                          const float4* __restrict__ dl, float rc2, int mlo, int64_t s, int p, int ei,
                                          const float4& me, uint64_t b0, uint64_t b1, Acc& acc, OtherM& oth) {
  const Rsrc rr = rsrcBelow(rec, O.lo);
  const Rsrc rtab = rsrcAt(reinterpret_cast<uintptr_t>(tb.pairZ));
  const Rsrc rtabD = rsrcAt(reinterpret_cast<uintptr_t>(tb.rhoD));
  const uint32_t o16 = static_cast<uint32_t>(s) * 16u;
  const uint32_t pairBase = static_cast<uint32_t>(ei * 3) * static_cast<uint32_t>(tb.nr);
  const uint32_t* sh = O.sh[p];
  const float4* D = dl + p * kMaxLatOffsets;
  // a group's entries past the mask's last offset get a lattice vector out
  // of range: beyond the cutoff, they add nothing
  forMaskGroupsFull<U>(b0, b1, [&](const int* ks, const bool* act) {
    float4 nb[U], d[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = act[u] ? ks[u] : kPadOffset;
      nb[u] = ldRec4(rr, o16, sh[k] * 16u);
      d[u] = D[k];
    }
    forceGroupM(me, me.w, ei, pairBase, nb, d, rc2, rtab, rtabD, tb, mlo, ks, acc, oth);
  });
  flushChunk3(acc);
}

template <int ACC, int MODE, int U>
__global__ __launch_bounds__(kBlock) void kForceM(Geom G, LatOffsets O, Tables<float> tb, CXPtr x, XPtr xn,
                                                  const int8_t* __restrict__ type, const float4* __restrict__ rec,
                                                  float4* __restrict__ recn, const float4* __restrict__ dl,
                                                  const uint64_t* __restrict__ wmask, XPtr v, XPtr f,
                                                  const uint64_t* __restrict__ id, VerletParams vp, StageArgs st,
                                                  Ctl* ctl, InterView iv, InterDev in, int mlo) {
  unsigned long long vb = 0;  // |v|^2 bits after the secondstep (MODE 0)
  unsigned long long db = 0;  // |dx|^2 bits of the drift (MODE 1)
  if (blockIdx.x < frontBlocks(G)) {
    interForceBody<float, MODE>(G, tb, iv, x, type, reinterpret_cast<const float*>(rec) + 3, 4, in, vp, frontWave(),
                                frontWaves(G));
    return;
  }
  const uint32_t b = blockIdx.x - frontBlocks(G);
  [&] {
    int64_t s;
    int p, cx, cy, cz;
    if (!siteOfBlock(G, b, threadIdx.x, s, p, cx, cy, cz)) return;
    const int8_t ti = type[s];
    if (isVacant(ti)) {  // vacancy: keeps its stale position (atom.cpp:43-47)
      vacancyForceM<MODE>(G, s, p, cx, cy, cz, x, xn, recn, f);
      return;
    }
    const int ei = species(ti);
    const float4 me = rec[s];
    Sum3<ACC> acc;
    OtherM oth;
    // the offsets the density pass found in range for some lane of this wavefront
    const uint32_t wv = waveId(b);
    forceSumM<U>(O, tb, rec, dl, static_cast<float>(G.rc2), mlo, s, p, ei, me, uniform64(wmask[2 * wv]),
                 uniform64(wmask[2 * wv + 1]), acc, oth);
    addOther3(acc, oth);
    forceTailM<ACC, MODE>(G, s, p, cx, cy, cz, ti, ei, me.w, acc, x, xn, type, rec, recn, v, f, id, vp, st, ctl, tb,
                          iv, vb, db);
  }();
  if (MODE == 0 && vp.vmax) waveMaxTo(vb, vp.vmax);
  if (MODE == 1) waveMaxTo(db, &ctl->dispmax2);
}

// The mixed force pass with four wavefronts to 64 sites (boxes with few
// sites): the chunk sums of a site meet in LDS, and the first wavefront takes
// them in order.
template <int ACC, int MODE, int U>
__global__ __launch_bounds__(kBlock) void kForceMP(Geom G, LatOffsets O, Tables<float> tb, CXPtr x, XPtr xn,
                                                   const int8_t* __restrict__ type, const float4* __restrict__ rec,
                                                   float4* __restrict__ recn, const float4* __restrict__ dl,
                                                   const uint64_t* __restrict__ wmask, XPtr v, XPtr f,
                                                   const uint64_t* __restrict__ id, VerletParams vp, StageArgs st,
                                                   Ctl* ctl, InterView iv, InterDev in, int mlo) {
  using Term = typename Sum3<ACC>::Term;
  __shared__ Term chunks[kChunks][3][64];
  __shared__ WaveSumsM others[3];
  __shared__ TailHits hits;
  if (blockIdx.x < frontBlocks(G)) {
    interForceBody<float, MODE>(G, tb, iv, x, type, reinterpret_cast<const float*>(rec) + 3, 4, in, vp, frontWave(),
                                frontWaves(G));
    return;
  }
  const SharedSite q = sharedSite(G, type, blockIdx.x - frontBlocks(G));
  const int lane = static_cast<int>(threadIdx.x & 63u);
  const int ei = species(q.ti);
  float4 me = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  OtherM oth;
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int k = 0; k < 3; ++k) chunks[4 * q.rg + t][k][lane] = 0;
  if (!isVacant(q.ti)) {
    me = rec[q.s];
    ChunkSums<ACC> sums;
    sums.chunk = 4 * q.rg;
    sums.out = chunks;
    uint64_t b0, b1;
    rangeBits(wmask, q.wv, q.rg, b0, b1);
    forceSumM<U>(O, tb, rec, dl, static_cast<float>(G.rc2), mlo, q.s, q.p, ei, me, b0, b1, sums, oth);
  }
  if (q.rg > 0) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      others[q.rg - 1].hi[c][lane] = oth.hi(c);
      others[q.rg - 1].lo[c][lane] = oth.lo[c];
    }
  }
  findTailHits(hits, q.rg, iv, x.c, type, G.rc2, q.p, q.s, q.ti);
  __syncthreads();
  if (q.rg > 0) return;
  unsigned long long vb = 0, db = 0;
  if (q.site && isVacant(q.ti)) {
    vacancyForceM<MODE>(G, q.s, q.p, q.cx, q.cy, q.cz, x, xn, recn, f);
  } else if (q.site) {
    Sum3<ACC> acc;
    for (int t = 0; t < kChunks; ++t) {
      acc.g0 = chunks[t][0][lane];
      acc.g1 = chunks[t][1][lane];
      acc.g2 = chunks[t][2][lane];
      acc.flush();
    }
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int c = 0; c < 3; ++c) oth.join(c, others[r].hi[c][lane], others[r].lo[c][lane]);
    addOther3(acc, oth);
    forceTailM<ACC, MODE>(G, q.s, q.p, q.cx, q.cy, q.cz, q.ti, ei, me.w, acc, x, xn, type, rec, recn, v, f, id, vp,
                          st, ctl, tb, iv, vb, db, &hits);
  }
  if (MODE == 0 && vp.vmax) waveMaxTo(vb, vp.vmax);
  if (MODE == 1) waveMaxTo(db, &ctl->dispmax2);
}

// The byte shift of a neighbour's record from the w of its offset's table
// entry: the shift itself, or a packed delta that a box turns into its own
// shift (scalar arithmetic where the entry was read by a scalar load).
struct RecShift {
  __device__ __forceinline__ uint32_t operator()(float w) const { return __float_as_uint(w); }
};
struct PackedShift {
  int32_t plane, NX, NY, lo;
  __device__ __forceinline__ uint32_t operator()(float w) const {
    const uint32_t u = __float_as_uint(w);
    const int32_t dp = static_cast<int8_t>(u & 0xffu), dz = static_cast<int8_t>((u >> 8) & 0xffu);
    const int32_t dy = static_cast<int8_t>((u >> 16) & 0xffu), dcx = static_cast<int8_t>(u >> 24);
    return static_cast<uint32_t>(dp * plane + (dz * NY + dy) * NX + dcx - lo) * 16u;
  }
};

// One virtual block of the LDS force pass (block b of a box): per site the
// same pairs and sums as kForceM.  dl holds, per pruned offset of either
// parity, the lattice vector and in w what shift(w) turns into the byte shift
// of the neighbour's record (RecShift, PackedShift), for scalar loads, and
// offT the same in LDS, for the lanes that work off noted pairs.  The next
// group's records are on their way while a group is computed: four
// wavefronts per SIMD do not cover their round trip.  Every lane of a wavefront with an
// atom stays to the end of the loop, since the noted pairs are worked off by
// the whole wavefront: a lane without an atom sits out of every cutoff.
template <int ACC, int MODE, int U, typename Shift>
__device__ __forceinline__ void forceVBlockL(const Geom& G, const LatOffsets& O, const Tables<float>& tb, CXPtr x,
                                             XPtr xn, const int8_t* __restrict__ type,
                                             const float4* __restrict__ rec, float4* __restrict__ recn,
                                             const uint64_t* __restrict__ wmask, XPtr v, XPtr f,
                                             const uint64_t* __restrict__ id, const VerletParams& vp,
                                             const StageArgs& st, Ctl* ctl, const InterView& iv, const float4* dl,
                                             const float4* offT, const float4* knT, int mlo, WaveQueueM& wq, WaveSumsM& ws, uint32_t b,
                                             uint32_t tl, Shift shift, unsigned long long& vb,
                                             unsigned long long& db) {
  int64_t s = 0;
  int p = 0, cx = 0, cy = 0, cz = 0;
  const bool site = siteOfBlock(G, b, tl, s, p, cx, cy, cz);
  int8_t ti = kVacant;
  if (site) {
    ti = type[s];
    if (isVacant(ti)) vacancyForceM<MODE>(G, s, p, cx, cy, cz, x, xn, recn, f);  // keeps its stale position
  }
  const bool live = !isVacant(ti);
  const uint64_t lives = __ballot(live);
  if (!lives) return;
  const Rsrc rr = rsrcBelow(rec, O.lo);
  const Rsrc rtab = rsrcAt(reinterpret_cast<uintptr_t>(tb.pairZ));
  const Rsrc rtabD = rsrcAt(reinterpret_cast<uintptr_t>(tb.rhoD));
  const float rc2 = static_cast<float>(G.rc2);
  const int ei = live ? species(ti) : 0;
  float4 me = make_float4(kNoAtom, kNoAtom, kNoAtom, 0.0f);
  if (live) me = rec[s];
  const uint32_t o16 = addressOfLives(static_cast<uint32_t>(s) * 16u, live, lives);
  const float dfi = me.w;
  const uint32_t pu = __builtin_amdgcn_readfirstlane((b >> 3) & 1u) * kMaxLatOffsets;
  const float4* T = offT + pu;
  const f32x4* dlp = reinterpret_cast<const f32x4*>(dl) + pu;
  Sum3<ACC> acc;
  const uint32_t wv = b * (kBlock / 64) + __builtin_amdgcn_readfirstlane(tl >> 6);
  uint64_t b0 = uniform64(wmask[2 * wv]), b1 = uniform64(wmask[2 * wv + 1]);
  int left = __builtin_popcountll(b0) + __builtin_popcountll(b1), base = 0;
  int groups = (left + U - 1) / U;
  int qn = 0;
  bool sums = false;
  // The next U offsets and their records' loads.  Entries past the mask's
  // last offset get a lattice vector out of range: beyond the cutoff, they
  // add nothing.
  struct Group {
    int ks[U];
    f32x4 d[U];
    float4 nb[U];
  } g, h;
  int k = 0;
  auto fetch = [&](Group& q) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (b0 == 0) {  // on to the mask's second word
        b0 = b1;
        b1 = 0;
        base = 64;
      }
      const bool act = u < left;
      const int t = __builtin_ctzll(b0 | (1ull << 63));
      b0 &= ~(1ull << t);
      k = act ? base + t : k;
      q.ks[u] = k;
      q.d[u] = scalarRead(dlp + (act ? k : kPadOffset));
    }
    left -= U;
#pragma unroll
    for (int u = 0; u < U; ++u) q.nb[u] = ldRec4(rr, o16, shift(q.d[u].w));
  };
  auto drain = [&](int least) {
    while (qn >= least) {
      if (!sums) {
        sums = true;
        for (int c = 0; c < 3; ++c) {
          ws.hi[c][threadIdx.x & 63u] = 0.0;
          ws.lo[c][threadIdx.x & 63u] = 0;
        }
      }
      waveLdsFence();
      const int n = qn < 64 ? qn : 64;
      drainQueueM(wq.q + (qn - n), n, me, o16, rr, rtab, rtabD, tb, T, shift, ws);
      qn -= n;
    }
  };
  fetch(g);  // also past the last group: the loads of the site's own record
  while (groups > 0) {
    fetch(h);
    forceGroupL<ACC, U>(me, dfi, ei, g.nb, g.d, rc2, tb, knT, mlo, g.ks, acc, wq, qn);
    fetch(g);
    if (groups > 1) forceGroupL<ACC, U>(me, dfi, ei, h.nb, h.d, rc2, tb, knT, mlo, h.ks, acc, wq, qn);
    groups -= 2;
    drain(groups > 0 ? 64 : 1);
  }
  flushChunk3(acc);
  OtherM oth;
  if (sums) {
    waveLdsFence();
    for (int c = 0; c < 3; ++c) oth.join(c, ws.hi[c][threadIdx.x & 63u], ws.lo[c][threadIdx.x & 63u]);
  }
  if (!live) return;
  addOther3(acc, oth);
  unsigned long long vbs = 0, dbs = 0;
  forceTailM<ACC, MODE>(G, s, p, cx, cy, cz, ti, ei, dfi, acc, x, xn, type, rec, recn, v, f, id, vp, st, ctl, tb,
                        iv, vbs, dbs);
  vb = vbs > vb ? vbs : vb;
  db = dbs > db ? dbs : db;
}

// One virtual block of the gather form of the LDS force pass: per site the same
// pairs and sums as kForceM, the Fe-Fe segments from knot `first` on from LDS
// (forceGroupG), as are the offsets' lattice vectors (offT).
template <int ACC, int MODE, int U, typename Shift>
__device__ __forceinline__ void forceVBlockG(const Geom& G, const LatOffsets& O, const Tables<float>& tb, CXPtr x,
                                             XPtr xn, const int8_t* __restrict__ type,
                                             const float4* __restrict__ rec, float4* __restrict__ recn,
                                             const uint64_t* __restrict__ wmask, XPtr v, XPtr f,
                                             const uint64_t* __restrict__ id, const VerletParams& vp,
                                             const StageArgs& st, Ctl* ctl, const InterView& iv, const float4* offT,
                                             const float4* knT, int mlo, int first, uint32_t b, uint32_t tl,
                                             Shift shift, unsigned long long& vb, unsigned long long& db) {
  int64_t s;
  int p, cx, cy, cz;
  if (!siteOfBlock(G, b, tl, s, p, cx, cy, cz)) return;
  const int8_t ti = type[s];
  if (isVacant(ti)) {  // vacancy: keeps its stale position (atom.cpp:43-47)
    vacancyForceM<MODE>(G, s, p, cx, cy, cz, x, xn, recn, f);
    return;
  }
  const Rsrc rr = rsrcBelow(rec, O.lo);
  const float rc2 = static_cast<float>(G.rc2);
  const int ei = species(ti);
  const float4 me = rec[s];
  const uint32_t o16 = static_cast<uint32_t>(s) * 16u;
  const uint32_t pairBase = static_cast<uint32_t>(ei * 3) * static_cast<uint32_t>(tb.nr);
  const float4* T = offT + p * kMaxLatOffsets;
  Sum3<ACC> acc;
  OtherM oth;
  const uint32_t wv = b * (kBlock / 64) + __builtin_amdgcn_readfirstlane(tl >> 6);
  // a group's entries past the mask's last offset get a lattice vector out
  // of range: beyond the cutoff, they add nothing
  forMaskGroupsFull<U>(uniform64(wmask[2 * wv]), uniform64(wmask[2 * wv + 1]), [&](const int* ks, const bool* act) {
    float4 nb[U], d[U];
#pragma unroll
    for (int u = 0; u < U; ++u) d[u] = T[act[u] ? ks[u] : kPadOffset];
#pragma unroll
    for (int u = 0; u < U; ++u) nb[u] = ldRec4(rr, o16 + shift(d[u].w), 0);
    forceGroupG(me, ei, pairBase, nb, d, rc2, tb, knT, mlo, first, ks, acc, oth);
  });
  flushChunk3(acc);
  addOther3(acc, oth);
  unsigned long long vbs = 0, dbs = 0;
  forceTailM<ACC, MODE>(G, s, p, cx, cy, cz, ti, ei, me.w, acc, x, xn, type, rec, recn, v, f, id, vp, st, ctl, tb,
                        iv, vbs, dbs);
  vb = vbs > vb ? vbs : vb;
  db = dbs > db ? dbs : db;
}

// The LDS knots of the force pass, the Fe-Fe r*phi cubics from knot mlo on and
// SLOPES entries further the Fe density slope cubics (one block fills them).
template <int SLOPES = kKnotsM>
__device__ __forceinline__ void fillKnots(const Tables<float>& tb, float4* knT, int mlo, int nkn) {
  const float4* z4 = reinterpret_cast<const float4*>(tb.pairZ);  // row (Fe, Fe) is the first
  const float4* s4 = reinterpret_cast<const float4*>(tb.rhoD);   // row Fe is the first
  for (int i = threadIdx.x; i < nkn; i += kBlockP) {
    knT[i] = z4[mlo + i];
    knT[SLOPES + i] = s4[mlo + i];
  }
}

// The mixed force pass in persistent blocks, one per compute unit, that hold
// in LDS the lattice vector and record shift of every pruned offset (read as
// one broadcast per offset), the Fe-Fe r*phi cubics and the Fe density slope
// cubics from knot mlo on (one block fills them once).  Per site the same
// pairs, in the same order and with the same rounding, as kForceM.
// 2M atoms with the fused half steps 308 -> 303 us, 16M-atom cascade 2.44 -> 2.35
// ms, against segments re-read under a mask, one group in flight and the two
// cubics side by side in LDS (280 and 2.24 while the terms of the queued pairs
// were rounded to 2^-36 eV/A on the way).  Its VALU issue (70 % of the cycles,
// 3,990 instructions per 64 sites), the texture-data units (86 % busy) and its LDS
// reads (43 %, half of that bank conflicts) bound it together.
template <int ACC, int MODE, int U>
__global__ __launch_bounds__(kBlockP) void kForceL(Geom G, LatOffsets O, Tables<float> tb, CXPtr x, XPtr xn,
                                                   const int8_t* __restrict__ type, const float4* __restrict__ rec,
                                                   float4* __restrict__ recn, const float4* __restrict__ dl,
                                                   const uint64_t* __restrict__ wmask, XPtr v, XPtr f,
                                                   const uint64_t* __restrict__ id, VerletParams vp, StageArgs st,
                                                   Ctl* ctl, InterView iv, InterDev in, int mlo, int nkn,
                                                   unsigned long long* zwork) {
  __shared__ float4 offT[2 * kMaxLatOffsets];  // {lattice vector, record shift * 16}
  __shared__ WaveQueueM queues[kBlockP / 64];
  __shared__ WaveSumsM sums[kBlockP / 64];
  extern __shared__ float4 knT[];  // Fe-Fe r*phi cubics, Fe density slope cubics (fillKnots)
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (int i = threadIdx.x; i < 2 * kMaxLatOffsets; i += kBlockP) offT[i] = dl[2 * kMaxLatOffsets + i];
  fillKnots(tb, knT, mlo, nkn);
  __syncthreads();
  unsigned long long vb = 0;  // |v|^2 bits after the secondstep (MODE 0), largest over the lane's sites
  unsigned long long db = 0;  // |dx|^2 bits of the drift (MODE 1), likewise
  const RecShift shift;
  interForceBody<float, MODE>(G, tb, iv, x, type, reinterpret_cast<const float*>(rec) + 3, 4, in, vp,
                              static_cast<int>(wave * gridDim.x + blockIdx.x),
                              static_cast<int>(gridDim.x) * (kBlockP / 64));
  forVirtualBlocks(G, [&](uint32_t b, uint32_t tl) {
    const long long t0 = zwork ? clock64() : 0;
    forceVBlockL<ACC, MODE, U>(G, O, tb, x, xn, type, rec, recn, wmask, v, f, id, vp, st, ctl, iv, dl + 2 * kMaxLatOffsets,
                               offT, knT, mlo, queues[wave], sums[wave], b, tl, shift, vb, db);
    if (zwork) addPlaneWork(G, zwork, b, tl, t0);
  });
  if (MODE == 0 && vp.vmax) waveMaxTo(vb, vp.vmax);
  if (MODE == 1) waveMaxTo(db, &ctl->dispmax2);
}

// The box record that is a kernel's first argument, read from the argument
// segment where it is used.  Arguments by value are loaded at the start and
// keep scalar registers to their last use; in kForceLG they left too few for
// the lane masks of the loop over the pairs, which then spilled to lanes (twice
// the instructions).
__device__ __forceinline__ const BatchBox& boxArgument() {
  auto p = (const __attribute__((address_space(4))) BatchBox*)__builtin_amdgcn_kernarg_segment_ptr();
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" : "+s"(p));
#endif
  return *(const BatchBox*)p;
}

// kForceL's gather form, for boxes with many pairs that are not held: the
// masked gathers of forceGroupG in place of the queue, whose room in LDS holds
// knots instead (4,988, from 0.01 A on where the table has 5000 over 5.6 A).
template <int ACC, int MODE, int U>
__global__ __launch_bounds__(kBlockP) void kForceLG(BatchBox, int mlo, int first, int nkn,
                                                    unsigned long long* zwork) {
  __shared__ float4 offT[2 * kMaxLatOffsets];
  extern __shared__ float4 knT[];
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  {
    const BatchBox& B = boxArgument();
    const int c = B.cur;
    for (int i = threadIdx.x; i < 2 * kMaxLatOffsets; i += kBlockP) offT[i] = B.dl[2 * kMaxLatOffsets + i];
    fillKnots<kKnotsG>(B.t32, knT, first, nkn);
    interForceBody<float, MODE>(B.G, B.t32, B.iv, cxp(B.x[c]), B.type, reinterpret_cast<const float*>(B.rec[c]) + 3,
                                4, B.in, B.vp, static_cast<int>(wave * gridDim.x + blockIdx.x),
                                static_cast<int>(gridDim.x) * (kBlockP / 64));
  }
  __syncthreads();
  unsigned long long vb = 0, db = 0;
  const RecShift shift;
  forVirtualBlocks(boxArgument().G, [&](uint32_t b, uint32_t tl) {
    const long long t0 = zwork ? clock64() : 0;
    const BatchBox& B = boxArgument();
    const int c = B.cur;
    forceVBlockG<ACC, MODE, U>(B.G, B.O, B.t32, cxp(B.x[c]), xp(B.x[1 - c]), B.type, B.rec[c], B.rec[1 - c], B.wmask,
                               xp(B.v), xp(B.f), B.id, B.vp, B.st, B.ctl, B.iv, offT, knT, mlo, first, b, tl, shift, vb, db);
    if (zwork) addPlaneWork(B.G, zwork, b, tl, t0);
  });
  const BatchBox& B = boxArgument();
  if (MODE == 0 && B.vp.vmax) waveMaxTo(vb, B.vp.vmax);
  if (MODE == 1) waveMaxTo(db, &B.ctl->dispmax2);
}

// Walks the virtual blocks of a batch's persistent launch: on each XCD those of
// box 0, then box 1, ...  body(box, block of the box, thread, maxima).
template <int MODE, typename Body>
__device__ __forceinline__ void forBatchBlocks(const BatchBox* __restrict__ boxes, const uint32_t* vstart, int nbox,
                                               Body body) {
  constexpr uint32_t V = kBlockP / kBlock;
  const uint32_t c = blockIdx.x & 7u, q = blockIdx.x >> 3, Q = gridDim.x >> 3;
  const uint32_t sub = __builtin_amdgcn_readfirstlane(threadIdx.x / kBlock);
  const uint32_t tl = threadIdx.x % kBlock;
  const uint32_t nvb = vstart[nbox];
  unsigned long long vb = 0, db = 0;
  int lastBox = -1;
  const auto close = [&] {  // the maxima go to the box they came from
    if (lastBox < 0) return;
    if (MODE == 0 && boxes[lastBox].vp.vmax) waveMaxTo(vb, boxes[lastBox].vp.vmax);
    if (MODE == 1) waveMaxTo(db, &boxes[lastBox].ctl->dispmax2);
  };
  for (uint32_t k = q * V + sub; k < nvb; k += Q * V) {
    const int bi = boxOfBlock(vstart, nbox, k);
    if (bi != lastBox) {
      close();
      vb = db = 0;
      lastBox = bi;
    }
    body(boxes[bi], c + 8u * (k - vstart[bi]), tl, vb, db);
  }
  close();
}

// The LDS force pass of every box of a batch in one persistent launch: on
// each XCD the blocks walk the virtual blocks of box 0, then box 1, ...
// (vstart[b] counts the virtual blocks per XCD before box b).  All boxes
// share the potential (the knots in LDS) and the pruned offsets (lattice
// vectors and packed deltas in dlp, 2 x kMaxLatOffsets); each turns a
// packed delta into its own record shift.
template <int ACC, int MODE, int U>
__global__ __launch_bounds__(kBlockP) void kForceLB(const BatchBox* __restrict__ boxes, const uint32_t* vstart,
                                                    int nbox, int flip, const float4* __restrict__ dlp, int mlo,
                                                    int nkn) {
  __shared__ float4 offT[2 * kMaxLatOffsets];
  __shared__ WaveQueueM queues[kBlockP / 64];
  __shared__ WaveSumsM sums[kBlockP / 64];
  extern __shared__ float4 knT[];
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (int i = threadIdx.x; i < 2 * kMaxLatOffsets; i += kBlockP) offT[i] = dlp[i];
  fillKnots(boxes[0].t32, knT, mlo, nkn);
  __syncthreads();
  forBatchBlocks<MODE>(boxes, vstart, nbox, [&](const BatchBox& B, uint32_t b, uint32_t tl, unsigned long long& vb,
                                                unsigned long long& db) {
    const int cb = B.cur ^ flip;
    const PackedShift shift{static_cast<int32_t>(B.G.plane), B.G.NX, B.G.NY, B.O.lo};
    forceVBlockL<ACC, MODE, U>(B.G, B.O, B.t32, cxp(B.x[cb]), xp(B.x[1 - cb]), B.type, B.rec[cb], B.rec[1 - cb],
                               B.wmask, xp(B.v), xp(B.f), B.id, B.vp, B.st, B.ctl, B.iv, dlp, offT, knT, mlo,
                               queues[wave], sums[wave], b, tl, shift, vb, db);
  });
}
// Its gather form (forceVBlockG).
template <int ACC, int MODE, int U>
__global__ __launch_bounds__(kBlockP) void kForceLGB(const BatchBox* __restrict__ boxes, const uint32_t* vstart,
                                                     int nbox, int flip, const float4* __restrict__ dlp, int mlo,
                                                     int first, int nkn) {
  __shared__ float4 offT[2 * kMaxLatOffsets];
  extern __shared__ float4 knT[];
  for (int i = threadIdx.x; i < 2 * kMaxLatOffsets; i += kBlockP) offT[i] = dlp[i];
  fillKnots<kKnotsG>(boxes[0].t32, knT, first, nkn);
  __syncthreads();
  forBatchBlocks<MODE>(boxes, vstart, nbox, [&](const BatchBox& B, uint32_t b, uint32_t tl, unsigned long long& vb,
                                                unsigned long long& db) {
    const int cb = B.cur ^ flip;
    const PackedShift shift{static_cast<int32_t>(B.G.plane), B.G.NX, B.G.NY, B.O.lo};
    forceVBlockG<ACC, MODE, U>(B.G, B.O, B.t32, cxp(B.x[cb]), xp(B.x[1 - cb]), B.type, B.rec[cb], B.rec[1 - cb],
                               B.wmask, xp(B.v), xp(B.f), B.id, B.vp, B.st, B.ctl, B.iv, offT, knT, mlo, first, b, tl,
                               shift, vb, db);
  });
}

// Offsets a group in the FP64 force passes.
constexpr int kUDouble = 2;

// LDS of the mixed force pass: kKnotsM knots (mixed_site.hpp) beside the
// kernel's static LDS (the offset table, 4 KB, the queues, 18 KB, and the sums
// of the pairs set aside, 36 KB) in the 160 KB of a compute unit.
constexpr int kForceLdsBytes = 32 * kKnotsM;
static_assert(kForceLdsBytes + 2 * kMaxLatOffsets * 16 +
                      static_cast<int>(kBlockP / 64 * (sizeof(WaveQueueM) + sizeof(WaveSumsM))) <=
                  160 * 1024,
              "the LDS of one block per compute unit");
struct LdsKnots {
  int mlo, nkn;
  size_t bytes;
};
LdsKnots ldsKnotsForce(int nr) {
  LdsKnots k;
  k.nkn = std::min(nr, kKnotsM);
  k.mlo = nr - k.nkn;
  k.bytes = kForceLdsBytes;
  return k;
}
// The FP64 pass's LDS knots, 40 bytes each (KnotsD), from knot mlo to the
// last, beside its queues (6 KB) and sums (24 KB): 3325 knots, from 1.88 A on
// where the table has 5000 over 5.6 A.
constexpr int kForceLdsBytesD =
    160 * 1024 - static_cast<int>(kBlockP / 64 * (sizeof(WaveQueueD<kUDouble>) + sizeof(WaveSums))) - 64;
LdsKnots ldsKnotsForceD(int nr) {
  LdsKnots k;
  k.nkn = std::min(nr, (kForceLdsBytesD - 16) / 40);
  k.mlo = nr - k.nkn;
  k.bytes = static_cast<size_t>(40) * static_cast<size_t>(k.nkn) + 16;
  return k;
}
// The FP64 density pass's LDS knots, 32 bytes each, beside its queues and
// sums: 4670 knots, from 0.37 A on where the table has 5000 over 5.6 A.
constexpr int kURhoD = 2;
constexpr int kRhoLdsBytesD =
    160 * 1024 - static_cast<int>(kBlockP / 64 * (sizeof(WaveQueueD<kURhoD>) + sizeof(WaveSum1))) - 64;
LdsKnots ldsKnotsRhoD(int nr) {
  LdsKnots k;
  k.nkn = std::min(nr, kRhoLdsBytesD / 32);
  k.mlo = nr - k.nkn;
  k.bytes = static_cast<size_t>(32) * static_cast<size_t>(k.nkn);
  return k;
}
// The energy pass's LDS knots: 7 doubles (56 bytes) a knot beside its static
// LDS (the block sums; 512 bytes are kept).
constexpr int kEnergyLdsBytes = 160 * 1024 - 512;
LdsKnots ldsKnotsEnergy(int nr) {
  LdsKnots k;
  k.nkn = std::min(nr, kEnergyLdsBytes / 56);
  k.mlo = nr - k.nkn;
  k.bytes = static_cast<size_t>(56) * static_cast<size_t>(k.nkn);
  return k;
}
// The FP64 force pass's gather form: the same 7 doubles a knot.
constexpr int kForceLdsBytesDG = kEnergyLdsBytes;
LdsKnots ldsKnotsForceDG(int nr) { return ldsKnotsEnergy(nr); }
// The mixed force pass's gather form: kKnotsG knots beside the offset table.
constexpr int kForceLdsBytesG = 32 * kKnotsG;
static_assert(kForceLdsBytesG + 2 * kMaxLatOffsets * 16 <= 160 * 1024, "the LDS of one block per compute unit");
LdsKnots ldsKnotsForceG(int nr) {
  LdsKnots k;
  k.nkn = std::min(nr, kKnotsG);
  k.mlo = nr - k.nkn;
  k.bytes = kForceLdsBytesG;
  return k;
}
bool setLdsBytes(const void* fn, int bytes) {
  return hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) == hipSuccess;
}
// One persistent block per compute unit, a whole number per XCD.
unsigned persistentGrid(const DevState& s) { return static_cast<unsigned>(s.ncu / 8 * 8); }
// The LDS-table passes: on request, or by default where the sites fill the
// persistent launch, 16 wavefronts a compute unit, one and a quarter times.  Just
// above once, its second round is nearly empty.  Step FP64 / mixed, with LDS
// against without: 60^3 cells, 1.65 times, 206/304 and 142/174 us, 6 % solutes
// 277/340 and 165/188; 56^3, 1.34 times, 208/247 and 139/149, 6 % 275/279 and
// 158/155; 52x51x53, 1.07 times, 205/213 and 131/126, 6 % 277/246 and 151/135.
bool fillsLaunch(const DevState& s, double times) {
  return static_cast<double>(siteGrid(s.G)) * kBlock >= times * persistentGrid(s) * kBlockP;
}
bool useLds(const DevState& s) {
  if (s.ncu < 8 || s.lds == kLdsOff) return false;
  return s.lds == kLdsOn || fillsLaunch(s, 1.25);
}
// Which form: by the share of pairs whose segments LDS does not hold, those
// with a solute and, where the knots held begin beyond the nearest neighbours,
// the like pairs below them.  The queue wins while they are few, masked gathers
// beyond, and the pass from global memory where next to nothing is held.
// 108^3 cells (2.5M atoms), 300 K, us with queue / gathers / neither, by
// solutes and by knots over 5.6 A (80^3 crosses over at the same shares):
//                      5000             10000             20000
//   FP64    0 %   505/ 537/ 986    718/ 626/1034   1203/1035/1077
//         1.5 %   665/ 781/1083    988/ 865/1161   1397/1236/1299
//           6 %   844/ 814/1131   1153/ 913/1222   1540/1349/1401
//          15 %  1122/ 857/1197   1389/1008/1314   1735/1591/1590
//          25 %  1394/ 945/1252   1641/1222/1396   1931/1793/1770
//          60 %  2000/1474/1403   2137/1721/1555   2333/2149/2055
//   mixed   0 %   313/ 311/ 435    463/ 358/ 533    743/ 475/ 778
//         1.5 %   373/ 445/ 498    516/ 459/ 594    796/ 566/ 815
//           6 %   448/ 467/ 531    585/ 494/ 675    916/ 647/ 903
//          15 %   572/ 491/ 622    749/ 545/ 834   1099/ 781/1054
//          60 %  1092/ 761/ 931   1358/ 950/1176   1597/1198/1377
//         100 %  (80^3)  - / 313/ 284
// A batch of 15 boxes, mixed, us a step with queue / gathers: 332/354 at 1.5 %,
// 354/365 at 6, 380/367 at 10, 586/483 at 60; 406/388 on 10000 knots.
double unheld(double solutes, double near) {
  const double like = (1.0 - solutes) * (1.0 - solutes);
  return 1.0 - like * (1.0 - near);
}
constexpr double kQueueShareD = 0.08, kGatherShareD = 0.83, kQueueShareM = 0.145, kGatherShareM = 0.985;
LdsForm forceForm(const DevState& s, bool mixed) {
  if (!useLds(s)) return kLdsNone;
  if (s.lds == kLdsOn) return kLdsQueue;
  if (unheld(s.solutes, mixed ? s.nearM : s.nearD) <= (mixed ? kQueueShareM : kQueueShareD))
    return kLdsQueue;
  if (mixed) return unheld(s.solutes, 0.0) <= kGatherShareM ? kLdsGather : kLdsNone;
  // With half of the pairs or more gathered, FP64 gains some 8 %, which a last
  // round of few blocks takes back: 56^3 cells, 1.3 rounds, 20000 knots 301 us a
  // step against 281 without LDS.
  const double share = unheld(s.solutes, s.nearDG);
  return share <= 0.5 || (share <= kGatherShareD && fillsLaunch(s, 2.0)) ? kLdsGather : kLdsNone;
}
// The FP64 density pass has no gather form: LDS cubics and queue against
// neither, by solutes, the same boxes: 0 % 380/553 us, 6 % 506/575, 15 %
// 597/598; 10000 knots 0 % 564/616, 1.5 % 656/629; 20000 knots 744/716.
constexpr double kQueueShareRho = 0.13;
bool rhoLdsPays(const DevState& s) {
  return s.lds == kLdsOn || s.solutes + (1.0 - s.solutes) * 0.5 * s.nearRhoD <= kQueueShareRho;
}

// Boxes whose sites fill at most this many wavefronts (64 sites each) take the
// passes that share 64 sites among four wavefronts.
constexpr int64_t kSharedWaves = 4096;
bool useShared(const DevState& s) {
  return static_cast<int64_t>(siteGrid(s.G)) * (kBlock / 64) <= kSharedWaves;
}

}  // namespace

void setNearShares(DevState& s, const std::vector<double>& lengths, double rc, int nr, double dr) {
  // a shell counts in proportion where the first knot lies within 0.15 A of it
  const auto share = [&](int mlo) {
    double below = 0.0, all = 0.0;
    for (const double len : lengths) {
      if (len >= rc) continue;
      all += 1.0;
      below += std::min(1.0, std::max(0.0, (mlo * dr - len) / 0.3 + 0.5));
    }
    return all > 0.0 ? below / all : 0.0;
  };
  s.nearD = share(ldsKnotsForceD(nr).mlo);
  s.nearDG = share(ldsKnotsForceDG(nr).mlo);
  s.nearRhoD = share(ldsKnotsRhoD(nr).mlo);
  s.nearM = share(ldsKnotsForce(nr).mlo);
}

int launchRhoDf(const DevState& s, const LatOffsets& o, const Tables<double>& t64, const Tables<float>& t32,
                bool mixed, int acc, bool store_rho, bool scan, hipStream_t st) {
  double* rho = store_rho ? s.rho : nullptr;
  const bool shared = useShared(s);
  const unsigned grid = frontBlocks(s.G) + (shared ? 4 : 1) * siteGrid(s.G);
  const InterView iv = interView(s, mixed);
  const CXPtr x = cxp(s.x[s.cur]);
  const double rcs = std::sqrt(s.G.rc2) + s.skin;
  if (!mixed) {
    const Rec64 r64{s.pxy[s.cur], s.pzw[s.cur]};
    const LdsKnots lk = ldsKnotsRhoD(t64.nr);
    static const bool ldsReady = setLdsBytes(reinterpret_cast<const void*>(&kRhoDL<kURhoD>), kRhoLdsBytesD);
    // With the skin's masks kRhoDL against kRhoDf, whole pass: 60^3 cells 101
    // against 117 us, 100^3 372 against 483, with 6 % solutes at 900 K 60^3 123
    // against 134, 90^3 344 against 397; where every pass scans all offsets
    // (766 000 atoms) 257 against 238, so those stay with kRhoDf.
    if (useLds(s) && rhoLdsPays(s) && ldsReady && !scan && s.skin > 0.0) {
      kRhoDL<kURhoD><<<persistentGrid(s), kBlockP, lk.bytes, st>>>(s.G, o, t64, x, s.type, s.df64, rho, s.wmask,
                                                                   s.smask, rcs * rcs, iv, s.in, r64, lk.mlo, lk.nkn);
      return 2;
    }
    if (shared)
      kRhoDfP<4><<<grid, kBlock, 0, st>>>(s.G, o, t64, x, s.type, s.df64, rho, s.wmask, s.smask, rcs * rcs, iv, s.in,
                                          r64, lk.mlo);
    else
      kRhoDf<4><<<grid, kBlock, 0, st>>>(s.G, o, t64, x, s.type, s.df64, rho, s.wmask, s.smask, rcs * rcs, iv, s.in,
                                         r64, lk.mlo);
  } else if (shared) {
    const float rcs2 = static_cast<float>(rcs * rcs);
#define MISA_RHO_MP(A)                                                                                          \
  kRhoDfMP<A, 4><<<grid, kBlock, 0, st>>>(s.G, o, t32, x, s.type, s.rec[s.cur], s.dl, rho, s.wmask, s.smask, \
                                              rcs2, iv, s.in)
    if (acc == 0) MISA_RHO_MP(0);
    else if (acc == 1) MISA_RHO_MP(1);
    else MISA_RHO_MP(2);
#undef MISA_RHO_MP
  } else {
    const float rcs2 = static_cast<float>(rcs * rcs);
#define MISA_RHO_M(A, U)                                                                                   \
  kRhoDfM<A, U><<<grid, kBlock, 0, st>>>(s.G, o, t32, x, s.type, s.rec[s.cur], s.dl, rho, s.wmask, s.smask, \
                                        rcs2, iv, s.in)
    const bool u8 = s.uRho == 8;
    if (acc == 0) {
      if (u8) MISA_RHO_M(0, 8);
      else MISA_RHO_M(0, 4);
    } else if (acc == 1) {
      if (u8) MISA_RHO_M(1, 8);
      else MISA_RHO_M(1, 4);
    } else {
      if (u8) MISA_RHO_M(2, 8);
      else MISA_RHO_M(2, 4);
    }
#undef MISA_RHO_M
  }
  return mixed ? 1 : 0;
}

int launchForce(const DevState& s, const LatOffsets& o, const Tables<double>& t64, const Tables<float>& t32,
                bool mixed, int acc, int mode, const VerletParams& vp, hipStream_t st) {
  int kind = mixed ? 1 : 0;
  const bool shared = useShared(s);
  const unsigned grid = frontBlocks(s.G) + (shared ? 4 : 1) * siteGrid(s.G);
  const CXPtr x = cxp(s.x[s.cur]);
  const XPtr xn = xp(s.x[1 - s.cur]);
  const StageArgs sa = stageOf(s);
  const InterView iv = interView(s, mixed);
  const LdsForm form = forceForm(s, mixed);
  const LdsKnots lk = ldsKnotsForce(t32.nr), lg = ldsKnotsForceG(t32.nr);
  const LdsKnots lkd = ldsKnotsForceD(t64.nr), lgd = ldsKnotsForceDG(t64.nr);
#define MISA_FORCE(M)                                                                                         \
  do {                                                                                                        \
    static const bool queueReady =                                                                            \
        setLdsBytes(reinterpret_cast<const void*>(&kForceDL<M, kUDouble>), kForceLdsBytesD);                 \
    static const bool gatherReady =                                                                           \
        setLdsBytes(reinterpret_cast<const void*>(&kForceDG<M, kUDouble>), kForceLdsBytesDG);                \
    const Rec64 r64{s.pxy[s.cur], s.pzw[s.cur]}, rn64{s.pxy[1 - s.cur], s.pzw[1 - s.cur]};                   \
    if (form == kLdsQueue && queueReady) {                                                                    \
      kind = 3;                                                                                               \
      kForceDL<M, kUDouble><<<persistentGrid(s), kBlockP, lkd.bytes, st>>>(                                   \
          s.G, o, t64, x, xn, s.type, s.df64, s.wmask, xp(s.v), xp(s.f), s.id, vp, sa, s.ctl, iv, s.in, r64,   \
          rn64, lkd.mlo, lkd.nkn);                                                                            \
    } else if (form == kLdsGather && gatherReady) {                                                           \
      kind = 5;                                                                                               \
      kForceDG<M, kUDouble><<<persistentGrid(s), kBlockP, lgd.bytes, st>>>(                                   \
          s.G, o, t64, x, xn, s.type, s.df64, s.wmask, xp(s.v), xp(s.f), s.id, vp, sa, s.ctl, iv, s.in, r64,   \
          rn64, lkd.mlo, lgd.mlo, lgd.nkn);                                                                   \
    } else if (shared) {                                                                                      \
      kForceP<M, kUDouble><<<grid, kBlock, 0, st>>>(s.G, o, t64, x, xn, s.type, s.df64, s.wmask, xp(s.v), \
                                                    xp(s.f), s.id, vp, sa, s.ctl, iv, s.in, r64, rn64,    \
                                                    lkd.mlo);                                             \
    } else {                                                                                                  \
      kForce<M, kUDouble><<<grid, kBlock, 0, st>>>(s.G, o, t64, x, xn, s.type, s.df64, s.wmask, xp(s.v),      \
                                                   xp(s.f), s.id, vp, sa, s.ctl, iv, s.in, r64, rn64,         \
                                                   lkd.mlo);                                                  \
    }                                                                                                         \
  } while (0)
#define MISA_FORCE_MU(A, M, U)                                                                                \
  do {                                                                                                        \
    static const bool queueReady =                                                                            \
        setLdsBytes(reinterpret_cast<const void*>(&kForceL<A, M, U>), kForceLdsBytes);                       \
    static const bool gatherReady =                                                                           \
        setLdsBytes(reinterpret_cast<const void*>(&kForceLG<A, M, U>), kForceLdsBytesG);                     \
    if (form == kLdsQueue && queueReady) {                                                                    \
      kind = 2;                                                                                               \
      kForceL<A, M, U><<<persistentGrid(s), kBlockP, lk.bytes, st>>>(                                         \
          s.G, o, t32, x, xn, s.type, s.rec[s.cur], s.rec[1 - s.cur], s.dl, s.wmask, xp(s.v), xp(s.f), s.id, vp, \
          sa, s.ctl, iv, s.in, lk.mlo, lk.nkn, s.zmeasure ? s.zwork : nullptr);                                     \
    } else if (form == kLdsGather && gatherReady) {                                                           \
      kind = 4;                                                                                               \
      kForceLG<A, M, U><<<persistentGrid(s), kBlockP, lg.bytes, st>>>(                                        \
          boxOf(s, o, t32, iv, vp), lk.mlo, lg.mlo, lg.nkn, s.zmeasure ? s.zwork : nullptr);                  \
    } else if (shared) {                                                                                      \
      kForceMP<A, M, U><<<grid, kBlock, 0, st>>>(s.G, o, t32, x, xn, s.type, s.rec[s.cur],                \
                                                     s.rec[1 - s.cur], s.dl, s.wmask, xp(s.v), xp(s.f), s.id, vp, \
                                                     sa, s.ctl, iv, s.in, lk.mlo);                                  \
    } else {                                                                                                  \
      kForceM<A, M, U><<<grid, kBlock, 0, st>>>(s.G, o, t32, x, xn, s.type, s.rec[s.cur], s.rec[1 - s.cur],    \
                                                s.dl, s.wmask, xp(s.v), xp(s.f), s.id, vp, sa, s.ctl, iv, s.in, \
                                                lk.mlo);                                                        \
    }                                                                                                         \
  } while (0)
#define MISA_FORCE_M(A, M)            \
  do {                                \
    if (s.uForce == 2)                \
      MISA_FORCE_MU(A, M, 2);         \
    else                              \
      MISA_FORCE_MU(A, M, 4);         \
  } while (0)
  if (!mixed) {
    if (mode == 0) MISA_FORCE(0);
    else if (mode == 1) MISA_FORCE(1);
    else MISA_FORCE(2);
  } else if (acc == 0) {
    if (mode == 0) MISA_FORCE_M(0, 0);
    else if (mode == 1) MISA_FORCE_M(0, 1);
    else MISA_FORCE_M(0, 2);
  } else if (acc == 1) {
    if (mode == 0) MISA_FORCE_M(1, 0);
    else if (mode == 1) MISA_FORCE_M(1, 1);
    else MISA_FORCE_M(1, 2);
  } else {
    if (mode == 0) MISA_FORCE_M(2, 0);
    else if (mode == 1) MISA_FORCE_M(2, 1);
    else MISA_FORCE_M(2, 2);
  }
#undef MISA_FORCE
#undef MISA_FORCE_M
#undef MISA_FORCE_MU
  return kind;
}

int64_t launchEnergyPass(const DevState& s, const LatOffsets& o, const Tables<double>& t64, bool every,
                         hipStream_t st) {
  static const bool ldsReady = setLdsBytes(reinterpret_cast<const void*>(&kEnergyDL), kEnergyLdsBytes);
  const Rec64 r64{s.pxy[s.cur], s.pzw[s.cur]};
  const int all = every ? 1 : 0;
  if (useLds(s) && ldsReady && 3 * static_cast<int64_t>(persistentGrid(s)) <= s.npartials) {
    const LdsKnots lk = ldsKnotsEnergy(t64.nr);
    const unsigned grid = persistentGrid(s);
    kEnergyDL<<<grid, kBlockP, lk.bytes, st>>>(s.G, o, s.in.full, t64, cxp(s.x[s.cur]), s.type, s.rho, s.df64,
                                               s.smask, all, r64, s.partials, lk.mlo, lk.nkn);
    return grid;
  }
  const unsigned grid = siteGrid(s.G);  // 3 partials per block fit: the buffer holds 7 per site block
  kEnergyD<<<grid, kBlock, 0, st>>>(s.G, o, s.in.full, t64, cxp(s.x[s.cur]), s.type, s.rho, s.df64, s.smask, all,
                                    r64, s.partials);
  return grid;
}

void launchRhoDfBatch(const BatchBox* boxes, const uint32_t* rhoStart, int nbox, unsigned blocks, int acc,
                      int flip, hipStream_t st) {
  if (acc == 0) kRhoDfMB<0, 4><<<blocks, kBlock, 0, st>>>(boxes, rhoStart, nbox, flip);
  else if (acc == 1) kRhoDfMB<1, 4><<<blocks, kBlock, 0, st>>>(boxes, rhoStart, nbox, flip);
  else kRhoDfMB<2, 4><<<blocks, kBlock, 0, st>>>(boxes, rhoStart, nbox, flip);
}

LdsForm batchForceForm(double solutes, double nearM) {
  return unheld(solutes, nearM) <= kQueueShareM ? kLdsQueue : kLdsGather;
}

bool launchForceBatch(const BatchBox* boxes, const uint32_t* vstart, int nbox, const float4* dl, int nr, int ncu,
                      int acc, LdsForm form, int flip, hipStream_t st) {
  const LdsKnots lk = ldsKnotsForce(nr), lg = ldsKnotsForceG(nr);
  const unsigned grid = static_cast<unsigned>(ncu / 8 * 8);
#define MISA_FORCE_B(A)                                                                                      \
  do {                                                                                                       \
    static const bool queueReady =                                                                           \
        setLdsBytes(reinterpret_cast<const void*>(&kForceLB<A, 1, 4>), kForceLdsBytes);                      \
    static const bool gatherReady =                                                                          \
        setLdsBytes(reinterpret_cast<const void*>(&kForceLGB<A, 1, 4>), kForceLdsBytesG);                    \
    if (!queueReady || !gatherReady) return false;                                                           \
    if (form == kLdsQueue)                                                                                   \
      kForceLB<A, 1, 4><<<grid, kBlockP, lk.bytes, st>>>(boxes, vstart, nbox, flip, dl, lk.mlo, lk.nkn);      \
    else                                                                                                     \
      kForceLGB<A, 1, 4><<<grid, kBlockP, lg.bytes, st>>>(boxes, vstart, nbox, flip, dl, lk.mlo, lg.mlo, lg.nkn); \
  } while (0)
  if (acc == 0) MISA_FORCE_B(0);
  else if (acc == 1) MISA_FORCE_B(1);
  else MISA_FORCE_B(2);
#undef MISA_FORCE_B
  return true;
}

}  // namespace misa
