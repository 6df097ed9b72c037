// mk_triple.h -- one 8x8 tile of rays by the four waves of a workgroup: the
// triple form of the render kernel, and of the request server's image tiles.
#pragma once
#include <type_traits>

#include "mk_device.h"

namespace mk {

constexpr int kSpinLimit = 1 << 24;  // polls before a bounded wait between waves gives up
constexpr int kPairComp = 9;         // state[8], dt

__device__ __forceinline__ void publish(int* cnt, int v) {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  if ((threadIdx.x & 63) == 0) __hip_atomic_store(cnt, v, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// ------------------------------------------------------------- triple form
// Three stages per tile -- geodesic, gather (lookup, cell loads,
// interpolation) and emission (fluid scalars, j and alpha, transfer) --
// chained by two LDS rings with the counters of the paired form.  One tile is
// one workgroup of four waves: a geodesic wave, two gather waves that take the
// rounds in turn, and an emission wave.  A lone gather wave's round (ring
// read, lookup, cell loads, interpolation: one latency after the other) takes
// about 3300 cycles, a geodesic step 2200, so one gather wave set the pace.
// The hardware puts a workgroup's four waves on the CU's four SIMDs and
// rotates the order from workgroup to workgroup, so with four workgroups per
// CU every SIMD holds one wave of each kind.  The block tables stay in global
// memory (each gather wave keeps its rays' last block record in registers):
// with 51 KB of them in LDS only two workgroups fit a CU, and where both fit
// the times are equal.
// 256^2, a = 0.9, i = 60 deg (a = 0.5, i = 30 deg): with four tiles and one
// gather wave each per workgroup, tables in LDS, plain FP64 3.99 (2.08) ms,
// mixed 3.38 (1.72) ms; with this split 3.48 (2.02) and 3.22 (1.57) ms; with
// rays ending outside the domain and nothing handed over on their way in 3.14
// (1.73) and 3.03 (1.46) ms.  160^2 at a = 0.9: plain 3.93 -> 2.70 ms, mixed
// 3.18 -> 2.65 ms.
// Ring A carries the state (in mixed the momentum already as the floats the
// emission rounds it to) and dt from the geodesic wave, ring B the eight
// interpolated primitives and the state in the emission's precision and dt in
// FP64 (0: nothing to add).
template <bool MIXED>
struct TriRings {
  using T = typename std::conditional<MIXED, float, double>::type;
  static constexpr int kDepthA = 4, kDepthB = MIXED ? 4 : 2;  // rounds (30 and 35 KB: four workgroups fit 160 KB)
  static constexpr int kCompB = 15;                           // P[8], s[1..7]
  // ring A, FP64: the state and dt (without the unused coordinate time the
  // geodesic loop is scheduled 1-2 % slower); mixed: position, dt and, as the
  // emission's floats in one 16-byte word, the momentum (a slot write of 8 bytes
  // costs the geodesic wave about 19 cycles: 256^2 1.422 -> 1.407 ms)
  static constexpr int kCompA = MIXED ? 4 : kPairComp, kPosA = MIXED ? 0 : 1;
  double a[kDepthA][kCompA][64];
  float4 av[MIXED ? kDepthA : 1][64];
  double bd[kDepthB][64];  // dt
  T bt[kDepthB][kCompB][64];
  int producedA, doneA, consumedB;
  int consumedA[2], producedB[2], doneB[2];  // per gather wave

  // before a tile, by one thread; a workgroup barrier follows
  __device__ __forceinline__ void reset() {
    producedA = consumedB = 0;
    doneA = -1;
    for (int g = 0; g < 2; ++g) {
      consumedA[g] = producedB[g] = 0;
      doneB[g] = -1;
    }
  }
};

// Polls *cnt until it reaches target: the value read, or -1 after `limit`
// polls.
__device__ __forceinline__ int wait_value(int* cnt, int target, int limit) {
  for (int spin = 0; spin < limit; ++spin) {
    const int v = __builtin_amdgcn_readfirstlane(
        __hip_atomic_load(cnt, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP));
    if (v >= target) return v;
    __builtin_amdgcn_s_sleep(1);
  }
  return -1;
}

// Waits for round t of a ring: 1 ready (*avail = rounds published), 0 the
// writer finished after fewer rounds, -1 failure (the writer gave up, or
// `limit` polls).
__device__ __forceinline__ int wait_round(int* produced, int* done, int t, int* avail, int limit) {
  for (int spin = 0; spin < limit; ++spin) {
    const int pr = __builtin_amdgcn_readfirstlane(
        __hip_atomic_load(produced, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP));
    if (pr > t) {
      *avail = pr;
      return 1;
    }
    const int dn = __builtin_amdgcn_readfirstlane(
        __hip_atomic_load(done, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP));
    if (dn == -2) return -1;
    if (dn >= 0 && t >= dn) return 0;
    __builtin_amdgcn_s_sleep(1);
  }
  return -1;
}

// The three roles of a tile's four waves; all four run theirs after
// ring.reset() and a workgroup barrier.  They are functions of their own, each
// with the loop over tiles around it where there is one: with one such loop
// around all three, what the compiler moves out of it is live in every role,
// and the FP64 gather and emission spill.  rp: a RenderDev or a request
// descriptor.

// Geodesic wave (0): the tile's 64 rays at image points (x_img, y_img), lanes
// of `valid` only.  steps: the accepted steps per lane (-1 after a failed wait);
// returns the steps of the longest ray.  ZONE (mixed): FP64 steps while any of
// the rays is in the zone (rp.fp64_r, rp.ring_r), as in the other forms; without
// it the zone code is compiled out.
template <bool MIXED, bool ZONE, typename Params>
__device__ __forceinline__ int tri_geodesic(TriRings<MIXED>& ring, const Params& rp, int spin_limit, double x_img,
                                            double y_img, bool valid, int& steps) {
  constexpr int DA = TriRings<MIXED>::kDepthA, CA = TriRings<MIXED>::kCompA;
  const int lane = threadIdx.x & 63;
  // A lane is alive while its dt is not 0; dead lanes step along with dt = 0
  // and are ignored, so the loop has no branches per lane.  All live lanes
  // have taken the same number of steps, k.
  double s[8], r = 0.0, dt = 0.0, drdl = 1e300;
  KsHead h{}, hn{};  // FP64: the position terms at s and at the candidate
  int k = 0, nacc = 0;
#pragma unroll
  for (int q = 0; q < 8; ++q) s[q] = 0.0;
  if (valid) {
    double sx[4], sv4[4];
    camera_ray(x_img, y_img, rp.ci, rp.si, rp.dist, sx, sv4);
    nullify(sx, sv4, rp.a, s);
    r = radius_cal(s[1], s[2], s[3], rp.a);
    dt = step_rule(r, rp.rEH, rp.div, rp.tol);
  }
  if constexpr (!MIXED) h = ks_head(s[1], s[2], s[3], rp.a);
  double lim = 1500.0;  // largest |r - r_EH| of a live ray
  // one RK4 step of every live lane into nw
  auto step = [&](double nw[8]) {
    if constexpr (!MIXED) {
      rk4_step64(s, h, dt, rp.a, nw);
    } else {
      bool fp64 = false;
      if constexpr (ZONE)
        fp64 = __any(dt != 0.0 && ((r < rp.fp64_r) || (r < rp.ring_r && __builtin_fabs(drdl) < rp.ring_drdl)));
      if (fp64) rk4_step<double>(s, dt, rp.a, nw);
      else rk4_step_mixed(s, dt, (float)rp.a, nw);
    }
  };
  // radius and step of the candidate; 0 ends the ray
  auto rule = [&](const double nw[8], double& rn) {
    double dtn;
    if constexpr (!MIXED) {
      hn = ks_head(nw[1], nw[2], nw[3], rp.a);
      rn = hn.r;
      dtn = step_rule(rn, rp.rEH, rp.div, rp.tol, lim);
    } else {
      rn = radius_f32(nw[1], nw[2], nw[3], rp.a);
      dtn = step_rule_fast(rn, rp.rEH, rp.inv_div, rp.div, rp.tol, lim);
    }
    return dt != 0.0 ? dtn : 0.0;
  };
  // The way in: no ray of the tile is inside the sphere around the domain,
  // so the steps are taken without handing anything over.  The step that
  // first takes a ray inside is left to the loop below.
  double nw[8];
  while (k < rp.N && __any(dt != 0.0)) {
    double rn;
    step(nw);
    const double dtn = rule(nw, rn);
    if (__any(dtn != 0.0 && rn <= rp.r_dom)) break;
    nacc += dtn != 0.0;
    if (ZONE) drdl = (rn - r) / dt;
#pragma unroll
    for (int q = 0; q < 8; ++q) s[q] = nw[q];
    dt = dtn;
    r = rn;
    h = hn;
    ++k;
  }
  // A ray inside the sphere of radius r_out ends when it leaves it again.
  if (r < rp.r_out) lim = __builtin_fmin(1500.0, rp.r_out - rp.rEH);
  bool ok = true;
  int t = 0;  // the next round
  for (; k < rp.N && __any(dt != 0.0); ++k, ++t) {
    // Slot t % DA is free once round t - DA has been read.  That count is
    // loaded here without waiting and checked after the RK4 step: a wait at
    // the loop head would also wait on this wave's slot writes of the round
    // before (-2 to -4 % in FP64, -1 % in mixed).
    int* readA = &ring.consumedA[t & 1];
    const int polled = __hip_atomic_load(readA, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    double* out = &ring.a[t % DA][0][lane];
    step(nw);
    double rn, dtn;
    // Mixed: step and rule are kept in front of what follows.  The compiler moves
    // them behind the wait, which leaves the LDS latency of the poll and of the
    // slot writes before it uncovered in every round (256^2 1.444 -> 1.422 ms, at
    // a = 0.9 3.03 -> 2.97; in FP64 2 % slower).
    if constexpr (MIXED) {
      dtn = rule(nw, rn);
#pragma unroll
      for (int q = 1; q < 8; ++q) asm volatile("" : "+v"(nw[q]));
      asm volatile("" : "+v"(dtn));
    }
    // release the previous round here: its slot writes were issued a whole
    // RK4 step ago, so the release fence does not wait on them
    if (t > 0) publish(&ring.producedA, t);
    if (__builtin_amdgcn_readfirstlane(polled) > t - DA) {
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    } else if (wait_value(readA, t - DA + 1, spin_limit) < 0) {
      ok = false;
      break;
    }
    if constexpr (!MIXED) dtn = rule(nw, rn);
    nacc += dtn != 0.0;
    if constexpr (MIXED) {
#pragma unroll
      for (int q = 0; q < 3; ++q) out[q * 64] = nw[1 + q];
      ring.av[t % DA][lane] = make_float4((float)nw[4], (float)nw[5], (float)nw[6], (float)nw[7]);
    } else {
#pragma unroll
      for (int q = 0; q < 8; ++q) out[q * 64] = nw[q];
    }
    out[(CA - 1) * 64] = dtn != 0.0 && k + 1 < rp.N ? dt : 0.0;  // row N is never emitted
    if (ZONE) drdl = (rn - r) / dt;
#pragma unroll
    for (int q = 0; q < 8; ++q) s[q] = nw[q];
    dt = dtn;
    r = rn;
    h = hn;
  }
  if (ok) publish(&ring.producedA, t);
  publish(&ring.doneA, ok ? t : -2);
  steps = ok ? nacc : -1;
  return k;
}

// Gather wave g (0, 1): lookup, cell loads, interpolation of every other round.
template <bool MIXED>
__device__ __forceinline__ void tri_gather(TriRings<MIXED>& ring, int g, const SnapView& sv, int spin_limit) {
  using R = TriRings<MIXED>;
  using T = typename R::T;
  constexpr int DA = R::kDepthA, DB = R::kDepthB;
  const int lane = threadIdx.x & 63;
  bool ok = true;
  int avail = 0, freed = 0;  // rounds of ring A published, of ring B read (last values seen)
  int cmb = -1;              // block of the ray's last sample and its record
  double crec[kMeta];
  int t = g;
  for (;; t += 2) {
    if (t >= avail) {
      const int st = wait_round(&ring.producedA, &ring.doneA, t, &avail, spin_limit);
      if (st <= 0) {
        ok = st == 0;
        break;
      }
    }
    if (t - DB + 1 > freed) {
      freed = wait_value(&ring.consumedB, t - DB + 1, spin_limit);
      if (freed < 0) {
        ok = false;
        break;
      }
    }
    const double* in = &ring.a[t % DA][0][lane];
    double pdt = in[(R::kCompA - 1) * 64];
    const double px = in[R::kPosA * 64], py = in[(R::kPosA + 1) * 64], pz = in[(R::kPosA + 2) * 64];
    T mom[4];
    if constexpr (MIXED) {
      const float4 m = ring.av[t % DA][lane];
      mom[0] = m.x;
      mom[1] = m.y;
      mom[2] = m.z;
      mom[3] = m.w;
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) mom[q] = in[(4 + q) * 64];
    }
    publish(&ring.consumedA[g], t + 1);  // ring A slot is in registers
    T* ob = &ring.bt[t % DB][0][lane];
    T P[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) P[q] = T(0);
    if (pdt != 0.0) {
      const Stencil stc = locate_cached(sv, sv.meta, sv.grid, px, py, pz, cmb, crec);
      if (stc.mb >= 0) {
        Corners cr;
        fetch<false>(sv, stc, cr);
        interp<T>(stc, cr, P);
      }
      if (stc.mb < 0 || P[0] == T(0)) pdt = 0.0;  // adds exactly nothing
    }
#pragma unroll
    for (int q = 0; q < 8; ++q) ob[q * 64] = P[q];
    ob[8 * 64] = (T)px;
    ob[9 * 64] = (T)py;
    ob[10 * 64] = (T)pz;
#pragma unroll
    for (int q = 0; q < 4; ++q) ob[(11 + q) * 64] = mom[q];
    ring.bd[t % DB][lane] = pdt;
    publish(&ring.producedB[g], t + 1);
  }
  publish(&ring.doneB[g], ok ? t : -2);
}

// Emission wave: emission and transfer in step order; the intensity, NaN after
// a failed wait, whichever wave's it was (then ok is false).
template <bool MIXED, typename Params>
__device__ __forceinline__ double tri_emission(TriRings<MIXED>& ring, const Params& rp, int spin_limit, bool& ok) {
  using R = TriRings<MIXED>;
  using T = typename R::T;
  constexpr int DB = R::kDepthB;
  const int lane = threadIdx.x & 63;
  double I = 0.0, trans = 1.0;
  ok = true;
  for (int t = 0;; ++t) {
    int avail = 0;
    const int st = wait_round(&ring.producedB[t & 1], &ring.doneB[t & 1], t, &avail, spin_limit);
    if (st <= 0) {
      ok = st == 0;
      break;
    }
    const T* ib = &ring.bt[t % DB][0][lane];
    const double pdt = ring.bd[t % DB][lane];
    T P[8];
    double ps[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) P[q] = ib[q * 64];
    ps[0] = 0.0;
#pragma unroll
    for (int q = 1; q < 8; ++q) ps[q] = (double)ib[(7 + q) * 64];
    publish(&ring.consumedB, t + 1);  // ring B slot is in registers
    if (pdt != 0.0) {
      T j, al;
      emission_from_prims<T>(rp.ip, P, ps, rp.a, j, al);
      const double cc = -pdt * rp.ip.L_unit;
      I += trans * (cc * (double)j);
      trans *= (1.0 - cc * (double)al);
    }
  }
  return ok ? I : __builtin_nan("");
}

}  // namespace mk
