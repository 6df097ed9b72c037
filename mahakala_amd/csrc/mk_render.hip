// mk_render.hip -- fused per-ray image kernel: camera ray, RK4 null geodesic
// in Cartesian Kerr-Schild, meshblock sampling, thermal synchrotron
// emission/absorption and transfer, one ray per lane (images.py:30-144 of
// the reference, with geodesics.py, athenak.py, electrons.py, transfer.py).
//
// The reference materialises the (T, npx, 8) history, samples every row and
// scans the explicit-Euler transfer backward from the far end:
//     I <- I - dt[i-1] L (j[i] - alpha[i] I),  i = T-1 .. 1.
// That recurrence is linear in I, so with c_i = -dt[i-1] L it equals
//     I = sum_{i>=1} c_i j_i prod_{k<i} (1 - c_k alpha_k),
// which this kernel accumulates in the order the ray is integrated, keeping
// no history.  Rows i > K (frozen) have dt = 0 and add nothing; row 0 never
// contributes; row N is never emitted, so the sample after step N-1 is
// skipped.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <map>
#include <mutex>
#include <tuple>
#include <type_traits>
#include <vector>

#include "mk_device.h"
#include "mk_internal.h"
#include "mk_render.h"
#include "mk_snapshot.h"
#include "mk_triple.h"

namespace mk {

// One ray.  The sample of an accepted step is located, fetched and added right
// after the step (in the order of the steps); the ray keeps its last block
// record and skips the lookup while its samples stay in that block.  ZONE
// (mixed): FP64 steps while a live ray of the wave is in the zone; a build of
// its own, since the second RK4 step's code costs every mixed launch (1024^2
// torus at a = 0.94, i = 17 deg: 9.35 -> 8.44 ms without it).
template <bool MIXED, bool ZONE>
__device__ __forceinline__ void trace_ray(const SnapView& sv, const RenderDev& rp, double x_img, double y_img,
                                          double& I_out, int& steps_out) {
  using T = typename std::conditional<MIXED, float, double>::type;
  double sx[4], sv4[4], s[8], nw[8], rn, dtn;
  camera_ray(x_img, y_img, rp.ci, rp.si, rp.dist, sx, sv4);
  nullify(sx, sv4, rp.a, s);
  double r = radius_cal(s[1], s[2], s[3], rp.a);
  double dt = step_rule(r, rp.rEH, rp.div, rp.tol);
  KsHead h{}, hn{};  // FP64: the position terms at s and at the candidate
  if constexpr (!MIXED) h = ks_head(s[1], s[2], s[3], rp.a);
  double I = 0.0, trans = 1.0, drdl = 1e300, lim = 1500.0;
  int nacc = 0, k = 0, cmb = -1;
  double crec[kMeta];
  // RK4 step to the candidate nw, its radius and its step (0 ends the ray)
  auto step = [&]() {
    if constexpr (!MIXED) {
      rk4_step64(s, h, dt, rp.a, nw);
      hn = ks_head(nw[1], nw[2], nw[3], rp.a);
      rn = hn.r;
      dtn = step_rule(rn, rp.rEH, rp.div, rp.tol, lim);
    } else {
      const bool fp64 = ZONE && __any(dt != 0.0 && ((r < rp.fp64_r) || (r < rp.ring_r && __builtin_fabs(drdl) < rp.ring_drdl)));
      if (fp64) rk4_step<double>(s, dt, rp.a, nw);
      else rk4_step_mixed(s, dt, (float)rp.a, nw);
      rn = radius_f32(nw[1], nw[2], nw[3], rp.a);
      dtn = step_rule_fast(rn, rp.rEH, rp.inv_div, rp.div, rp.tol, lim);
    }
  };
  auto accept = [&]() {
    if (ZONE) drdl = (rn - r) / dt;
#pragma unroll
    for (int q = 0; q < 8; ++q) s[q] = nw[q];
    dt = dtn;
    r = rn;
    h = hn;
  };
  // the way in, as in the triple form: no sample until a ray of the wave is
  // inside the domain's sphere, and the step that takes it there is left to
  // the loop below
  while (k < rp.N && __any(dt != 0.0)) {
    step();
    dtn = dt != 0.0 ? dtn : 0.0;
    if (__any(dtn != 0.0 && rn <= rp.r_dom)) break;
    nacc += dtn != 0.0;
    accept();
    ++k;
  }
  // a ray inside the sphere of radius r_out ends when it leaves it again
  if (r < rp.r_out) lim = __builtin_fmin(1500.0, rp.r_out - rp.rEH);
  for (; k < rp.N && dt != 0.0; ++k) {
    step();
    if (dtn == 0.0) break;
    ++nacc;
    if (k + 1 < rp.N) {  // row N is never emitted
      const Stencil st = locate_cached(sv, sv.meta, sv.grid, nw[1], nw[2], nw[3], cmb, crec);
      // Outside the domain (all primitives zero) and wherever the density is
      // zero, the reference's j and alpha come out 0 (or NaN, then 0), and the
      // step adds exactly nothing: those samples skip the emission arithmetic.
      if (st.mb >= 0) {
        Corners c;
        T P[8], j, al;
        fetch(sv, st, c);
        interp<T>(st, c, P);
        if (P[0] != T(0)) {
          emission_from_prims<T>(rp.ip, P, nw, rp.a, j, al);
          const double cc = -dt * rp.ip.L_unit;
          I += trans * (cc * (double)j);
          trans *= (1.0 - cc * (double)al);
        }
      }
    }
    accept();
  }
  I_out = I;
  steps_out = nacc;
}

// Pixel of lane: each wave takes an 8x8 tile; workgroup ids are remapped so
// each of the 8 XCDs (hardware assigns workgroups round-robin) walks a
// contiguous band of tiles and shares snapshot lines in its own L2.
__device__ __forceinline__ bool pixel_of_lane(const RenderDev& rp, int& i, int& j) {
  const unsigned nwg = gridDim.x, wg = blockIdx.x;
  const unsigned per = nwg / 8;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  long tile;
  if (rp.order) {  // workgroups start in index order: the longest tiles first
    const long k = (long)wg * (blockDim.x >> 6) + wave;
    if (k >= rp.ntiles) return false;
    tile = rp.order[k];
  } else {
    const unsigned lwg = (nwg % 8 == 0) ? (wg % 8) * per + wg / 8 : wg;
    tile = (long)lwg * (blockDim.x >> 6) + wave;
  }
  if (tile >= rp.ntiles) return false;
  const int ti = (int)(tile / rp.tiles_x), tj = (int)(tile % rp.tiles_x);
  i = ti * 8 + (lane >> 3);
  j = tj * 8 + (lane & 7);
  return i < rp.res && j < rp.res;
}

// Copies the block geometry and the leaf lookup grid into LDS (paired form).
__device__ __forceinline__ void stage_tables(const SnapView& sv, double* lds, const double*& meta, const int*& grid) {
  const int nm = sv.nmb * kMeta, ng = sv.gx * sv.gy * sv.gz;
  for (int t = threadIdx.x; t < nm; t += blockDim.x) lds[t] = sv.meta[t];
  int* g = reinterpret_cast<int*>(lds + nm);
  for (int t = threadIdx.x; t < ng; t += blockDim.x) g[t] = sv.grid[t];
  __syncthreads();
  meta = lds;
  grid = g;
}

// Three waves per SIMD in mixed (168 VGPRs), two in FP64.  The block tables are
// read from global memory: against one copy of them in LDS per CU (workgroups
// of 12 or 8 waves) mixed 768^2 at a = 0.9, i = 60 deg 7.05 against 7.88 ms,
// 1024^2 at a = 0.94, i = 17 deg 8.60 against 8.53 ms, plain FP64 8.3 against
// 9.1 and 11.7 against 11.9 ms, and a launch needs no staging and no limit on
// the number of blocks.  (Two waves with the sample pipelined behind the next
// step, the form before for FP64 and for tables beyond 53 KB: 1024^2 octree
// 10.5 ms mixed, 13.0 ms FP64 at a = 0.94.)
//
// With rp.next_tile the grid holds only the workgroups resident at once, and
// each of their waves takes the next tile (in tile
// order) from the counter until none is left, so a wave whose tile ends early
// starts another instead of idling until its workgroup's longest tile ends.
// next_tile[1] counts the waves that found none left; the last of them sets
// both words back to 0, so the next launch on the stream starts from 0.
template <bool MIXED, bool ZONE>
__global__ void __launch_bounds__(256, MIXED ? 3 : 2) k_render(SnapView sv, RenderDev rp, double* __restrict__ img,
                                                               int32_t* __restrict__ steps) {
  if (rp.next_tile) {
    const int lane = threadIdx.x & 63;
    while (true) {
      int k = 0;
      if (lane == 0) k = atomicAdd(rp.next_tile, 1);
      k = __builtin_amdgcn_readfirstlane(__shfl(k, 0));
      if (k >= rp.ntiles) {
        // every other wave has taken its last ticket before it counts itself
        // here, so the last one to count leaves no taker behind
        if (lane == 0 && atomicAdd(rp.next_tile + 1, 1) == (int)(gridDim.x * (blockDim.x >> 6)) - 1) {
          __hip_atomic_store(rp.next_tile, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          __hip_atomic_store(rp.next_tile + 1, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        break;
      }
      const long tile = rp.order ? rp.order[k] : k;
      const int i = (int)(tile / rp.tiles_x) * 8 + (lane >> 3), j = (int)(tile % rp.tiles_x) * 8 + (lane & 7);
      if (i < rp.res && j < rp.res) {
        double I;
        int n;
        trace_ray<MIXED, ZONE>(sv, rp, grid_coord(rp.lo, rp.step, i), grid_coord(rp.lo, rp.step, j), I, n);
        const long p = (long)i * rp.res + j;
        img[p] = I;
        if (steps) steps[p] = n;
      }
    }
    return;
  }
  int i, j;
  if (!pixel_of_lane(rp, i, j)) return;
  double I;
  int n;
  trace_ray<MIXED, ZONE>(sv, rp, grid_coord(rp.lo, rp.step, i), grid_coord(rp.lo, rp.step, j), I, n);
  const long p = (long)i * rp.res + j;
  img[p] = I;
  if (steps) steps[p] = n;
}

// --------------------------------------------------------------- paired form
// For launches of at most one tile per SIMD (a 256^2 image is 1024 tiles on
// 1024 SIMDs) the time is the slowest tile's step count times the step
// latency of a wave alone on its SIMD.  The paired form gives each tile two
// waves: a geodesic wave (camera ray, RK4, step rule) and a transfer wave
// (block lookup, gather, interpolation, emission, transfer).  They run
// concurrently and hand samples over through a ring of kPairDepth slots in
// LDS, synchronised by two counters per pair (rounds produced, rounds
// consumed) with release/acquire ordering at workgroup scope; no barrier
// couples different tiles.  Waits are bounded: after kSpinLimit polls a wave
// gives up and writes NaN for its pixels, so every wave exits.  The transfer
// wave adds the samples in step order with the same expressions as the
// classic form.
constexpr int kPairTiles = 4;   // tiles per workgroup (geodesic + transfer wave each)
constexpr int kPairDepth = 4;   // ring slots per tile
constexpr size_t kPairRingDoubles = (size_t)kPairTiles * kPairDepth * kPairComp * 64;
constexpr size_t kPairLdsExtra = kPairRingDoubles * sizeof(double) + kPairTiles * 4 * sizeof(int);

// Polls *cnt (LDS) until it reaches target; false after `limit` polls.
__device__ __forceinline__ bool wait_at_least(int* cnt, int target, int limit) {
  for (int spin = 0; spin < limit; ++spin) {
    const int v = __builtin_amdgcn_readfirstlane(
        __hip_atomic_load(cnt, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP));
    if (v >= target) return true;
    __builtin_amdgcn_s_sleep(1);
  }
  return false;
}

template <bool MIXED>
__global__ void __launch_bounds__(128 * kPairTiles) k_render_pair(SnapView sv, RenderDev rp, double* __restrict__ img,
                                                                  int32_t* __restrict__ steps, int tab_doubles) {
  using T = typename std::conditional<MIXED, float, double>::type;
  extern __shared__ double lds[];
  double* ring_all = lds + tab_doubles;
  int* ctr = reinterpret_cast<int*>(ring_all + kPairRingDoubles);  // per tile: produced, consumed, done, pad
  if (threadIdx.x < 4 * kPairTiles) ctr[threadIdx.x] = ((threadIdx.x & 3) == 2) ? -1 : 0;
  const double* meta;
  const int* grid;
  stage_tables(sv, lds, meta, grid);  // ends with a workgroup barrier
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int pair = wave % kPairTiles;
  const bool geo = wave < kPairTiles;
  double* ring = ring_all + (size_t)pair * kPairDepth * kPairComp * 64 + lane;
  int* produced = ctr + 4 * pair;
  int* consumed = produced + 1;
  int* done = produced + 2;
  const unsigned nwg = gridDim.x, wg = blockIdx.x, per = nwg / 8;
  const unsigned lwg = (nwg % 8 == 0) ? (wg % 8) * per + wg / 8 : wg;
  const long tile = (long)lwg * kPairTiles + pair;
  int pi = 0, pj = 0;
  bool valid = tile < rp.ntiles;
  if (valid) {
    pi = (int)(tile / rp.tiles_x) * 8 + (lane >> 3);
    pj = (int)(tile % rp.tiles_x) * 8 + (lane & 7);
    valid = pi < rp.res && pj < rp.res;
  }
  const long p = (long)pi * rp.res + pj;
  if (geo) {
    double s[8], r = 0.0, dt = 0.0, drdl = 1e300;
    KsHead h{}, hn{};  // FP64: the position terms at s and at the candidate
    int k = 0, nacc = 0;
    bool alive = false;
    if (valid) {
      double sx[4], sv4[4];
      camera_ray(grid_coord(rp.lo, rp.step, pi), grid_coord(rp.lo, rp.step, pj), rp.ci, rp.si, rp.dist, sx, sv4);
      nullify(sx, sv4, rp.a, s);
      r = radius_cal(s[1], s[2], s[3], rp.a);
      dt = step_rule(r, rp.rEH, rp.div, rp.tol);
      if constexpr (!MIXED) h = ks_head(s[1], s[2], s[3], rp.a);
      alive = true;
    }
    const bool zone = MIXED && (rp.fp64_r > 0.0 || rp.ring_r > 0.0);
    bool ok = true;
    int t = 0;
    while (__any(alive)) {
      if (!wait_at_least(consumed, t - kPairDepth + 1, rp.spin_limit)) {
        ok = false;
        break;
      }
      double* out = ring + (size_t)(t % kPairDepth) * kPairComp * 64;
      bool wrote = false;
      if (alive) {
        if (k >= rp.N || dt == 0.0) {
          alive = false;
        } else {
          double nw[8];
          if constexpr (!MIXED) {
            rk4_step64(s, h, dt, rp.a, nw);
          } else {
            const bool fp64 = zone && __any((r < rp.fp64_r) || (r < rp.ring_r && __builtin_fabs(drdl) < rp.ring_drdl));
            if (fp64) rk4_step<double>(s, dt, rp.a, nw);
            else rk4_step_mixed(s, dt, (float)rp.a, nw);
          }
          double rn, dtn;
          if constexpr (!MIXED) {
            hn = ks_head(nw[1], nw[2], nw[3], rp.a);
            rn = hn.r;
            dtn = step_rule(rn, rp.rEH, rp.div, rp.tol);
          } else {
            rn = radius_f32(nw[1], nw[2], nw[3], rp.a);
            dtn = step_rule_fast(rn, rp.rEH, rp.inv_div, rp.div, rp.tol);
          }
          if (dtn == 0.0) {
            alive = false;
          } else {
            ++nacc;
            if (k + 1 < rp.N) {  // row N is never emitted
#pragma unroll
              for (int c = 0; c < 8; ++c) out[c * 64] = nw[c];
              out[8 * 64] = dt;
              wrote = true;
            }
            if (zone) drdl = (rn - r) / dt;
#pragma unroll
            for (int c = 0; c < 8; ++c) s[c] = nw[c];
            dt = dtn;
            r = rn;
            h = hn;
            if (++k >= rp.N) alive = false;
          }
        }
      }
      if (!wrote) out[8 * 64] = 0.0;
      publish(produced, ++t);
    }
    publish(done, ok ? t : -2);
    if (valid && steps) steps[p] = ok ? nacc : -1;
    return;
  }
  // transfer wave
  double I = 0.0, trans = 1.0, ps[8], pdt = 0.0;
  bool pend = false, ok = true;
  Stencil pst;
  Corners pc;
  auto consume = [&]() {
    if (pst.mb < 0) return;
    T P[8], j, al;
    interp<T>(pst, pc, P);
    if (P[0] == T(0)) return;
    emission_from_prims<T>(rp.ip, P, ps, rp.a, j, al);
    const double c = -pdt * rp.ip.L_unit;
    I += trans * (c * (double)j);
    trans *= (1.0 - c * (double)al);
  };
  for (int t = 0;; ++t) {
    // round t is ready, or the geodesic wave has finished after fewer rounds
    int state = 0;
    for (int spin = 0; spin < rp.spin_limit; ++spin) {
      const int pr = __builtin_amdgcn_readfirstlane(
          __hip_atomic_load(produced, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP));
      if (pr > t) {
        state = 1;
        break;
      }
      const int dn = __builtin_amdgcn_readfirstlane(
          __hip_atomic_load(done, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP));
      if (dn == -2 || (dn >= 0 && t >= dn)) {
        state = dn == -2 ? -1 : 2;
        break;
      }
      __builtin_amdgcn_s_sleep(1);
    }
    if (state != 1) {
      ok = state == 2;
      break;
    }
    if (pend) {
      consume();
      pend = false;
    }
    const double* in = ring + (size_t)(t % kPairDepth) * kPairComp * 64;
    pdt = in[8 * 64];
    if (pdt != 0.0) {
#pragma unroll
      for (int c = 0; c < 8; ++c) ps[c] = in[c * 64];
      pst = locate(sv, meta, grid, ps[1], ps[2], ps[3]);
      fetch(sv, pst, pc);
      pend = true;
    }
    publish(consumed, t + 1);  // the slot is in registers now
  }
  if (pend) consume();
  if (valid) img[p] = ok ? I : __builtin_nan("");
}

// ZONE: see tri_geodesic.
template <bool MIXED, bool ZONE>
__global__ void __launch_bounds__(256, 4) k_render_tri(SnapView sv, RenderDev rp, double* __restrict__ img,
                                                       int32_t* __restrict__ steps) {
  __shared__ TriRings<MIXED> ring;
  if (threadIdx.x == 0) ring.reset();
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // workgroups start in index order: with a tile order the longest tiles go
  // first; without one each of the 8 XCDs takes a contiguous band of tiles
  const unsigned nwg = gridDim.x, wg = blockIdx.x;
  long tile = (!rp.order && nwg % 8 == 0) ? (wg % 8) * (nwg / 8) + wg / 8 : wg;
  if (rp.order) tile = rp.order[tile];
  const int pi = (int)(tile / rp.tiles_x) * 8 + (lane >> 3), pj = (int)(tile % rp.tiles_x) * 8 + (lane & 7);
  const bool valid = pi < rp.res && pj < rp.res;
  const long p = (long)pi * rp.res + pj;
  if (wave == 0) {
    int n;
    tri_geodesic<MIXED, ZONE>(ring, rp, rp.spin_limit, grid_coord(rp.lo, rp.step, pi), grid_coord(rp.lo, rp.step, pj),
                              valid, n);
    if (valid && steps) steps[p] = n;
  } else if (wave <= 2) {
    tri_gather<MIXED>(ring, wave - 1, sv, rp.spin_limit);
  } else {
    bool ok;
    const double I = tri_emission<MIXED>(ring, rp, rp.spin_limit, ok);
    if (valid) img[p] = I;
  }
}

// Critical curve of a distant camera at inclination theta (Bardeen 1973):
// spherical photon orbits of radius r in [r_pro, r_retro] appear at
// alpha = -xi / sin(theta), beta = +-sqrt(eta + a^2 cos^2(theta) -
// xi^2 cot^2(theta)), with xi = (r^2 (3 - r) - a^2 (r + 1)) / (a (r - 1)) and
// eta = r^3 (4 a^2 - r (r - 3)^2) / (a^2 (r - 1)^2).  Image x is alpha and
// image y is beta in this camera's convention.  Returned as a polar table
// R(phi) about the curve's centre (cx, 0), kBins bins; a = 0 gives the circle
// of radius sqrt(27).
namespace {
constexpr int kBins = 256;
void critical_curve_polar(double a, double inc_deg, double* cx, double R[kBins]) {
  const double th = std::min(std::max(inc_deg, 1.0), 179.0) * M_PI / 180.0;
  *cx = 0.0;
  if (std::fabs(a) < 1e-3) {
    for (int k = 0; k < kBins; ++k) R[k] = std::sqrt(27.0);
    return;
  }
  const double aa = std::fabs(a) > 0.999 ? (a > 0 ? 0.999 : -0.999) : a;
  const double r1 = 2.0 * (1.0 + std::cos(2.0 / 3.0 * std::acos(-std::fabs(aa))));
  const double r2 = 2.0 * (1.0 + std::cos(2.0 / 3.0 * std::acos(std::fabs(aa))));
  const double ct = std::cos(th) / std::sin(th), c2 = std::cos(th) * std::cos(th);
  std::vector<double> al, be;
  const int n = 2048;
  for (int q = 0; q <= n; ++q) {
    const double r = std::min(r1, r2) + (std::fabs(r2 - r1)) * q / n;
    if (std::fabs(r - 1.0) < 1e-9) continue;
    const double xi = (r * r * (3.0 - r) - aa * aa * (r + 1.0)) / (aa * (r - 1.0));
    const double eta = r * r * r * (4.0 * aa * aa - r * (r - 3.0) * (r - 3.0)) / (aa * aa * (r - 1.0) * (r - 1.0));
    const double b2 = eta + aa * aa * c2 - xi * xi * ct * ct;
    if (!(b2 >= 0.0)) continue;
    al.push_back(-xi / std::sin(th));
    be.push_back(std::sqrt(b2));
  }
  if (al.size() < 8) {
    for (int k = 0; k < kBins; ++k) R[k] = std::sqrt(27.0);
    return;
  }
  *cx = 0.5 * (*std::min_element(al.begin(), al.end()) + *std::max_element(al.begin(), al.end()));
  std::vector<double> sum(kBins, 0.0);
  std::vector<int> cnt(kBins, 0);
  for (size_t q = 0; q < al.size(); ++q)
    for (int sgn = -1; sgn <= 1; sgn += 2) {
      const double dx = al[q] - *cx, dy = sgn * be[q];
      int k = (int)std::floor((std::atan2(dy, dx) + M_PI) / (2.0 * M_PI) * kBins);
      k = std::min(std::max(k, 0), kBins - 1);
      sum[k] += std::sqrt(dx * dx + dy * dy);
      ++cnt[k];
    }
  // empty bins take the nearest filled bin's radius (circularly)
  for (int k = 0; k < kBins; ++k) {
    if (cnt[k]) {
      R[k] = sum[k] / cnt[k];
      continue;
    }
    for (int d = 1; d < kBins; ++d) {
      const int u = (k + d) % kBins, v = (k - d + kBins) % kBins;
      if (cnt[u]) { R[k] = sum[u] / cnt[u]; break; }
      if (cnt[v]) { R[k] = sum[v] / cnt[v]; break; }
    }
  }
}
}  // namespace

std::vector<int> ring_first_tile_order(int res, double lo, double step, double a, double inc_deg) {
  double cx, R[kBins];
  critical_curve_polar(a, inc_deg, &cx, R);
  const int tx = (res + 7) / 8, nt = tx * tx;
  std::vector<double> d(nt);
  for (int t = 0; t < nt; ++t) {
    // tile centre: pixel 8 t + 3.5 at coordinate (2 i + 1) step + lo
    const double x = (16.0 * (t / tx) + 8.0) * step + lo - cx, y = (16.0 * (t % tx) + 8.0) * step + lo;
    int k = (int)std::floor((std::atan2(y, x) + M_PI) / (2.0 * M_PI) * kBins);
    k = std::min(std::max(k, 0), kBins - 1);
    d[t] = std::fabs(std::sqrt(x * x + y * y) - R[k]);
  }
  std::vector<int> ord(nt);
  for (int t = 0; t < nt; ++t) ord[t] = t;
  std::stable_sort(ord.begin(), ord.end(), [&](int u, int v) { return d[u] < d[v]; });
  return ord;
}

// Device copies of tile orders, one per (device, resolution, fov, spin,
// inclination), made on first use and kept until the process ends (immutable,
// so launches in flight never see them change).  An entry is published only
// once its copy is in memory: any stream may use it from then on.  Past
// kOrderCacheBytes, or while the stream is being captured into a graph (no
// allocation there), launches use row-major tiles.
namespace {
std::mutex g_order_mu;
std::map<std::tuple<int, int, double, double, double>, int*> g_orders;
std::map<int, hipStream_t> g_order_streams;  // per device, for these copies alone
size_t g_order_bytes = 0;
constexpr size_t kOrderCacheBytes = (size_t)64 << 20;
}  // namespace

// One tile counter (two ints: next tile, waves done) per (device, stream) for
// the classic form's queue: allocated and zeroed on the stream on first use,
// and left at zero by every launch that uses it.
static std::mutex g_counter_mu;
static std::map<std::pair<int, hipStream_t>, int*> g_counters;

static int* tile_counter(hipStream_t st) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return nullptr;
  std::lock_guard<std::mutex> lk(g_counter_mu);
  auto it = g_counters.find({dev, st});
  if (it != g_counters.end()) return it->second;
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(st, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone) return nullptr;
  int* c = nullptr;
  if (hipMalloc(&c, 2 * sizeof(int)) != hipSuccess) return nullptr;
  if (hipMemsetAsync(c, 0, 2 * sizeof(int), st) != hipSuccess) {
    (void)hipFree(c);
    return nullptr;
  }
  g_counters.emplace(std::make_pair(dev, st), c);
  return c;
}

static const int* render_tile_order(const RenderDev& rp, const mk_render_params* p, hipStream_t st) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return nullptr;
  const auto key = std::make_tuple(dev, rp.res, p->fov, p->bhspin, p->inclination);
  std::lock_guard<std::mutex> lk(g_order_mu);
  auto it = g_orders.find(key);
  if (it != g_orders.end()) return it->second;
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(st, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone) return nullptr;
  const size_t bytes = (size_t)rp.ntiles * sizeof(int);
  if (g_order_bytes + bytes > kOrderCacheBytes) return nullptr;
  std::vector<int> ord = ring_first_tile_order(rp.res, rp.lo, rp.step, p->bhspin, p->inclination);
  int* d = nullptr;
  if (hipMalloc(&d, bytes) != hipSuccess) return nullptr;
  // on the caller's stream if it is idle, else on one of its own (made once, 4 ms), so as not to wait for that work
  hipStream_t copy = st;
  hipError_t e = hipStreamQuery(st);
  if (e == hipErrorNotReady) {
    (void)hipGetLastError();
    hipStream_t& own = g_order_streams[dev];
    e = own ? hipSuccess : hipStreamCreateWithFlags(&own, hipStreamNonBlocking);
    copy = own;
  }
  if (e == hipSuccess) e = hipMemcpyAsync(d, ord.data(), bytes, hipMemcpyHostToDevice, copy);
  if (e == hipSuccess) e = hipStreamSynchronize(copy);
  if (e != hipSuccess) {
    (void)hipFree(d);
    return nullptr;
  }
  g_orders.emplace(key, d);
  g_order_bytes += bytes;
  return d;
}

size_t table_bytes(const SnapView& sv) {
  return (size_t)sv.nmb * kMeta * sizeof(double) + (size_t)sv.gx * sv.gy * sv.gz * sizeof(int);
}

// r_dom: no point of the domain has a larger Kerr-Schild radius (r^2 <= x^2 +
// y^2 + z^2; the corner's distance with a margin for the radius in FP32).
// r_out: a ray that moves outward beyond it, outside the domain, never returns
// (a null geodesic has no outer turning point beyond the photon orbits, r <= 4 M),
// so every later step would add exactly nothing and the ray may end: an escaping
// ray takes about 120 of its 530 steps out there.  Infinite when the caller asks
// for step counts, which cover the whole ray.
void set_domain_radii(const SnapView& sv, bool whole_rays, double* r_dom, double* r_out) {
  double s = 0.0;
  for (int d = 0; d < 3; ++d) {
    const double m = std::max(std::fabs(sv.dom_lo[d]), std::fabs(sv.dom_hi[d]));
    s += m * m;
  }
  *r_dom = 1.001 * std::sqrt(s);
  *r_out = whole_rays ? HUGE_VAL : std::max(1.1 * *r_dom, 12.0);
}

int fill_render_dev(const mk_render_params* p, RenderDev* rp) {
  MK_REQUIRE(p->resolution > 0 && p->max_nsteps >= 1 && p->div != 0.0, "render: bad resolution/max_nsteps/div");
  MK_REQUIRE(p->precision == 0 || p->precision == 1, "render: precision must be 0 (plain FP64) or 1 (mixed)");
  MK_REQUIRE(std::fabs(p->bhspin) <= 1.0, "render: |bhspin| must be <= 1");
  MK_REQUIRE(p->observing_frequency > 0.0 && p->M_bh > 0.0 && p->mass_scale > 0.0, "render: bad units");
  const double inc = p->inclination * M_PI / 180;
  rp->a = p->bhspin;
  rp->ci = std::cos(inc);
  rp->si = std::sin(inc);
  rp->dist = p->distance;
  rp->lo = -p->fov / 2.0;
  rp->step = (p->fov / 2.0 - (-p->fov / 2.0)) / (double)(2 * p->resolution);
  rp->rEH = 1.0 + std::sqrt(1.0 - p->bhspin * p->bhspin);
  rp->div = p->div;
  rp->inv_div = 1.0 / p->div;
  rp->tol = p->tol;
  rp->res = p->resolution;
  rp->N = p->max_nsteps;
  rp->tiles_x = (p->resolution + 7) / 8;
  rp->ntiles = (long)rp->tiles_x * rp->tiles_x;
  // grmhd.py:40-55
  const double G = 6.6743e-8, CL = 2.99792458e10, MP = 1.6726e-24, ME = 9.1094e-28;
  const double L = G * p->M_bh / (CL * CL);
  const double dens_unit = p->mass_scale / (L * L * L);
  rp->ip.fluid_gamma = p->fluid_gamma;
  rp->ip.r_high = p->r_high;
  rp->ip.Ne_unit = dens_unit / (MP + ME);
  rp->ip.B_unit = CL * std::sqrt(4.0 * M_PI * dens_unit);
  rp->ip.L_unit = L;
  rp->ip.nu_obs = p->observing_frequency;
  rp->ip.fallback_cos = std::cos(p->fallback_pitch);
  rp->ip.sigma_cut = p->sigma_cut;
  rp->fp64_r = p->fp64_radius;
  rp->ring_r = p->ring_radius;
  rp->ring_drdl = p->ring_drdl;
  rp->spin_limit = (p->flags & MK_RENDER_WAIT_TEST) ? 1 : kSpinLimit;
  rp->order = nullptr;
  rp->next_tile = nullptr;
  return MK_OK;
}

}  // namespace mk

using namespace mk;

template <bool MIXED, bool ZONE>
static int launch_tri(const SnapView& sv, const RenderDev& rp, double* d_image, int32_t* d_steps, hipStream_t st) {
  k_render_tri<MIXED, ZONE><<<dim3((unsigned)rp.ntiles), dim3(256), 0, st>>>(sv, rp, d_image, d_steps);
  MK_LAUNCH_CHECK();
  return MK_OK;
}

static int choose_form(const SnapView& sv, const RenderDev& rp, int precision, int flags, int* form) {
  const size_t tab = (table_bytes(sv) + 15) / 16 * 16;
  const bool fits2 = table_bytes(sv) <= kMaxTableLds && tab + kPairLdsExtra <= 160 * 1024;
  *form = MK_RENDER_CLASSIC;
  if (flags & MK_RENDER_CLASSIC) return MK_OK;
  if (flags & MK_RENDER_TRIPLE) {
    *form = MK_RENDER_TRIPLE;
    return MK_OK;
  }
  if (flags & MK_RENDER_PAIRED) {
    if (fits2) *form = MK_RENDER_PAIRED;
    return MK_OK;
  }
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) {
    set_error("mk_render: no device");
    return MK_ERR_HIP;
  }
  // triple form up to 15.5 tiles per CU in mixed precision (a 496^2 image on
  // 256 CUs) and 11 in FP64 (424^2); the classic form beyond, where every
  // SIMD holds waves of whole rays.  a = 0.5, i = 30 deg (a = 0.9, i = 60 deg),
  // triple against classic: mixed 480^2 3.10 (3.15) and 4.72 (7.51) ms, 640^2
  // 4.9 (4.7) and 4.7 (8.0) ms; plain FP64 416^2 3.45 (3.50) and 4.31 (8.54) ms.
  // Beyond |a sin i| = 0.5 the rays at the prograde edge take so many steps
  // that a classic launch lasts as long as their tiles do, at half the triple
  // form's rate, so the line moves up with them.  Triple against classic, mixed
  // (FP64): a = 0.7, i = 50 deg, 576^2 4.36 and 4.60 (5.88 and 5.53) ms; a = 0.9,
  // i = 60 deg, 640^2 5.14 and 6.95 (6.93 and 8.29), 768^2 7.22 and 7.29 (9.7 and
  // 8.5); a = 0.97, i = 80 deg, 768^2 7.24 and 13.1 (9.7 and 15.6), 1024^2 12.8
  // and 15.5 (17.1 and 18.5) ms.
  // The line moves with the field of view f (in M) too: the wider, the smaller the
  // share of tiles with long rays, and the more such a launch waits for them.
  // Times where the forms are level, in tiles per CU, |a sin i| <= 0.25, mixed (FP64):
  // f = 5 M 5 (3), 8 M 10 (6), 12 M 11 (8), 20 M 16 (12), 36 M 20 (17), 60 M 28 (22),
  // 100 M 36 (32), 300 M 36 (34).  The factor f / (0.355 f + 12.9) is 1 at 20 M and
  // 0.34, 0.70, 1.75 and 2.5 at 5, 12, 60 and 300 M.  Octree of 512 blocks, mixed,
  // a = 0, f = 60 M, 512^2: triple 2.06, classic 3.14 ms; a = 0.9, i = 60 deg, f = 12 M,
  // 768^2 9.1 and 7.7 ms.  At most 8 in all: 1408^2 is the largest image measured.
  const double x2 = rp.a * rp.a * rp.si * rp.si, f = std::fabs(2.0 * rp.lo);
  const double edge = x2 > 0.25 ? (x2 < 0.75 ? 1.0 / (1.0 - x2) : 4.0) : 1.0;
  const double scale = std::min(edge * f / (0.355 * f + 12.9), 8.0);
  if ((double)(2 * rp.ntiles) <= scale * (double)((precision == 1 ? 31L : 22L) * cus)) *form = MK_RENDER_TRIPLE;
  return MK_OK;
}

extern "C" int mk_render_form(const mk_snapshot* snap, const mk_render_params* p, int32_t* h_form) {
  MK_REQUIRE(snap && p && h_form, "mk_render_form: null argument");
  RenderDev rp;
  int rc = fill_render_dev(p, &rp);
  if (rc) return rc;
  int form = 0;
  rc = choose_form(snap->view(), rp, p->precision, p->flags, &form);
  *h_form = form;
  return rc;
}

extern "C" int mk_render(const mk_snapshot* snap, const mk_render_params* p, double* d_image, int32_t* d_steps,
                         void* stream) {
  MK_REQUIRE(snap && p && d_image, "mk_render: null argument");
  RenderDev rp;
  int rc = fill_render_dev(p, &rp);
  if (rc) return rc;
  const SnapView sv = snap->view();
  set_domain_radii(sv, d_steps != nullptr, &rp.r_dom, &rp.r_out);
  // a tile's FP64 zone is decided by its live rays: none may end inside it
  rp.r_out = std::max(rp.r_out, 1.1 * std::max(rp.fp64_r, rp.ring_r));
  const size_t lds = table_bytes(sv);
  hipStream_t st = as_stream(stream);
  const size_t tab = (lds + 15) / 16 * 16;
  int form = 0;
  rc = choose_form(sv, rp, p->precision, p->flags, &form);
  if (rc) return rc;
  if (form != MK_RENDER_PAIRED && !(p->flags & MK_RENDER_ROW_MAJOR)) rp.order = render_tile_order(rp, p, st);
  if (form == MK_RENDER_TRIPLE) {
    if (p->precision == 0) return launch_tri<false, false>(sv, rp, d_image, d_steps, st);
    return rp.fp64_r > 0.0 || rp.ring_r > 0.0 ? launch_tri<true, true>(sv, rp, d_image, d_steps, st)
                                              : launch_tri<true, false>(sv, rp, d_image, d_steps, st);
  }
  if (form == MK_RENDER_PAIRED) {
    long nwg2 = (rp.ntiles + kPairTiles - 1) / kPairTiles;
    nwg2 = (nwg2 + 7) / 8 * 8;
    const size_t lds2 = tab + kPairLdsExtra;
    const int tabd = (int)(tab / sizeof(double));
    if (p->precision == 0)
      k_render_pair<false><<<dim3((unsigned)nwg2), dim3(128 * kPairTiles), lds2, st>>>(sv, rp, d_image, d_steps, tabd);
    else
      k_render_pair<true><<<dim3((unsigned)nwg2), dim3(128 * kPairTiles), lds2, st>>>(sv, rp, d_image, d_steps, tabd);
    MK_LAUNCH_CHECK();
    return MK_OK;
  }
  const bool zoned = rp.fp64_r > 0.0 || rp.ring_r > 0.0;
  auto kern = p->precision == 0 ? k_render<false, false> : (zoned ? k_render<true, true> : k_render<true, false>);
  const int threads = 256, waves = threads / 64;
  dim3 g((unsigned)(((rp.ntiles + waves - 1) / waves + 7) / 8 * 8));
  if (!(p->flags & MK_RENDER_STATIC_TILES)) {  // tiles from a counter (5-12 % faster at 1024^2)
    int dev = 0, cus = 0, per_cu = 0;
    rp.next_tile = tile_counter(st);
    if (rp.next_tile && hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess &&
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, threads, 0) == hipSuccess && per_cu > 0) {
      const long resident = (long)per_cu * cus;
      if (resident < (long)g.x) g = dim3((unsigned)resident);
    } else {
      rp.next_tile = nullptr;
    }
  }
  kern<<<g, dim3(threads), 0, st>>>(sv, rp, d_image, d_steps);
  MK_LAUNCH_CHECK();
  return MK_OK;
}
