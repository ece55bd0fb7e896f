// The regions of the persistent applies (k_apply_tile for hard shapes,
// k_apply_lj for isotropic pair energies): region geometry, the staging of a
// region's box into LDS, the neighbour synchronisation between passes and
// the reload of the halo cells a pass changed.
#pragma once
#include "sweep_device.hpp"

namespace hmc {

// ------------------------------------------------ persistent apply (mixed) --
// One launch runs every cycle and colour of an apply.  Workgroup
// b owns a region of 2 T spaces per axis (the last region along an axis may
// be shorter) and keeps the region plus a one-space halo -- every cell its
// trials can read -- in LDS for the whole apply: staged once, its own cells
// updated in place by its accepted moves, and before a pass the halo cells
// that neighbours have changed and this pass is the first to read reloaded
// from the FP64 sites.  Consecutive passes are separated by a neighbour
// synchronisation (below), not by a grid barrier.
//
// An LDS entry holds the site relative to the box centre, in FP32 (mixed
// precision) or FP64, NaN for a site without images, with the body index in w.

// A region's box is staged as in k_pass_tile: ri (rows + 1 uint4: LDS offset
// of the row, first run start, first run length, second run start), coff
// (rows x (E_last + 1) LDS offsets of the cell boundaries, 16-bit: a box
// holds at most kTileLds / 16 entries), then the site entries.

// Neighbour synchronisation of the persistent apply.  Every region has one
// 64-bit progress word (kMailboxStride words apart): the launch's tag and the
// passes the region has finished in it.
//
// What a region waits for before pass j.  Its box's halo holds cells of the
// neighbour regions; a cell that lies in the halo along the axes A (a
// non-empty subset) has the space parity its side fixes: odd on the lower
// side (-1 along the axis), even on the upper one (region lengths are even).
// The trials of colour j mod 2^D sit on even cells along the axes where j's
// colour bit is 0 and read only the lower side there, on odd cells where it is
// 1 and read only the upper side.  So of the 3^D - 1 neighbours only the
// 2^D - 1 on j's sides are read, one per A, and of their cells only those of
// colours k whose bits differ from j's on every axis of A.  The region
// therefore waits, per A, until that neighbour has finished the last such
// pass k < j (k = j - 1 for one to 2^D - 1 of the subsets: three of seven on
// average in 3D), and the others may run ahead or behind.
//
// Why nothing it reads is being written.  The neighbour Y writes the cells of
// colour k in this region X's halo along A in passes of k's bits on A, which
// are exactly the passes whose sides make Y wait for X over A: before writing
// them again in pass k + 2^D (or for the first time in pass k) Y has waited
// for X's last pass with the other bits on A, which is or follows every pass of
// X that reads the values of Y's pass before.  That covers the halo copies,
// the FP64 sites that re-tests read in place, and regions staged late.
//
// The FP64 sites that neighbours read are written with device-scope stores;
// every wave waits for its stores to complete before the progress word is
// stored, and neighbours read the sites with device-scope loads (no cache
// writeback or invalidation).  Every region is resident (launch_resident), and
// the region whose pass is lowest never waits for one ahead of it, so all of them finish.  Waits are bounded: past the bound the state's
// error word is set and the wait returns, so every wave still ends.
//
// The counters that all 26 neighbours incremented every pass, which this
// replaces, made every pass last as long as the slowest of 27 regions.
// wave_publish: by the wavefront that made all of the pass's stores.
__device__ __forceinline__ void wave_publish(uint32_t* mbox, uint32_t tile, uint32_t tag, uint32_t done) {
  __builtin_amdgcn_s_waitcnt(0);  // this wave's stores have completed
  if (__lane_id() == 0)
    __hip_atomic_store((unsigned long long*)&mbox[tile * kMailboxStride], ((unsigned long long)tag << 32) | done,
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void region_publish(uint32_t* mbox, uint32_t tile, uint32_t tag, uint32_t done) {
  __builtin_amdgcn_s_waitcnt(0);  // this wave's stores have completed
  __syncthreads();
  if (threadIdx.x < 64u) wave_publish(mbox, tile, tag, done);
}

// The staged sites of a box in the region's scalar S: x, y, z and the body
// index in w (S = float: a mixed-precision region; double: an FP64 one).
template <class S>
struct Staged;
template <>
struct Staged<float> {
  using type = float4;
  __device__ __forceinline__ static float4 make(const float* r, uint32_t body) {
    return make_float4(r[0], r[1], r[2], __int_as_float((int)body));
  }
  __device__ __forceinline__ static uint32_t body(const float4& e) { return (uint32_t)__float_as_int(e.w); }
};
template <>
struct Staged<double> {
  using type = double4;
  __device__ __forceinline__ static double4 make(const double* r, uint32_t body) {
    return make_double4(r[0], r[1], r[2], __longlong_as_double((long long)body));
  }
  __device__ __forceinline__ static uint32_t body(const double4& e) { return (uint32_t)__double_as_longlong(e.w); }
};
template <class S>
using Ent = typename Staged<S>::type;

// Box-relative position: the image of x nearest the box centre c, relative to
// c, computed in FP64 and rounded once to S.  (Selects, not branches: this is
// inlined where a pass's latency counts.)
template <int D, class S, class G>
__device__ __forceinline__ void box_relative64(const G& g, const double* c, const double* x, S* r) {
#pragma unroll
  for (int a = 0; a < D; ++a) {
    const double L = g.L[a], half = g.half[a], u = x[a] - c[a];
    r[a] = (S)(u - (u >= half ? L : u < -half ? -L : 0.0));
  }
}
// LDS entry of a site: as above, NaN for a site without images (one outside
// [-L/2, L/2) on some axis, as in ghost_flags), body index in w.
template <int D, class S>
__device__ __forceinline__ Ent<S> stage_entry64(const Geometry& g, const double* c, const double* x, uint32_t body) {
  S r[3] = {0, 0, 0};
  box_relative64<D>(g, c, x, r);
#pragma unroll
  for (int a = 0; a < D; ++a)
    if (x[a] < -g.half[a] || x[a] >= g.half[a]) r[0] = (S)__builtin_nanf("");
  return Staged<S>::make(r, body);
}

// The system's constants read through the scalar cache where they are used:
// held in registers across the passes they would not fit (spilled scalars cost
// a lane read at every use).  Opaque, so that the loads stay in the loop.
typedef const __attribute__((address_space(4))) Geometry* GeoPtr;
__device__ __forceinline__ GeoPtr geo_ptr(const Geometry* self) {
  // (uniform, also where it was read from LDS)
  const uintptr_t u = (uintptr_t)self;
  uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)u), hi = __builtin_amdgcn_readfirstlane((uint32_t)(u >> 32));
  asm volatile("" : "+s"(lo), "+s"(hi));
  return (GeoPtr)(((uintptr_t)hi << 32) | lo);
}

// What a proposal x = body + displacement makes of a trial (translate moves):
// x = wrap(x) (generate_trial_moves: wrap(propose(..))), in: x lies in the
// trial's own space (multi-index own, as space_of forms it), t = wrap(x) the
// trial body and site, n = wrap(t + 0) the site update_body_properties stores
// (microstate.rs:985-1034), flags its ghost images.
//
// One lane's latency counts here, so it is all selects: a divergent branch
// costs a wavefront 40 cycles, an FP64 operation 6.  Quotients by the box
// edges and space widths are div_const_fast's; a numerator below its range, or
// constants it does not cover, take trial_site_general (a coordinate of exactly
// 0 does; other sums and differences of coordinates are far above 2^-900).
template <int D>
struct TrialSite {
  double t[3], n[3];
  uint32_t flags;
  bool in;
};
__device__ __forceinline__ double wrap_lambda(double lambda, double L) {
  lambda = lambda - round(lambda);
  return (lambda == 0.5 ? -0.5 : lambda) * L;
}
template <int D>
__device__ __noinline__ TrialSite<D> trial_site_general(const Geometry* gp, const ApplyState* st, double x0, double x1,
                                                        double x2, uint32_t s) {
  const Geometry& g = *gp;
  TrialSite<D> o;
  double x[3] = {x0, x1, x2};
  for (int a = 0; a < D; ++a) x[a] = wrap1(g, a, x[a]);
  o.in = space_of<D>(g, st->origin, x) == s;
  for (int a = 0; a < 3; ++a) o.t[a] = o.n[a] = 0.0;
  for (int a = 0; a < D; ++a) o.t[a] = wrap1(g, a, x[a]);
  for (int a = 0; a < D; ++a) o.n[a] = wrap1(g, a, o.t[a] + 0.0);
  o.flags = ghost_flags<D>(g, o.n);
  return o;
}
template <int D>
__device__ __forceinline__ TrialSite<D> trial_site(GeoPtr g, const ApplyState* st, const double* origin,
                                                   const double* x0, const uint32_t* own, uint32_t s) {
  TrialSite<D> o;
  o.in = true;
  o.flags = 0;
  o.t[2] = o.n[2] = 0.0;
  double least = 1.0;  // of the numerators' magnitudes
  bool images = true;
#pragma unroll
  for (int a = 0; a < D; ++a) {
    const double L = g->L[a], y = g->inv_L[a], wd = g->width[a], yw = g->inv_width[a];
    const double x = wrap_lambda(div_const_fast(x0[a], L, y), L);
    const double p = x - origin[a];
    double q = floor(div_const_fast(p, wd, yw));
    q = q == (double)g->shape[a] ? 0.0 : q;
    o.in = o.in & (q == (double)own[a]);
    const double t = wrap_lambda(div_const_fast(x, L, y), L);
    const double n = wrap_lambda(div_const_fast(t + 0.0, L, y), L);
    least = fmin(fmin(least, fabs(x0[a])), fmin(fmin(fabs(x), fabs(p)), fabs(t)));
    least = fmin(least, fmin(y, yw));
    o.t[a] = t;
    o.n[a] = n;
    images = images & (n >= -g->half[a]) & (n < g->half[a]);
    o.flags |= (n > g->ghost_hi[a] ? 2u : n < g->ghost_lo[a] ? 1u : 0u) << (2 * a);
  }
  o.flags = images ? o.flags : kNoImages;
  if (!(least >= 0x1p-900)) o = trial_site_general<D>((const Geometry*)(uintptr_t)g, st, x0[0], x0[1], D == 3 ? x0[2] : 0.0, s);
  return o;
}
// Squared distances from a site in space `own` to the space's lower and upper
// faces (0 where it lies beyond one by rounding).
template <int D>
__device__ __forceinline__ void face_gaps2(GeoPtr g, const double* origin, const uint32_t* own, const double* x,
                                           float* lo, float* hi) {
#pragma unroll
  for (int a = 0; a < D; ++a)
    face_gap2(x[a] - origin[a], (double)own[a], g->width[a], g->L[a], &lo[a], &hi[a]);
}

// The neighbour spaces of a trial (each once, as the reference's cell list
// visits them) as rows along the last axis, listed by a group of G lanes, a lane
// per row.  issue() loads each row's slots, before the proposal is drawn; list()
// writes its runs to LDS and returns the number of candidates.
//
// With three or more spaces along every axis and a scan of one space (`plain`), a row
// is a lower, an own and an upper space, and rows and row ends whose nearest
// point is the cutoff away are left out: 27 spaces become 20 on average.
// (face_gaps2 to the faces; cut2 holds a margin for its roundings.)  Otherwise a
// row is one run of slots, or two across the periodic face.
template <int D, int G>
struct NeighbourRows {
  static constexpr uint32_t kRows = D == 3 ? 25 : 5, H = (kRows + G - 1) / G;  // at most 5^(D - 1) rows
  uint32_t nrow, nn1, inv1;
  bool plain;
  uint32_t e[H][6];  // plain: first and last slots of the lower, own and upper space; else of the two runs
  __device__ __forceinline__ void issue(const Geometry& g, const uint32_t* start, const int32_t* m, bool have,
                                        uint32_t kl) {
    constexpr int AL = D - 1;
    uint32_t nn[3] = {1, 1, 1}, first[3] = {0, 0, 0};
    plain = true;
#pragma unroll
    for (int a = 0; a < D; ++a) plain = plain && g.reach[a] == 1 && g.shape[a] >= 3;
#pragma unroll
    for (int a = 0; a < D; ++a) {
      const uint32_t sh = (uint32_t)g.shape[a], r = (uint32_t)g.reach[a], x = (uint32_t)m[a];
      const bool all = 2u * r + 1u >= sh && !plain;  // (of three spaces, too, the lower one comes first)
      nn[a] = min(2u * r + 1u, sh);
      first[a] = all ? 0u : (x >= r ? x - r : x + sh - r);
    }
    nn1 = D == 3 ? nn[1] : 1u;
    nrow = D == 3 ? nn[0] * nn[1] : nn[0];
    inv1 = (256u + nn1 - 1u) / nn1;
    const uint32_t sh = (uint32_t)g.shape[AL], ml = (uint32_t)m[AL];
#pragma unroll
    for (uint32_t h = 0; h < H; ++h) {
#pragma unroll
      for (int q = 0; q < 6; ++q) e[h][q] = 0;
      const uint32_t j = kl + h * G;
      if (!have || j >= nrow) continue;
      const uint32_t i0 = (j * inv1) >> 8, i1 = j - i0 * nn1;
      uint32_t y0 = first[0] + i0;
      y0 = y0 >= (uint32_t)g.shape[0] ? y0 - (uint32_t)g.shape[0] : y0;
      uint32_t sb = y0 * g.stride[0];
      if constexpr (D == 3) {
        const uint32_t y1 = first[1] + i1;
        sb += (y1 >= (uint32_t)g.shape[1] ? y1 - (uint32_t)g.shape[1] : y1) * g.stride[1];
      }
      if (plain) {
        const uint32_t lo = sb + first[AL], mid = sb + ml, hi = sb + (ml + 1u == sh ? 0u : ml + 1u);
        e[h][0] = start[lo];
        e[h][1] = start[lo + 1u];
        e[h][2] = start[mid];
        e[h][3] = start[mid + 1u];
        e[h][4] = start[hi];
        e[h][5] = start[hi + 1u];
      } else {
        const uint32_t end = first[AL] + nn[AL];
        e[h][2] = start[sb + first[AL]];
        e[h][3] = start[sb + min(end, sh)];
        e[h][4] = start[sb];
        e[h][5] = end > sh ? start[sb + end - sh] : e[h][4];
      }
    }
  }
  // rows[j] = {first slot of the first run, its length, second run's first slot
  // less that length, index of the row's first candidate}
  __device__ __forceinline__ uint32_t list(const Geometry& g, const int32_t* m, uint32_t kl, bool active, float cut2,
                                           const float* flo, const float* fhi, uint4* rows) const {
    constexpr int AL = D - 1;
    const bool wlo = m[AL] == 0, whi = m[AL] + 1 == g.shape[AL];  // the lower / upper space lies across the face
    uint32_t tot = 0;
#pragma unroll
    for (uint32_t h = 0; h < H; ++h) {
      if (h && h * G >= nrow) break;  // uniform
      const uint32_t j = kl + h * G;
      const bool mine = active && j < nrow;
      uint32_t ra = e[h][2], ea = e[h][3], rb = e[h][4], eb = e[h][5];
      if (plain) {
        const uint32_t i0 = (j * inv1) >> 8, i1 = j - i0 * nn1;
        float d = i0 == 0 ? flo[0] : i0 == 2 ? fhi[0] : 0.0f;
        if constexpr (D == 3) d += i1 == 0 ? flo[1] : i1 == 2 ? fhi[1] : 0.0f;
        const bool lo = !(d + flo[AL] >= cut2), hi = !(d + fhi[AL] >= cut2);
        ra = lo && !wlo ? e[h][0] : ra;
        ea = hi && !whi ? e[h][5] : ea;
        rb = wlo ? e[h][0] : e[h][4];
        eb = wlo ? (lo ? e[h][1] : rb) : (whi && hi ? e[h][5] : rb);
        if (d >= cut2) ea = ra, eb = rb;
      }
      const uint32_t la = ea - ra, cnt = mine ? la + (eb - rb) : 0u;
      uint32_t incl = cnt;
#pragma unroll
      for (uint32_t dd = 1; dd < G; dd <<= 1) {
        const uint32_t u = __shfl_up(incl, dd, G);
        if (kl >= dd) incl += u;
      }
      if (mine) rows[j] = make_uint4(ra, la, rb - la, tot + incl - cnt);
      tot += __shfl(incl, (int)(__lane_id() | (G - 1)), 64);
    }
    return tot;
  }
  // slot of candidate c: in the last row whose first candidate is <= c
  __device__ __forceinline__ uint32_t slot_of(const uint4* rows, uint32_t c) const {
    uint32_t j = 0;
    for (uint32_t sw = nrow > 16u ? 16u : 8u; sw >= 1; sw >>= 1) {
      const uint32_t mid = j + sw;
      if (mid < nrow && rows[mid].w <= c) j = mid;
    }
    const uint4 q = rows[j];
    const uint32_t i = c - q.w;
    return (i < q.y ? q.x : q.z) + i;
  }
};

// Residency probe (tc.probe): the persistent launch relies on every region
// being resident at once, which the host checks with the occupancy API; the
// probe checks it on the device with the kernel's own resources.  Thread 0 of
// every region adds 1 to a counter (word 2 of region 0's mailbox) and waits,
// bounded, until all regions have arrived; a region that times out sets
// kErrBarrier.  Every wavefront of the workgroup stays until then (a
// wavefront that ended early would free its SIMD slot and registers for a
// later workgroup, which the real apply does not).  The host clears the
// counter after the probe.
__device__ __forceinline__ void region_probe(ApplyState* st, uint32_t* mbox, uint32_t ntiles) {
  if (threadIdx.x == 0) {
    uint32_t* ctr = &mbox[2];
    __hip_atomic_fetch_add(ctr, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    uint32_t spins = 0;
    while (__hip_atomic_load(ctr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < ntiles) {
      __builtin_amdgcn_s_sleep(1);
      if (++spins > kBarrierSpins / 16) {
        atomicOr(&st->error, kErrBarrier);
        break;
      }
    }
  }
  __syncthreads();
}

// Geometry of region `tile`: its spaces org .. org + rl - 1 per axis, its box
// org - 1 .. org + 2 T (E spaces), the two slot runs of every box row along
// the last axis (p cells from m0, then the rest from 0) and the box centre.
struct Region {
  uint32_t tcd[3];
  int32_t org[3], mlo[3], rl[3];
  uint32_t p, m0;
  double c64[3];
};

// Position of a region whose sites are not staged, and its space for trial t of
// a colour (false: none there).
template <int D>
__device__ __forceinline__ Region wave_region(const Geometry& g, const TileCfg& tc, uint32_t tile) {
  Region rg{};
  for (int a = D - 1; a >= 0; --a) {
    rg.tcd[a] = tile % tc.nt[a];
    tile /= tc.nt[a];
    rg.org[a] = (int32_t)(2 * rg.tcd[a] * tc.T[a]);
    rg.rl[a] = min((int32_t)(2 * tc.T[a]), g.shape[a] - rg.org[a]);
  }
  return rg;
}
template <int D>
__device__ __forceinline__ bool wave_region_space(const Geometry& g, const TileCfg& tc, const Region& rg,
                                                  uint32_t colour, uint32_t t, uint32_t* s, int32_t* m) {
  bool have = t < tc.trials;
  uint32_t sp = 0;
  m[0] = m[1] = m[2] = 0;
#pragma unroll
  for (int a = D - 1; a >= 0; --a) {
    const int32_t l = (int32_t)(2 * (t % tc.T[a]) + ((colour >> (D - 1 - a)) & 1u));
    t /= tc.T[a];
    have = have && l < rg.rl[a];
    m[a] = rg.org[a] + l;
    sp += (uint32_t)m[a] * g.stride[a];
  }
  *s = have ? sp : 0u;
  return have;
}

template <int D>
__device__ __forceinline__ Region region_of(const Geometry& g, const TileCfg& tc, const double* origin,
                                            uint32_t tile) {
  constexpr int AL = D - 1;
  Region rg{};
  uint32_t r = tile;
  for (int a = D - 1; a >= 0; --a) {
    rg.tcd[a] = r % tc.nt[a];
    r /= tc.nt[a];
  }
  for (int a = 0; a < 3; ++a) {
    rg.org[a] = 0;
    rg.mlo[a] = 0;
    rg.rl[a] = 1;
    rg.c64[a] = 0.0;
  }
  for (int a = 0; a < D; ++a) {
    rg.org[a] = (int32_t)(2 * rg.tcd[a] * tc.T[a]);
    rg.mlo[a] = rg.org[a] - 1;
    rg.rl[a] = min((int32_t)(2 * tc.T[a]), g.shape[a] - rg.org[a]);
  }
  const int32_t SL = g.shape[AL], ml = rg.mlo[AL], EL = (int32_t)tc.E[AL];
  rg.p = ml < 0 ? 1u : (uint32_t)min(EL, SL - ml);
  rg.m0 = (uint32_t)(ml < 0 ? ml + SL : ml);
  for (int a = 0; a < D; ++a) {
    double c = origin[a] + ((double)rg.mlo[a] + 0.5 * (double)tc.E[a]) * g.width[a];
    c -= g.L[a] * floor((c + g.half[a]) / g.L[a]);
    rg.c64[a] = c;
  }
  return rg;
}

// Passes back from pass j to the last one whose colour differs from j's on
// every axis of `axes` (colour-bit mask, non-zero): 1 .. 2^D - 1.
__host__ __device__ __forceinline__ uint32_t pass_distance(uint32_t j, uint32_t axes) {
  uint32_t d = 1;
  while ((((j - d) ^ j) & axes) != axes) ++d;
  return d;
}

// Waits before pass j for the neighbours on j's sides (lane A - 1 of the
// wavefront: the axes A).  Every wavefront polls for itself, so that each goes
// on to its halo loads without a barrier.
template <int D>
__device__ __forceinline__ void region_wait(ApplyState* st, uint32_t* mbox, const TileCfg& tc, const Region& rg,
                                            uint32_t tile, uint32_t j) {
  constexpr uint32_t NS = (1u << D) - 1u;
  const uint32_t lane = __lane_id();
  if (lane < NS) {
    const uint32_t axes = lane + 1u, d = pass_distance(j, axes);
    uint32_t nb = 0;
#pragma unroll
    for (int a = 0; a < D; ++a) {
      const uint32_t bit = 1u << (D - 1 - a), n = tc.nt[a];
      uint32_t t = rg.tcd[a];
      if (axes & bit) t = (j & bit) ? (t + 1u == n ? 0u : t + 1u) : (t == 0u ? n - 1u : t - 1u);
      nb = nb * n + t;
    }
    if (j >= d && nb != tile) {
      const uint32_t need = j - d + 1u;
      const unsigned long long* word = (const unsigned long long*)&mbox[nb * kMailboxStride];
      uint32_t spins = 0;
      for (;;) {
        const unsigned long long v = __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if ((uint32_t)(v >> 32) == tc.tag && (uint32_t)v >= need) break;
        __builtin_amdgcn_s_sleep(1);
        if (++spins > kBarrierSpins) {
          atomicOr(&st->error, kErrBarrier);
          atomicCAS(&st->wait_at, 0u, (tile << 12) | ((j & 0xfffu) + 1u));
          break;
        }
      }
    }
  }
  // (no later load of this wavefront moves above the polls)
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// LDS of a region's box: ri (staging only), whose space the halo cell lists
// take over afterwards, coff, then the site entries.
template <class S>
struct RegionLds {
  uint4* ri;
  uint16_t* halo;
  uint16_t* coff;
  Ent<S>* lb;
};
// bytes of ri / the halo lists
__host__ __device__ inline uint32_t region_head_bytes(uint32_t rows, uint32_t halo_cells) {
  const uint32_t a = 16u * (rows + 1), b = (2u * halo_cells + 15u) & ~15u;
  return a > b ? a : b;
}
template <int D, class S>
__device__ __forceinline__ RegionLds<S> region_lds(unsigned char* smem, const TileCfg& tc) {
  const uint32_t R = tc.rows, CW = tc.E[D - 1] + 1;
  const uint32_t head = region_head_bytes(R, tc.hoff[kHaloLists]);
  RegionLds<S> l;
  l.ri = (uint4*)smem;
  l.halo = (uint16_t*)smem;
  l.coff = (uint16_t*)(smem + head);
  l.lb = (Ent<S>*)(smem + ((head + 2u * R * CW + 15u) & ~15u));
  return l;
}

// Stages the region's box into LDS once per apply: every row's runs and cell
// starts, then the sites (their FP64 copies as box-relative FP32 entries with
// the body index).  A thread per row loads its runs, wave 0 scans the row
// lengths, and a half-wave per row copies its cell starts and its runs,
// kStageRows rows in flight together.  Ends with a barrier; returns the number of
// sites (uniform over the workgroup) when it exceeds the LDS capacity tc.maxb, in
// which case no entries were written, else 0.  PAD entries out of reach follow the
// box's.  *odd (zeroed before) is set when a staged site has
// no images, i.e. its entry is NaN.
//
// Written for few instructions: every launch fetches its code anew, a cache
// line at a time, and straight-line code that runs once costs more in fetches
// than in execution.  (With the cell starts taken 16 to a thread in unrolled
// loops and the image selection in branches, the part of the kernel before
// the first trial took 50 us of C2's 280 us apply.)
template <int D, class S, int PAD>
__device__ __forceinline__ uint32_t region_stage(const Geometry& g, const TileCfg& tc, const Region& rg, const Bodies& B,
                                             const Cells& C, const Work& w, const RegionLds<S>& l, uint32_t* odd) {
  constexpr int AL = D - 1;
  const uint32_t R = tc.rows, EL = tc.E[AL], CW = EL + 1;
  const uint32_t tid = threadIdx.x, NT = blockDim.x;
  const uint32_t p = rg.p, m0 = rg.m0;
  uint4* ri = l.ri;
  uint16_t* coff = l.coff;
  Ent<S>* lb = l.lb;
  // per row: its runs' lengths, first slots and the space it starts at (a run
  // past 16 bits is no box that fits)
  const uint32_t e1m = D == 3 ? (65536u + tc.E[1] - 1u) / tc.E[1] : 0u;  // row / E1 (rows <= 256)
  for (uint32_t r = tid; r < R; r += NT) {
    const uint32_t e0 = D == 3 ? (r * e1m) >> 16 : r;
    const uint32_t e[2] = {e0, D == 3 ? r - e0 * tc.E[1] : 0u};
    uint32_t sb = 0;
#pragma unroll
    for (int a = 0; a < AL; ++a) {
      const int32_t sh = g.shape[a], mm = rg.mlo[a] + (int32_t)e[a];
      sb += (uint32_t)(mm < 0 ? mm + sh : (mm >= sh ? mm - sh : mm)) * g.stride[a];
    }
    const uint32_t a0 = w.start[sb + m0], a1 = w.start[sb + m0 + p], b0 = w.start[sb], b1 = w.start[sb + (EL - p)];
    ri[r] = make_uint4(min(a1 - a0, 0xffffu) | (min(b1 - b0, 0xffffu) << 16), a0, b0, sb);
  }
  __syncthreads();
  if (tid < 64) {
    const uint32_t rpl = (R + 63) / 64, r0 = tid * rpl, r1 = min(r0 + rpl, R);
    uint32_t sum = 0;
    for (uint32_t r = r0; r < r1; ++r) sum += (ri[r].x & 0xffffu) + (ri[r].x >> 16);
    const uint32_t incl = wave_incl_scan(sum);
    uint32_t off = incl - sum;
    for (uint32_t r = r0; r < r1; ++r) {
      const uint32_t x = ri[r].x;
      ri[r].x = (off & 0xffffu) | (x << 16);  // LDS offset, first run's length
      off += (x & 0xffffu) + (x >> 16);
    }
    if (tid == 63) ri[R].x = incl;
  }
  __syncthreads();
  const uint32_t total = ri[R].x;
  const bool overflow = total > tc.maxb;  // uniform over the workgroup; else every offset fits 16 bits
  if (!overflow) {
    if (tid < (uint32_t)PAD) lb[total + tid] = Ent<S>{(S)kTileFar, 0, 0, 0};
    const uint32_t hw = tid >> 5, hl = tid & 31u, NH = NT >> 5;
    // boundary j of a row (j <= p) is the start of space m0 + j, the next ones
    // that of j - p - 1 after the wrap; its LDS offset is written at j or j - 1
    auto boundary = [&](const uint4& q, uint32_t r, uint32_t j, uint32_t start) {
      const uint32_t o = q.x & 0xffffu;
      coff[r * CW + (j <= p ? j : j - 1)] = (uint16_t)(j <= p ? o + (start - q.y) : o + (q.x >> 16) + (start - q.z));
    };
    auto slot_of = [&](const uint4& q, uint32_t e) {
      return e < (q.x >> 16) ? q.y + e : q.z + (e - (q.x >> 16));
    };
    auto put = [&](uint32_t dst, const double4& sp, uint32_t body) {
      const double x[3] = {sp.x, sp.y, sp.z};
      const Ent<S> en = stage_entry64<D, S>(g, rg.c64, x, body);
      lb[dst] = en;
      if (!(en.x == en.x)) *odd = 1;
    };
#pragma unroll 1
    for (uint32_t r0 = hw; r0 < R; r0 += NH * kStageRows) {
      uint4 q[kStageRows];
      uint32_t len[kStageRows], bod[kStageRows], raw[kStageRows];
#pragma unroll
      for (int u = 0; u < kStageRows; ++u) {
        const uint32_t r = min(r0 + (uint32_t)u * NH, R - 1);
        q[u] = ri[r];
        len[u] = (ri[r + 1].x & 0xffffu) - (q[u].x & 0xffffu);
        if (r0 + (uint32_t)u * NH >= R) len[u] = 0;
        if (hl < len[u]) bod[u] = C.body[slot_of(q[u], hl)];
        if (hl < EL + 2) raw[u] = w.start[q[u].w + (hl <= p ? m0 + hl : hl - p - 1)];
      }
      double4 tmp[kStageRows];
#pragma unroll
      for (int u = 0; u < kStageRows; ++u)
        if (hl < len[u]) tmp[u] = B.spos[bod[u]];
#pragma unroll
      for (int u = 0; u < kStageRows; ++u) {
        const uint32_t r = min(r0 + (uint32_t)u * NH, R - 1);  // (the last row again: the same values)
        if (hl < EL + 2) boundary(q[u], r, hl, raw[u]);
        if (hl < len[u]) put((q[u].x & 0xffffu) + hl, tmp[u], bod[u]);
      }
      // entries and boundaries past the first 32 of a row
#pragma unroll 1
      for (int u = 0; u < kStageRows; ++u) {
        const uint32_t r = min(r0 + (uint32_t)u * NH, R - 1);
        const uint4 qr = ri[r];
        const uint32_t o = qr.x & 0xffffu, n = (ri[r + 1].x & 0xffffu) - o;
        for (uint32_t e = 32u + hl; e < max(n, EL + 2); e += 32u) {
          if (e < EL + 2) boundary(qr, r, e, w.start[qr.w + (e <= p ? m0 + e : e - p - 1)]);
          if (e < n) {
            const uint32_t bd = C.body[slot_of(qr, e)];
            put(o + e, B.spos[bd], bd);
          }
        }
      }
    }
  }
  __syncthreads();
  return overflow ? total : 0u;
}

// The halo cells of the box by the pass class (pass mod 2^D) that first reads
// them after they change: list q holds, at halo[hoff[q]], the hcnt[q] cells
// (index of their first boundary in coff) to reload before the passes j = q
// (mod 2^D).  A cell of colour k in the halo along A is first read in the next
// pass whose bits differ from k's on A.  Geometry alone decides, so the lists'
// places are those of a full region (hoff, filled by the host); a shorter
// region at the end of an axis has no more cells in any of them.  hcnt must be
// zero, and a barrier must separate the staging from this and this from the
// first reload.  (Listing by cell, not by entry: no capacity to overflow, and
// built while the first proposals are drawn.)
template <int D>
__host__ __device__ __forceinline__ uint32_t halo_list(const int32_t* lc, const int32_t* rl) {
  uint32_t axes = 0, k = 0;
  for (int a = 0; a < D; ++a) {
    const uint32_t bit = 1u << (D - 1 - a);
    if (lc[a] > rl[a]) return UINT32_MAX;  // past the halo of a short region
    if (lc[a] < 0 || lc[a] == rl[a]) axes |= bit;
    if (lc[a] & 1) k |= bit;  // (-1 is odd)
  }
  if (!axes) return UINT32_MAX;
  uint32_t d = 1;
  while (((k ^ (k + d)) & axes) != axes) ++d;
  return (k + d) & ((1u << D) - 1u);
}
template <int D, class S>
__device__ __forceinline__ void region_halo_lists(const TileCfg& tc, const Region& rg, const RegionLds<S>& l,
                                                  uint32_t* hcnt) {
  constexpr int AL = D - 1;
  const uint32_t EL = tc.E[AL], E1 = D == 3 ? tc.E[1] : 1u;
  const uint32_t elm = 0xffffffffu / EL + 1u, e1m = (65536u + E1 - 1u) / E1;  // / EL, / E1
#pragma unroll 1
  for (uint32_t ci = threadIdx.x; ci < tc.ncell; ci += blockDim.x) {
    const uint32_t row = __umulhi(ci, elm), j = ci - row * EL, e0 = D == 3 ? (row * e1m) >> 16 : row;
    const int32_t lc[3] = {(int32_t)e0 - 1, D == 3 ? (int32_t)(row - e0 * E1) - 1 : (int32_t)j - 1, (int32_t)j - 1};
    const uint32_t q = halo_list<D>(lc, rg.rl);
    if (q != UINT32_MAX) l.halo[tc.hoff[q] + atomicAdd(&hcnt[q], 1u)] = (uint16_t)(row * (EL + 1) + j);
  }
}

// After the wait before pass j: reloads the halo cells whose new values pass j
// is the first to read, from the FP64 sites with device-scope loads.  LPC lanes
// per cell (lane `sub` takes entries sub, sub + LPC, ...).  issue() puts HELD
// entries of CELLS cells per lane in flight together; commit() writes
// their LDS entries and takes whatever is left (cells of more than HELD LPC
// entries, lists of more than CELLS NT / LPC cells), one memory latency
// per round.  *odd is set where an entry is NaN (a site without images).  No
// barrier: one must follow before other wavefronts read the entries.
template <int D, class S, int LPC, int CELLS, int HELD>
struct RegionReload {
  const Geometry& g;
  const Region& rg;
  const Bodies& B;
  const RegionLds<S>& l;
  const uint16_t* list;
  uint32_t n, step, c0;
  uint32_t e[CELLS], eb[CELLS];
  double v[CELLS][HELD][3];

  __device__ __forceinline__ RegionReload(const Geometry& g_, const TileCfg& tc, const Region& rg_, const Bodies& B_,
                                          const RegionLds<S>& l_, const uint32_t* hcnt, uint32_t j,
                                          uint32_t threads = blockDim.x)
      : g(g_), rg(rg_), B(B_), l(l_) {
    const uint32_t q = j & ((1u << D) - 1u);
    n = threadIdx.x < threads ? hcnt[q] : 0u;
    list = l.halo + tc.hoff[q];
    step = threads / LPC;
    c0 = threadIdx.x / LPC;
  }
  __device__ __forceinline__ void issue() {
    const uint32_t sub = threadIdx.x % LPC;
#pragma unroll
    for (int u = 0; u < CELLS; ++u) {
      const uint32_t c = c0 + (uint32_t)u * step;
      e[u] = eb[u] = 0;
      if (c < n) {
        const uint32_t cell = list[c];
        e[u] = l.coff[cell] + sub;
        eb[u] = l.coff[cell + 1];
      }
    }
    uint32_t bd[CELLS][HELD];
#pragma unroll
    for (int u = 0; u < CELLS; ++u)
#pragma unroll
      for (int h = 0; h < HELD; ++h)
        if (e[u] + (uint32_t)(h * LPC) < eb[u]) bd[u][h] = Staged<S>::body(l.lb[e[u] + (uint32_t)(h * LPC)]);
#pragma unroll
    for (int u = 0; u < CELLS; ++u)
#pragma unroll
      for (int h = 0; h < HELD; ++h)
        if (e[u] + (uint32_t)(h * LPC) < eb[u]) fetch(bd[u][h], v[u][h]);
  }
  __device__ __forceinline__ void fetch(uint32_t body, double* sp) const {
    const double* q = (const double*)&B.spos[body];
#pragma unroll
    for (int a = 0; a < D; ++a) sp[a] = __longlong_as_double((long long)ld_dev(q + a));
  }
  __device__ __forceinline__ void put(uint32_t x, const double* sp, uint32_t* odd) const {
    const Ent<S> en = stage_entry64<D, S>(g, rg.c64, sp, Staged<S>::body(l.lb[x]));
    l.lb[x] = en;
    if (!(en.x == en.x)) *odd = 1;
  }
  __device__ __forceinline__ void commit(uint32_t* odd) {
#pragma unroll
    for (int u = 0; u < CELLS; ++u)
#pragma unroll
      for (int h = 0; h < HELD; ++h)
        if (e[u] + (uint32_t)(h * LPC) < eb[u]) put(e[u] + (uint32_t)(h * LPC), v[u][h], odd);
    // what is left: entries past HELD of the cells in hand, then further cells
    uint32_t c = c0, held = (uint32_t)(HELD * LPC);
#pragma unroll 1
    for (; c < n; c += step) {
      if (c >= c0 + CELLS * step) held = 0;
      const uint32_t cell = list[c];
#pragma unroll 1
      for (uint32_t x = l.coff[cell] + threadIdx.x % LPC + held; x < l.coff[cell + 1]; x += LPC) {
        double sp[3];
        fetch(Staged<S>::body(l.lb[x]), sp);
        put(x, sp, odd);
      }
    }
  }
};

}  // namespace hmc
