// Isotropic pair energies (LJ, shifted LJ, the overlap penalty) in FP64, systems
// beyond k_apply_small: a group of G lanes per trial, 64 / G trials per wavefront.
//
// A trial of the overlap penalty has 20 candidates, one of LJ 300. A wavefront per
// trial and a launch per pass (48 us per pass of 17,576 trials) spent its time on
// the chain of one trial, with 20 of 64 lanes in use and eleven wavefronts per
// slot one after another.  Measured us per step, before and now: 131,072
// overlap-penalty bodies 1049 and 254, 16,384 288 and 157; LJ at density 0.8,
// 2,048 bodies 5270 and 2887, 131,072 2445 and 1447, 442,368 (one launch per
// colour) 3012 and 2239.  Bound by the latency of a pass's chain (start slots,
// body, proposal, candidates, decision), about 11 us.
#include "persist.hpp"

namespace hmc {

constexpr uint32_t kIsoBatch = 4;  // rounds of G candidates with their loads in flight together

template <int D, int G>
struct IsoWave {
  static constexpr uint32_t kTrials = 64 / G, kRows = NeighbourRows<D, G>::kRows, kCap = 2 * kIsoBatch * G;
  uint4 row[kTrials][kRows];     // (NeighbourRows)
  double list[kTrials][kCap];    // squared distances within the cutoff (negative: the initial site's)
};

template <int G>
__device__ __forceinline__ double group_sum(double v) {
#pragma unroll
  for (int d = G / 2; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
  return v;
}

// The trials of one wavefront: lane group k's in space s (multi-index m) where
// `have` holds (all lanes of a group alike), each the one of trial_lj
// (parallel_sweep.rs:234-277) with FP64 energies.  A group lists its rows of
// neighbour spaces, draws the proposal, and calls ready() (by the whole
// wavefront) before it reads other spaces' sites; its lanes then share out the
// candidate sites.  Squared distances within the cutoff are listed and the
// energies (a square root and a division each) evaluated from the list.
// Energies, magnitudes and counts are summed over the group and decided with
// the bound on the summation-order difference.  DEV: sites are read and stored
// with device scope (the persistent apply).
template <int D, int G, bool DEV, class Ready>
__device__ __forceinline__ void iso_trials(const Geometry& g, ApplyState* st, const Bodies& B, const Cells& C,
                                           const Work& w, IsoWave<D, G>& W, const double* zx, const double* zf,
                                           bool have, uint32_t s, const int32_t* m, uint32_t colour, uint32_t substep,
                                           unsigned* blk_acc, Ready ready) {
  constexpr uint32_t kBatch = kIsoBatch;
  const uint32_t lane = __lane_id(), k = lane / G, kl = lane % G;
  const GeoPtr gp = geo_ptr(g.self);
  NeighbourRows<D, G> nbr;
  nbr.issue(g, w.start, m, have, kl);
  bool tried = false;
  uint32_t slot = 0xFFFFFFFFu, body = 0;
  Sfc64 rng = {0, 0, 0, 0};
  if (have) {
    const uint32_t s0 = w.start[s];
    const uint32_t n = w.start[s + 1] - s0;
    if (n) {
      tried = true;
      rng = counter_rng<DEV>(st->step, substep, st->seed, s);
      slot = s0 + choose_index(rng, n);
      body = C.body[slot];
    }
  }
  if (!DEV && G == 64 && !tried) return;  // (uniform; half of 50,000 LJ bodies' time where 63 of 64 spaces are empty)
  double4 bp = make_double4(0.0, 0.0, 0.0, 0.0), sp = bp;
  double v[3] = {0.0, 0.0, 0.0};
  TrialSite<D> ts{};
  const double origin[3] = {st->origin[0], st->origin[1], st->origin[2]};
  const uint32_t own[3] = {(uint32_t)m[0], (uint32_t)m[1], (uint32_t)m[2]};
  if (tried) {
    bp = B.bpos[body];
    sp = B.spos[body];
    ball_sample<D>(rng, st->max_move, zx, zf, v);
    const double x0[3] = {bp.x + v[0], bp.y + v[1], bp.z + v[2]};
    ts = trial_site<D>(gp, st, origin, x0, own, s);
  }
  const bool active = tried && ts.in;
  const double xi[3] = {sp.x, sp.y, sp.z};
  float flo[3], fhi[3], glo[3], ghi[3];
  face_gaps2<D>(gp, origin, own, ts.t, flo, fhi);
  face_gaps2<D>(gp, origin, own, xi, glo, ghi);
#pragma unroll
  for (int a = 0; a < D; ++a) {
    flo[a] = fminf(flo[a], glo[a]);
    fhi[a] = fminf(fhi[a], ghi[a]);
  }
  const uint32_t tot = nbr.list(g, m, kl, active, g.row_cut2, flo, fhi, W.row[k]);
  wave_lds_order();
  ready();
  double ef = 0.0, ei = 0.0, mag = 0.0;
  uint32_t nf = 0, ni = 0, nl = 0;  // (the same in a group's lanes)
  const uint32_t sh = k * G;
  constexpr unsigned long long kGroup = G == 64 ? ~0ull : (1ull << (G & 63)) - 1ull;
  const unsigned long long below = (1ull << kl) - 1ull;
  double* ls = W.list[k];
  for (uint32_t c0 = 0; __any(c0 < tot); c0 += G * kBatch) {
    uint32_t qv[kBatch];
    bool ok[kBatch];
#pragma unroll
    for (uint32_t r = 0; r < kBatch; ++r) {
      const uint32_t c = c0 + G * r + kl;
      ok[r] = c < tot;
      qv[r] = ok[r] ? nbr.slot_of(W.row[k], c) : slot;
      ok[r] = ok[r] && qv[r] != slot;
    }
    double4 sjv[kBatch];
#pragma unroll
    for (uint32_t r = 0; r < kBatch; ++r) {
      sjv[r] = make_double4(0.0, 0.0, 0.0, 0.0);
      if (ok[r]) {
        if constexpr (DEV)
          sjv[r] = ld_dev_d4(&C.pos64[qv[r]]);
        else
          sjv[r] = C.pos64[qv[r]];
      }
    }
#pragma unroll
    for (uint32_t r = 0; r < kBatch; ++r) {
      if (!__any(ok[r])) break;
      const double r2f = lj_r2<D>(g, ts.t, sjv[r]), r2i = lj_r2<D>(g, xi, sjv[r]);
      const bool inf_ = ok[r] && r2f < g.lj_rc2, ini = ok[r] && r2i < g.lj_rc2;
      const unsigned long long mf = (__ballot(inf_) >> sh) & kGroup, mi = (__ballot(ini) >> sh) & kGroup;
      const uint32_t cf = (uint32_t)__popcll(mf), ci = (uint32_t)__popcll(mi);
      if (inf_) ls[nl + (uint32_t)__popcll(mf & below)] = r2f;
      if (ini) ls[nl + cf + (uint32_t)__popcll(mi & below)] = -r2i;
      nl += cf + ci;
      nf += cf;
      ni += ci;
    }
    wave_lds_order();
    for (uint32_t q = kl; __any(q < nl); q += G) {
      if (q >= nl) continue;
      const double r2 = ls[q], en = lj_energy(g, fabs(r2));
      const bool fin = __double_as_longlong(r2) >= 0;
      ef += fin ? en : 0.0;
      ei += fin ? 0.0 : en;
      mag += fabs(en);
    }
    nl = 0;
    wave_lds_order();
  }
  ef = group_sum<G>(ef);
  ei = group_sum<G>(ei);
  mag = group_sum<G>(mag);
  if (kl == 0 && tried) {
    bool accept = false;
    if (active) {
      // energy_final - energy_initial (pairwise_cutoff.rs:919-941): an infinite
      // final energy is rejected, an infinite initial one accepted
      if (ef == INFINITY) {
        accept = false;
      } else if (ei == INFINITY) {
        accept = true;
      } else {
        const double dH = ef - ei;
        const double nmax = (double)max(max(nf, ni), 1u);
        const double gam = nmax * 0x1p-53 * (1.0 + 0x1p-20);  // >= n u / (1 - n u) for n < 2^32
        const double delta = (2.0 * gam * mag + 0x1p-52 * fabs(dH)) * (1.0 + 0x1p-20) + 0x1p-1070;
        bool amb = false;
        accept = lj_metropolis(rng, dH, delta, st->kT, &amb) != 0;
        if (amb) atomicAdd(&st->ambiguous, 1ull);
      }
    }
    if (accept) {
      // update_body_properties (microstate.rs:985-1034)
      B.bpos[body] = make_double4(ts.t[0], ts.t[1], ts.t[2], move_stamp(st->epoch));
      const double4 np = pack_site(ts.n, ts.flags);
      B.spos[body] = np;
      if constexpr (DEV)
        st_dev_d4(&C.pos64[slot], np);
      else
        C.pos64[slot] = np;
      atomicAdd(blk_acc, 1u);
    }
    if (w.tracing) {
      unsigned long long ti = atomicAdd((unsigned long long*)&st->trace_n, 1ull);
      if (ti < w.trace_cap) {
        hmc_trace_record rec;
        rec.substep = substep;
        rec.color = colour;
        rec.space = s;
        rec.body = (int64_t)body;
        rec.status = accept ? 1 : 0;
        rec.pad = 0;
        w.trace[ti] = rec;
      }
    }
  }
}

// One colour of one cycle.  (Four wavefronts per SIMD: the registers allow it.)
template <int D, int G>
__global__ void __launch_bounds__(kBlock, 4) k_pass_iso(Geometry g, ApplyState* st, Bodies B, Cells C, Work w,
                                                     uint32_t colour, uint32_t cycle, uint32_t xcd_chunk) {
  if (cycle >= st->cycles) return;  // uniform over the grid
  __shared__ double zx[257], zf[257];
  __shared__ unsigned blk_acc;
  __shared__ IsoWave<D, G> iw[kBlock / 64];
  if (D == 3) stage_zig(zx, zf);
  if (threadIdx.x == 0) blk_acc = 0;
  __syncthreads();
  const uint32_t b = blockIdx.x;
  const uint32_t lb = (b & 7u) * xcd_chunk + (b >> 3);
  const uint32_t t = (lb * kBlock + threadIdx.x) / G;
  int32_t m[3] = {0, 0, 0};
  uint32_t s = 0;
  const bool have = t < g.per_colour;
  if (have) s = colour_space<D>(g, colour, t, m);
  iso_trials<D, G, false>(g, st, B, C, w, iw[threadIdx.x >> 6], zx, zf, have, s, m, colour, st->substep0 + cycle,
                          &blk_acc, [] {});
  __syncthreads();
  if (threadIdx.x == 0 && blk_acc) atomicAdd(&w.acc_slots[b & (kAccSlots - 1)], (unsigned long long)blk_acc);
}

// Every cycle and colour of an apply in one launch, a wavefront per
// region with at most 64 / G trials of a colour (as k_apply_convex).  Against one
// launch per colour: 131,072 LJ bodies 1467 and 1956 us per step, 16,384
// overlap-penalty bodies with 8 lanes 221 and 236.
template <int D, int G>
__global__ void __launch_bounds__(64, 3) k_apply_iso(Geometry g, ApplyState* st, Bodies B, Cells C, Work w, TileCfg tc) {
  const uint32_t b = blockIdx.x;
  const uint32_t tile = (b & 7u) * tc.xcd_chunk + (b >> 3);  // XCD-aware region order
  if (tile >= tc.ntiles) return;  // padding workgroups (grid rounded up to 8) take part in nothing
  if (tc.probe) {
    region_probe(st, w.mbox, tc.ntiles);
    return;
  }
  __shared__ double zx[257], zf[257];
  __shared__ unsigned blk_acc;
  __shared__ IsoWave<D, G> iw;
  if (D == 3) stage_zig(zx, zf);
  if (threadIdx.x == 0) blk_acc = 0;
  const Region rg = wave_region<D>(g, tc, tile);
  const uint32_t cycles = st->cycles, substep0 = st->substep0;
  __syncthreads();
  for (uint32_t i = 0; i < cycles << D; ++i) {
    const uint32_t colour = i & ((1u << D) - 1u);
    if (i) region_publish(w.mbox, tile, tc.tag, i);
    int32_t m[3];
    uint32_t s;
    const bool have = wave_region_space<D>(g, tc, rg, colour, __lane_id() / G, &s, m);
    iso_trials<D, G, true>(g, st, B, C, w, iw, zx, zf, have, s, m, colour, substep0 + (i >> D), &blk_acc, [&] {
      if (i) region_wait<D>(st, w.mbox, tc, rg, tile, i);
    });
  }
  __syncthreads();
  if (threadIdx.x == 0 && blk_acc) atomicAdd(&w.acc_slots[b & (kAccSlots - 1)], (unsigned long long)blk_acc);
}

#define HMC_ISO(D, G) \
  template __global__ void k_apply_iso<D, G>(Geometry g, ApplyState* st, Bodies B, Cells C, Work w, TileCfg tc);
#define HMC_ISO_PASS(D, G)                                                                                           \
  template __global__ void k_pass_iso<D, G>(Geometry g, ApplyState* st, Bodies B, Cells C, Work w, uint32_t colour,  \
                                            uint32_t cycle, uint32_t xcd_chunk);
HMC_ISO(2, 8)
HMC_ISO(2, 16)
HMC_ISO(2, 64)
HMC_ISO(3, 8)
HMC_ISO(3, 16)
HMC_ISO(3, 64)
HMC_ISO_PASS(2, 8)
HMC_ISO_PASS(2, 64)
HMC_ISO_PASS(3, 8)
HMC_ISO_PASS(3, 64)
#undef HMC_ISO
#undef HMC_ISO_PASS

}  // namespace hmc
