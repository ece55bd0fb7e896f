// A whole apply of a small system with isotropic pair energies in FP64 (LJ,
// shifted LJ, the overlap penalty) by one workgroup, the system in its LDS.
//
// 864 LJ bodies are 64 spaces: a colour pass is 8 trials, and an apply 112 of
// them. One launch per pass cost 15 us each, of which the trials' arithmetic is
// little; regions with halos (k_apply_lj) need six spaces per axis. Here a
// barrier separates the passes: 1.81 ms per apply became 0.63 (5.6 us a pass, the
// pair distances of its trials on one compute unit's four SIMDs; the proposals
// are 0.5 us of it).
//
// LDS holds every site (its FP64 position, ghost flags and body) and body in
// slot order, the spaces' first slots, and the proposals of a cycle. A trial's
// proposal depends on the counter and on bodies of its own space, which no
// other space's trial changes: all of a cycle's proposals are drawn at its
// start, one lane per space. Then, per colour, `wpt` wavefronts to a trial:
//  - the rows of neighbour spaces along the last axis (one run of slots, or two
//    across the periodic face) are shared out over the lanes;
//  - the squared distances of the final and the initial site, as the reference
//    forms them, are listed where they lie within the cutoff (about one in
//    seven), and the pair energies (a square root and a division each) evaluated
//    from the list with all lanes in use;
//  - energies, magnitudes and counts are summed in FP64; one lane decides as
//    trial_lj does, with the bound on the summation-order difference.
#include "persist.hpp"

namespace hmc {

// A space's proposal, and what its trial needs that is the same for every cycle.
struct SmallProp {
  Sfc64 rng;      // the trial's stream after the proposal
  double t[3];    // trial body position wrap(wrap(x + v)), and the site before wrap(.. + 0)
  double n[3];    // the site an acceptance stores: wrap(t + 0)
  uint32_t slot;  // the chosen body's slot (UINT32_MAX: an empty space)
  uint32_t flags; // the accepted site's ghost flags; bit 31: the trial stays in its space
};
static_assert(sizeof(SmallProp) == SmallLds::kPropBytes, "proposal size counted in the host's LDS budget");

// lj_r2 from a site and its ghost image per axis (the site again where there is
// none): the smaller displacement by selects.  Nearly every site of a small box
// has ghosts, and the shared image's sum x + T is formed once per move.
template <int D>
__device__ __forceinline__ double small_r2(const Geometry& g, const double* q, const double* x, const double* gx) {
  double d2 = 0.0;
#pragma unroll
  for (int a = 0; a < D; ++a) {
    const double d = q[a] - x[a], dg = q[a] - gx[a];
    const double e = fabs(dg) < fabs(d) ? dg : d;
    d2 = d2 + e * e;
  }
  return d2;
}

template <int D>
__global__ void __launch_bounds__(kSmallThreads) k_apply_small(Geometry g, ApplyState* st, Bodies B, Cells C, Work w,
                                                               uint32_t wpt) {
  constexpr int AL = D - 1;
  constexpr uint32_t NCOL = 1u << D;
  extern __shared__ __align__(16) unsigned char smem[];
  const SmallLds o = SmallLds::of(g);
  double4* site = (double4*)(smem + o.site);  // w: ghost flags << 32 | body
  double* bpos = (double*)(smem + o.body);    // 3 per slot
  double* ghost = (double*)(smem + o.ghost);  // 3 per slot
  SmallProp* prop = (SmallProp*)(smem + o.prop);
  uint16_t* start = (uint16_t*)(smem + o.start);
  uint16_t* order = (uint16_t*)(smem + o.order);  // the spaces by colour, in colour_space's order
  ushort4* rows = (ushort4*)(smem + o.rows);      // per space and row: first run's slot and length, second run's slot, length of both
  __shared__ double zx[257], zf[257];
  __shared__ double list[kSmallThreads / 64][kSmallList];  // a wavefront's squared distances within the cutoff
  __shared__ double part[kSmallThreads / 64][5];
  __shared__ uint32_t acc, amb;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wid = tid >> 6;
  const uint32_t cycles = st->cycles, substep0 = st->substep0, seed = st->seed;
  const uint64_t step = st->step;
  const double kT = st->kT, max_move = st->max_move, stamp = move_stamp(st->epoch);
  const double origin[3] = {st->origin[0], st->origin[1], st->origin[2]};
  // rows of neighbour spaces along the last axis: nr of them, nl spaces long
  uint32_t nsp[3] = {1, 1, 1};
#pragma unroll
  for (int a = 0; a < D; ++a) nsp[a] = min(2u * (uint32_t)g.reach[a] + 1u, (uint32_t)g.shape[a]);
  const uint32_t nr = D == 3 ? nsp[0] * nsp[1] : nsp[0];
  auto put = [&](uint32_t p, const double* x, uint32_t fl, uint32_t b) {
    site[p] = make_double4(x[0], x[1], x[2], __longlong_as_double(((long long)fl << 32) | (long long)b));
#pragma unroll
    for (int a = 0; a < D; ++a) {
      const uint32_t f = (fl >> (2 * a)) & 3u;
      ghost[3 * p + a] = f ? x[a] + (f == 1u ? g.L[a] : -g.L[a]) : x[a];
    }
  };
  if (tid == 0) acc = amb = 0;
  if (D == 3) stage_zig(zx, zf);
  for (uint32_t s = tid; s <= g.n_spaces; s += kSmallThreads) start[s] = (uint16_t)w.start[s];
  for (uint32_t p = tid; p < g.n_bodies; p += kSmallThreads) {
    const uint32_t b = C.body[p];
    const double4 sp = B.spos[b], bp = B.bpos[b];
    const double x[3] = {sp.x, sp.y, sp.z};
    put(p, x, (uint32_t)__double_as_longlong(sp.w), b);
    bpos[3 * p] = bp.x;
    bpos[3 * p + 1] = bp.y;
    bpos[3 * p + 2] = bp.z;
  }
  __syncthreads();
  // the spaces of each colour, and the rows of neighbour slots of each space
  for (uint32_t q = tid; q < g.n_spaces; q += kSmallThreads) {
    int32_t m[3] = {0, 0, 0};
    const uint32_t s = colour_space<D>(g, q / g.per_colour, q % g.per_colour, m);
    order[q] = (uint16_t)s;
    uint32_t first[3] = {0, 0, 0};
#pragma unroll
    for (int a = 0; a < D; ++a) {
      const uint32_t sh = (uint32_t)g.shape[a], r = (uint32_t)g.reach[a], x = (uint32_t)m[a];
      first[a] = nsp[a] == sh ? 0u : (x >= r ? x - r : x + sh - r);
    }
    const uint32_t sh = (uint32_t)g.shape[AL], end = first[AL] + nsp[AL];
    for (uint32_t r = 0; r < nr; ++r) {
      uint32_t sb = 0, x[2] = {D == 3 ? r / nsp[1] : r, D == 3 ? r % nsp[1] : 0u};
#pragma unroll
      for (int a = 0; a < AL; ++a) {
        const uint32_t y = first[a] + x[a];
        sb += (y >= (uint32_t)g.shape[a] ? y - (uint32_t)g.shape[a] : y) * g.stride[a];
      }
      const uint32_t ra = start[sb + first[AL]], la = start[sb + min(end, sh)] - ra, rb = start[sb];
      const uint32_t lb = end > sh ? start[sb + end - sh] - rb : 0u;
      rows[s * nr + r] = make_ushort4((uint16_t)ra, (uint16_t)la, (uint16_t)rb, (uint16_t)(la + lb));
    }
  }
  __syncthreads();
  // This wavefront's share of a trial: part wq of wpt.  Of the trial's 64 wpt
  // lanes lpr take each row (rstep rows at a time): lane's first row and entry.
  const uint32_t groups = (kSmallThreads / 64) / wpt, grp = wid / wpt, wq = wid % wpt;
  const uint32_t lanes = 64u * wpt, gl = 64u * wq + lane;
  const uint32_t lpr = max(1u, lanes / nr), rstep = lanes / lpr, row0 = gl / lpr, e0 = gl % lpr;
  double* ls = list[wid];
  for (uint32_t cyc = 0; cyc < cycles; ++cyc) {
    const uint32_t substep = substep0 + cyc;
    // ---- the proposals of the cycle
    for (uint32_t s = tid; s < g.n_spaces; s += kSmallThreads) {
      SmallProp& pr = prop[s];
      const uint32_t s0 = start[s], n = start[s + 1] - s0;
      if (n == 0) {
        pr.slot = UINT32_MAX;
        continue;
      }
      Sfc64 rng = counter_rng<true>(step, substep, seed, s);
      const uint32_t slot = s0 + choose_index(rng, n);
      double v[3] = {0.0, 0.0, 0.0}, x[3] = {0.0, 0.0, 0.0};
      ball_sample<D>(rng, max_move, zx, zf, v);
      uint32_t own[3] = {0, 0, 0};
#pragma unroll
      for (int a = 0; a < D; ++a) {
        x[a] = bpos[3 * slot + a] + v[a];
        own[a] = (s / g.stride[a]) % (uint32_t)g.shape[a];
      }
      const TrialSite<D> ts = trial_site<D>(geo_ptr(g.self), st, origin, x, own, s);
      for (int a = 0; a < 3; ++a) {
        pr.t[a] = ts.t[a];
        pr.n[a] = ts.n[a];
      }
      pr.flags = ts.flags | (ts.in ? 0x80000000u : 0u);
      pr.rng = rng;
      pr.slot = slot;
    }
    __syncthreads();
    // ---- the colours
    for (uint32_t col = 0; col < NCOL; ++col) {
      for (uint32_t t0 = 0; t0 < g.per_colour; t0 += groups) {  // uniform over the workgroup
        const uint32_t k = t0 + grp;
        uint32_t s = 0, slot = UINT32_MAX, flags = 0;
        if (k < g.per_colour) {
          s = order[col * g.per_colour + k];
          slot = prop[s].slot;
          flags = prop[s].flags;
        }
        const bool run = slot != UINT32_MAX && (flags & 0x80000000u);  // uniform over the wavefront
        double ef = 0.0, ei = 0.0, mag = 0.0;
        uint32_t nf = 0, ni = 0;  // (uniform over the wavefront)
        if (run) {
          const double t[3] = {prop[s].t[0], prop[s].t[1], prop[s].t[2]};
          const double4 own = site[slot];
          const double xi[3] = {own.x, own.y, own.z};
          uint32_t nl = 0;  // listed squared distances of this wavefront (final and initial)
          // energies of the listed squared distances: the sign bit marks the
          // initial site's
          auto flush = [&]() {
            wave_lds_order();
            for (uint32_t q = lane; q < nl; q += 64) {
              const double r2 = ls[q], en = lj_energy(g, fabs(r2));
              const bool fin = __double_as_longlong(r2) >= 0;
              ef += fin ? en : 0.0;
              ei += fin ? 0.0 : en;
              mag += fabs(en);
            }
            nl = 0;
            wave_lds_order();
          };
          for (uint32_t rb0 = 0; rb0 < nr; rb0 += rstep) {
            const uint32_t r = rb0 + row0;
            ushort4 q = make_ushort4(0, 0, 0, 0);
            if (r < nr) q = rows[s * nr + r];
            for (uint32_t e = e0; __any(e < q.w); e += lpr) {
              const uint32_t c = e < q.y ? q.x + e : q.z + (e - q.y);
              const bool ok = e < q.w && c != slot;
              const uint32_t cc = ok ? c : slot;
              const double4 sj = site[cc];
              const double x[3] = {sj.x, sj.y, sj.z}, gx[3] = {ghost[3 * cc], ghost[3 * cc + 1], D == 3 ? ghost[3 * cc + 2] : 0.0};
              double r2f = small_r2<D>(g, t, x, gx), r2i = small_r2<D>(g, xi, x, gx);
              // within 2^-30 of the cutoff: the spatial-structure rule (lj_r2)
              const bool edge = ok && ((r2f >= g.lj_rc2_edge && r2f < g.lj_rc2) || (r2i >= g.lj_rc2_edge && r2i < g.lj_rc2));
              if (__any(edge)) {
                const double4 sf = make_double4(sj.x, sj.y, sj.z, __longlong_as_double((long long)((unsigned long long)__double_as_longlong(sj.w) >> 32)));
                r2f = lj_r2<D>(g, t, sf);
                r2i = lj_r2<D>(g, xi, sf);
              }
              const bool inf_ = ok && r2f < g.lj_rc2, ini = ok && r2i < g.lj_rc2;
              const unsigned long long mf = __ballot(inf_), mi = __ballot(ini), below = (1ull << lane) - 1ull;
              const uint32_t cf = (uint32_t)__popcll(mf), ci = (uint32_t)__popcll(mi);
              if (inf_) ls[nl + (uint32_t)__popcll(mf & below)] = r2f;
              if (ini) ls[nl + cf + (uint32_t)__popcll(mi & below)] = -r2i;
              nl += cf + ci;
              nf += cf;
              ni += ci;
              if (nl + 128u > (uint32_t)kSmallList) flush();
            }
          }
          flush();
          ef = wave_sum_dpp(ef);
          ei = wave_sum_dpp(ei);
          mag = wave_sum_dpp(mag);
          if (wq && lane == 0) {
            part[wid][0] = ef;
            part[wid][1] = ei;
            part[wid][2] = mag;
            part[wid][3] = (double)nf;
            part[wid][4] = (double)ni;
          }
        }
        if (wpt > 1) __syncthreads();  // (uniform: every wavefront passes here for every t0)
        // ---- the decision (one lane of the trial's first wavefront)
        if (slot != UINT32_MAX && wq == 0 && lane == 0) {
          bool accept = false;
          const SmallProp& pr = prop[s];
          const uint32_t body = (uint32_t)(unsigned long long)__double_as_longlong(site[slot].w);
          if (run) {
            double cf = (double)nf, ci = (double)ni;
            for (uint32_t q = 1; q < wpt; ++q) {
              ef += part[wid + q][0];
              ei += part[wid + q][1];
              mag += part[wid + q][2];
              cf += part[wid + q][3];
              ci += part[wid + q][4];
            }
            // energy_final - energy_initial (pairwise_cutoff.rs:919-941)
            if (ef == INFINITY) {
              accept = false;
            } else if (ei == INFINITY) {
              accept = true;
            } else {
              const double dH = ef - ei;
              const double nmax = fmax(fmax(cf, ci), 1.0);
              const double gam = nmax * 0x1p-53 * (1.0 + 0x1p-20);  // >= n u / (1 - n u) for these n
              const double delta = (2.0 * gam * mag + 0x1p-52 * fabs(dH)) * (1.0 + 0x1p-20) + 0x1p-1070;
              Sfc64 rng = pr.rng;
              bool open = false;
              accept = lj_metropolis(rng, dH, delta, kT, &open) != 0;
              if (open) atomicAdd(&amb, 1u);
            }
          }
          if (accept) {
            const uint32_t fl = flags & 0x7fffffffu;
            B.bpos[body] = make_double4(pr.t[0], pr.t[1], pr.t[2], stamp);
            B.spos[body] = pack_site(pr.n, fl);
            for (int a = 0; a < 3; ++a) bpos[3 * slot + a] = pr.t[a];
            put(slot, pr.n, fl, body);
            atomicAdd(&acc, 1u);
          }
          if (w.tracing) {
            unsigned long long ti = atomicAdd((unsigned long long*)&st->trace_n, 1ull);
            if (ti < w.trace_cap) {
              hmc_trace_record rec;
              rec.substep = substep;
              rec.color = col;
              rec.space = s;
              rec.body = (int64_t)body;
              rec.status = accept ? 1 : 0;
              rec.pad = 0;
              w.trace[ti] = rec;
            }
          }
        }
        // trials of one colour do not read one another's sites; the partial
        // sums are written again only after the next barrier
        if (wpt > 1 && t0 + groups < g.per_colour) __syncthreads();
      }
      __syncthreads();
    }
  }
  if (tid == 0) {
    if (acc) atomicAdd(&w.acc_slots[0], (unsigned long long)acc);
    if (amb) atomicAdd(&st->ambiguous, (unsigned long long)amb);
  }
}

template __global__ void k_apply_small<2>(Geometry g, ApplyState* st, Bodies B, Cells C, Work w, uint32_t wpt);
template __global__ void k_apply_small<3>(Geometry g, ApplyState* st, Bodies B, Cells C, Work w, uint32_t wpt);

}  // namespace hmc
