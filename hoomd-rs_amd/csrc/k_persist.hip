// The persistent apply of hard spheres and disks (mixed precision and FP64): one
// launch runs every cycle and colour of an apply.
#include "persist.hpp"

namespace hmc {


// FP64 re-test of a band pair (rare; out of line), the site given by body,
// read with device-scope loads (another region may have written it).
template <int D>
__device__ __noinline__ bool retest64_body(const Geometry* gp, const double4* spos, uint32_t body, double t0,
                                           double t1, double t2) {
  const double t[3] = {t0, t1, t2};
  return overlap64<D>(*gp, t, ld_dev_d4(&spos[body]));
}

// The trial of space s (slots [s0, s0 + n)) from global memory with exact FP64
// pair tests on the sites, for a region whose box holds more bodies than its
// LDS copy (rare).  Same proposal and decision as every other path.
template <int D>
__device__ __noinline__ TrialOut trial_global_dev(const Geometry* gp, ApplyState* st, double4* bpos, double4* spos,
                                                  const uint32_t* cbody, const uint32_t* start,
                                                  hmc_trace_record* trace, unsigned long long trace_cap,
                                                  const double* zx, const double* zf, uint32_t s, uint32_t s0,
                                                  uint32_t n, uint32_t colour, uint32_t substep) {
  const Geometry& g = *gp;
  TrialOut o{0, 0};
  int32_t m[3] = {0, 0, 0};
  for (int a = 0; a < D; ++a) m[a] = (int32_t)((s / g.stride[a]) % (uint32_t)g.shape[a]);
  Sfc64 rng = counter_rng(st->step, substep, st->seed, s);
  const uint32_t pick = choose_index(rng, n);
  double v[3] = {0.0, 0.0, 0.0};
  ball_sample<D>(rng, st->max_move, zx, zf, v);
  const uint32_t slot = s0 + pick;
  const uint32_t body = cbody[slot];
  const double4 bp = bpos[body];
  double x[3] = {bp.x, bp.y, bp.z};
  for (int a = 0; a < D; ++a) x[a] += v[a];
  for (int a = 0; a < D; ++a) x[a] = wrap1(g, a, x[a]);
  bool accept = false;
  if (space_of<D>(g, st->origin, x) == s) {
    double t[3] = {0.0, 0.0, 0.0};
    for (int a = 0; a < D; ++a) t[a] = wrap1(g, a, x[a]);
    bool hit = false;
    for (int i0 = -1; i0 <= 1 && !hit; ++i0)
      for (int i1 = -1; i1 <= 1 && !hit; ++i1)
        for (int i2 = (D == 3 ? -1 : 0); i2 <= (D == 3 ? 1 : 0) && !hit; ++i2) {
          const int di[3] = {i0, i1, i2};
          uint32_t ns = 0;
          for (int a = 0; a < D; ++a) {
            const int32_t sh = g.shape[a];
            int32_t mm = m[a] + di[a];
            mm = mm < 0 ? mm + sh : (mm >= sh ? mm - sh : mm);
            ns += (uint32_t)mm * g.stride[a];
          }
          const uint32_t q0 = start[ns], q1 = start[ns + 1];
          for (uint32_t q = q0; q < q1 && !hit; ++q) {
            if (q == slot) continue;
            hit = overlap64<D>(g, t, ld_dev_d4(&spos[cbody[q]]));
          }
        }
    accept = !hit;
    if (accept) {
      double nsp[3] = {0.0, 0.0, 0.0};
      for (int a = 0; a < D; ++a) nsp[a] = wrap1(g, a, t[a] + 0.0);
      const uint32_t fl = ghost_flags<D>(g, nsp);
      bpos[body] = make_double4(t[0], t[1], t[2], move_stamp(st->epoch));
      st_dev_d4(&spos[body], pack_site(nsp, fl));
    }
  }
  o.accepted = accept ? 1u : 0u;
  if (trace) {
    unsigned long long ti = atomicAdd((unsigned long long*)&st->trace_n, 1ull);
    if (ti < trace_cap) {
      hmc_trace_record rec;
      rec.substep = substep;
      rec.color = colour;
      rec.space = s;
      rec.body = (int64_t)body;
      rec.status = accept ? 1 : 0;
      rec.pad = 0;
      trace[ti] = rec;
    }
  }
  return o;
}

// Squared distance of a staged site from the trial site in the region's scalar
// (fused: three roundings, within the band's relative term).
template <int D, class S>
__device__ __forceinline__ S tile_dist2(const Ent<S>& q, const S* tr) {
  const S dx = q.x - tr[0], dy = q.y - tr[1];
  if (D == 3) {
    const S dz = q.z - tr[2];
    return fma(dx, dx, fma(dy, dy, dz * dz));
  }
  return fma(dx, dx, dy * dy);
}
template <class S>
__device__ __forceinline__ S band_lo(const TileCfg& tc) {
  return std::is_same<S, float>::value ? (S)tc.band_lo : (S)tc.band64_lo;
}
template <class S>
__device__ __forceinline__ S band_hi(const TileCfg& tc) {
  return std::is_same<S, float>::value ? (S)tc.band_hi : (S)tc.band64_hi;
}

// The rows of a trial: the 3^D cells around the trial's own are 3^(D-1) rows
// of three cells, contiguous among the staged sites.  key[r] = the row's
// length << 16 | its first entry, longest first.
//
// A cell whose nearest point is a diameter away holds nothing to test: rows
// and row ends are cut by the distance from the trial site (box-relative, tr)
// to the faces of its cell cb (27 cells become 20 on average).  Spaces are
// exact in FP64 and a body stays in its space for the whole apply, so the
// cut's margin of 10^-4 covers every rounding (coordinates of some tens of
// diameters in FP32).
//
// Sorted by length so that the walk below runs as many slots as the
// wavefront's fullest lanes have sites: on C2 32 for 27 candidates a lane,
// where rounds over all rows in place took 71.
template <int D, class S>
__device__ __forceinline__ void tile_rows(GeoPtr g, const TileCfg& tc, const uint16_t* coff,
                                          const uint32_t* cb, const S* tr, uint32_t* key) {
  constexpr int AL = D - 1, NR = D == 3 ? 9 : 3;
  const float cut = (float)band_hi<S>(tc) * (1.0f + 1e-4f);
  // squared distance from the trial site to the lower and upper face of its cell
  float flo[3] = {0.0f, 0.0f, 0.0f}, fhi[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int a = 0; a < D; ++a) {
    const float wd = (float)g->width[a];
    const float u = (float)tr[a] - ((float)cb[a] - 0.5f * (float)tc.E[a]) * wd;
    const float dl = fmaxf(u, 0.0f), dh = fmaxf(wd - u, 0.0f);
    flo[a] = dl * dl;
    fhi[a] = dh * dh;
  }
  const uint32_t s1 = tc.E[AL] + 1, s0 = D == 3 ? tc.E[1] * s1 : s1;  // cells between neighbouring rows
  const uint32_t c0 = D == 3 ? cb[0] * s0 + cb[1] * s1 + cb[2] : cb[0] * s0 + cb[1];
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const int i0 = D == 3 ? r / 3 : r, i1 = D == 3 ? r % 3 : 1;
    float d = i0 == 0 ? flo[0] : i0 == 2 ? fhi[0] : 0.0f;
    if (D == 3) d += i1 == 0 ? flo[1] : i1 == 2 ? fhi[1] : 0.0f;
    const uint32_t c = c0 + (uint32_t)(i0 - 1) * s0 + (D == 3 ? (uint32_t)(i1 - 1) * s1 : 0u);
    const uint32_t b = coff[c - (d + flo[AL] < cut ? 1u : 0u)];
    const uint32_t e = coff[c + (d + fhi[AL] < cut ? 2u : 1u)];
    key[r] = d < cut ? ((e - b) << 16) | b : 0u;
  }
  auto order = [&](int i, int j) {
    const uint32_t hi = max(key[i], key[j]), lo = min(key[i], key[j]);
    key[i] = hi;
    key[j] = lo;
  };
  if (D == 3) {
    // Floyd's 25-comparator network for nine elements
    order(0, 3), order(1, 7), order(2, 5), order(4, 8);
    order(0, 7), order(2, 4), order(3, 8), order(5, 6);
    order(0, 2), order(1, 3), order(4, 5), order(7, 8);
    order(1, 4), order(3, 6), order(5, 7);
    order(0, 1), order(2, 4), order(3, 5), order(6, 8);
    order(2, 3), order(4, 5), order(6, 7);
    order(1, 2), order(3, 4), order(5, 6);
  } else {
    order(0, 2), order(0, 1), order(1, 2);
  }
}

// Does the trial site (FP64 t, box-relative tr) overlap a staged site of
// its rows other than its own, entry `self` (value old) of lb?
//
// Three rows at a time, one site of each per round, while any lane has a site
// left in the longest of them.  A lane past the end of its row reads on into
// the sites that follow: they are sites of the box too, either in the trial's
// neighbourhood or a space's width or more away (a site's coordinates never
// leave its space by more than rounding, also while another trial moves it),
// and at the end of the box kTilePad entries out of reach.  So no slot
// needs a validity test; the own entry is moved out of reach for the walk.
// (The LDS reads of 12 or 24 bytes at scattered entries bound the walk.)
//
// Pairs inside the band are re-tested in FP64 after the walk when no certain
// overlap was found.  `odd`: the box holds a site without images, whose entry
// is NaN and which is always re-tested; such a box, and a row longer than
// kTilePad, is walked one site at a time.  lb[self] holds `old` again on
// return.
template <int D, class S>
__device__ __forceinline__ bool tile_overlaps(const Geometry& g, const TileCfg& tc, Ent<S>* lb, const double4* spos,
                                              const double* t, const S* tr, uint32_t* key, uint32_t self,
                                              const Ent<S>& old, bool odd, unsigned* retests) {
  constexpr int NR = D == 3 ? 9 : 3;
  const S lo = band_lo<S>(tc), hi = band_hi<S>(tc);
  lb[self].x = (S)kTileFar;
  bool hit = false, walk = __any(odd || (key[0] >> 16) > (uint32_t)kTilePad);
  if (!walk) {  // uniform
    const Ent<S>* p[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) p[r] = lb + (key[r] & 0xffffu);
    S near2 = (S)__builtin_inf();
    auto slots = [&](int r0, uint32_t k) {
      const Ent<S> a = p[r0][k], b = p[r0 + 1][k], c = p[r0 + 2][k];
      near2 = fmin(near2, tile_dist2<D, S>(a, tr));
      near2 = fmin(near2, fmin(tile_dist2<D, S>(b, tr), tile_dist2<D, S>(c, tr)));
    };
    for (uint32_t k = 0; __any(!(near2 < lo) && (key[0] >> 16) > k); ++k) {
      slots(0, k);
      if (D == 3) {
        if (!__any((key[3] >> 16) > k)) continue;
        slots(3, k);
        if (!__any((key[6] >> 16) > k)) continue;
        slots(6, k);
      }
    }
    hit = near2 < lo;
    walk = near2 < hi && !hit;
  }
  if (walk) {
#pragma unroll 1
    for (int r = 0; r < NR && !hit; ++r) {
      const uint32_t b = key[0] & 0xffffu, n = key[0] >> 16;
#pragma unroll
      for (int i = 0; i + 1 < NR; ++i) key[i] = key[i + 1];
#pragma unroll 1
      for (uint32_t k = 0; k < n && !hit; ++k) {
        const Ent<S> q = lb[b + k];
        const S d2 = tile_dist2<D, S>(q, tr);
        if (d2 < lo) hit = true;
        if (d2 < lo || d2 >= hi) continue;
        ++*retests;
        hit = retest64_body<D>(g.self, spos, Staged<S>::body(q), t[0], t[1], t[2]);
      }
    }
  }
  lb[self] = old;
  return hit;
}

// Every cycle and colour of one apply for region `tile` of the system (g, st,
// w.start, w.mbox); the region's accepted moves are added to *acc.  zx, zf:
// the ziggurat layers (an LDS copy, or the constant tables).
//
// A pass is a chain of latencies (two wavefronts per SIMD: one lane per trial
// of a colour fills the chip no further), so what a pass does not need from
// its neighbours is taken off the chain.  After the trials of pass i:
//   publish (stores acknowledged, progress word);
//   the draws of pass i + 1: random numbers, chosen body, displacement;
//   each wavefront polls the progress words it needs (usually there by now)
//   and issues the loads of its halo entries;
//   the rest of the proposal while they are in flight: wrapped positions,
//   space test, the entries an acceptance writes, the rows to walk;
//   the halo entries into LDS, a barrier, the trials.
// None of the proposal reads what pass i or a neighbour changed: a trial's
// body belongs to its own colour's cell, and cells' offsets are static.
template <int D, class S, int CELLS>
__device__ __forceinline__ void apply_tile_run(const Geometry& g, ApplyState* st, const Bodies& B, const Cells& C,
                                               const Work& w, const TileCfg& tc, uint32_t tile,
                                               unsigned long long* acc, const double* zx, const double* zf) {
  constexpr int AL = D - 1;  // the row axis (stride 1)
  constexpr uint32_t NCOL = 1u << D;
  extern __shared__ __align__(16) unsigned char smem[];
  const RegionLds<S> l = region_lds<D, S>(smem, tc);
  const uint32_t CW = tc.E[AL] + 1;
  const uint16_t* coff = l.coff;
  Ent<S>* lb = l.lb;
  __shared__ unsigned blk_acc;
  __shared__ uint32_t hcnt[kHaloLists];
  __shared__ uint32_t odd;  // the box holds (or held) a site without images
  const uint32_t tid = threadIdx.x;
  const uint32_t cycles = st->cycles, substep0 = st->substep0;
  const uint64_t step = st->step;
  const uint32_t seed = st->seed;
  const double max_move = st->max_move;
  const double stamp = move_stamp(st->epoch);
  double origin[3] = {0.0, 0.0, 0.0};
  for (int a = 0; a < D; ++a) origin[a] = st->origin[a];
  const Region rg = region_of<D>(g, tc, origin, tile);
  const int32_t* org = rg.org;
  const int32_t* rl = rg.rl;
  const double* c64 = rg.c64;
  // this thread's trial digits (one space of each colour)
  uint32_t hh[3] = {0, 0, 0};
  {
    uint32_t r = tid;
    for (int a = D - 1; a >= 0; --a) {
      hh[a] = r % tc.T[a];
      r /= tc.T[a];
    }
  }
  const bool has_trial = tid < tc.trials;

  if (tid == 0) blk_acc = odd = 0;
  if (tid < (uint32_t)kHaloLists) hcnt[tid] = 0;
  const uint32_t beyond = region_stage<D, S, kTilePad>(g, tc, rg, B, C, w, l, &odd);
  const bool overflow = beyond != 0;

  unsigned retests = 0;
  // the proposal of this thread's trial
  bool pgo = false, pin = false;
  uint32_t ps = 0, self = 0, body = 0;
  uint32_t pcb[3] = {0, 0, 0}, key[9];
  double v[3] = {0.0, 0.0, 0.0}, pt[3] = {0.0, 0.0, 0.0};
  S ptr[3] = {0, 0, 0};
  double4 bp = make_double4(0.0, 0.0, 0.0, 0.0), psp = bp;
  Ent<S> pent{}, pold{};
  for (int r = 0; r < 9; ++r) key[r] = 0;
  // the draws of pass i (cycle i / 2^D, colour i mod 2^D)
  auto draw = [&](uint32_t i) {
    const uint32_t colour = i & (NCOL - 1), substep = substep0 + (i >> D);
    bool active = has_trial && !overflow;
    uint32_t s = 0;
    for (int a = 0; a < D; ++a) {
      const uint32_t h = 2 * hh[a] + ((colour >> (D - 1 - a)) & 1u);
      if ((int32_t)h >= rl[a]) active = false;
      s += (uint32_t)(org[a] + (int32_t)h) * g.stride[a];
      pcb[a] = h + 1;
    }
    ps = s;
    pgo = false;
    if (!active) return;
    const uint32_t c = (D == 3 ? pcb[0] * tc.E[1] + pcb[1] : pcb[0]) * CW + pcb[AL];
    const uint32_t e0 = coff[c], n = coff[c + 1] - e0;
    if (!n) return;
    pgo = true;
    // the choice first (a few draws), then the chosen body's position in
    // flight during the displacement draw
    Sfc64 rng = counter_rng<true>(step, substep, seed, s);
    self = e0 + choose_index(rng, n);
    pold = lb[self];
    body = Staged<S>::body(pold);
    bp = B.bpos[body];
    ball_sample<D>(rng, max_move, zx, zf, v);
  };
  // the rest of the proposal: everything of the trial that depends on it alone
  auto finish = [&]() {
    if (!pgo) return;
    const GeoPtr gp = geo_ptr(g.self);
    const double x[3] = {bp.x + v[0], bp.y + v[1], bp.z + v[2]};
    uint32_t own[3];
    for (int a = 0; a < D; ++a) own[a] = (uint32_t)org[a] + pcb[a] - 1u;
    const TrialSite<D> ts = trial_site<D>(gp, st, origin, x, own, ps);
    pin = ts.in;
    for (int a = 0; a < D; ++a) pt[a] = ts.t[a];
    psp = pack_site(ts.n, ts.flags);
    box_relative64<D>(*gp, c64, ts.t, ptr);
    S e[3] = {0, 0, 0};
    box_relative64<D>(*gp, c64, ts.n, e);
    e[0] = ts.flags == kNoImages ? (S)__builtin_nanf("") : e[0];
    pent = Staged<S>::make(e, body);
    tile_rows<D, S>(gp, tc, coff, pcb, ptr, key);
  };

  const uint32_t npass = cycles * NCOL;
  for (uint32_t i = 0; i < npass; ++i) {
    // (one copy of the proposal and of the reload for every pass)
    const uint32_t colour = i & (NCOL - 1), substep = substep0 + (i >> D);
    if (i) region_publish(w.mbox, tile, tc.tag, i);
    draw(i);
    if (i) region_wait<D>(st, w.mbox, tc, rg, tile, i);
    // the body's position is here before the halo loads are issued: the
    // compiler cannot count those, and would wait for them all to use it
    asm volatile("" : "+v"(bp.x), "+v"(bp.y), "+v"(bp.z));
    RegionReload<D, S, 1, CELLS, 3> reload(g, tc, rg, B, l, hcnt, i);
    if (i && !overflow) reload.issue();
    finish();
    if (i && !overflow) reload.commit(&odd);
    if (i == 0) region_halo_lists<D, S>(tc, rg, l, hcnt);  // (read after the next barrier)
    if (i) __syncthreads();
    unsigned accepted = 0;
    if (has_trial && overflow) {
      bool active = true;
      uint32_t s = 0;
      for (int a = 0; a < D; ++a) {
        const uint32_t h = 2 * hh[a] + ((colour >> (D - 1 - a)) & 1u);
        if ((int32_t)h >= rl[a]) active = false;
        s += (uint32_t)(org[a] + (int32_t)h) * g.stride[a];
      }
      const uint32_t s0 = active ? w.start[s] : 0u, n = active ? w.start[s + 1] - s0 : 0u;
      if (n) {
        const TrialOut o = trial_global_dev<D>(g.self, st, B.bpos, B.spos, C.body, w.start,
                                               w.tracing ? w.trace : nullptr, w.trace_cap, zx, zf, s, s0, n,
                                               colour, substep);
        accepted = o.accepted;
        retests += o.retests;
      }
    } else if (pgo) {
      // ---- the trial of this pass from LDS
      if (pin && !tile_overlaps<D, S>(g, tc, lb, B.spos, pt, ptr, key, self, pold, odd != 0, &retests)) {
        // update_body_properties (microstate.rs:985-1034), formed with the proposal
        B.bpos[body] = make_double4(pt[0], pt[1], pt[2], stamp);
        st_dev_d4(&B.spos[body], psp);
        lb[self] = pent;
        if (!(pent.x == pent.x)) odd = 1;
        accepted = 1;
      }
      if (w.tracing) {
        unsigned long long ti = atomicAdd((unsigned long long*)&st->trace_n, 1ull);
        if (ti < w.trace_cap) {
          hmc_trace_record rec;
          rec.substep = substep;
          rec.color = colour;
          rec.space = ps;
          rec.body = (int64_t)body;
          rec.status = (int32_t)accepted;
          rec.pad = 0;
          w.trace[ti] = rec;
        }
      }
    }
    const unsigned long long mk = __ballot(accepted != 0);
    if (__lane_id() == 0 && mk) atomicAdd(&blk_acc, (unsigned)__popcll(mk));
  }
  lane_add(&st->band_retests, retests);
  if (tid == 0 && overflow) {
    atomicAdd(&st->tile_overflows, 1ull);
    atomicMax(&st->box_most, beyond);
  }
  __syncthreads();
  if (tid == 0 && blk_acc) atomicAdd(acc, (unsigned long long)blk_acc);
}

template <int D, class S>
__global__ void __launch_bounds__(kTileThreads, 2) k_apply_tile(Geometry g, ApplyState* st, Bodies B, Cells C, Work w,
                                                             TileCfg tc) {
  const uint32_t b = blockIdx.x;
  const uint32_t tile = (b & 7u) * tc.xcd_chunk + (b >> 3);  // XCD-aware region order
  if (tile >= tc.ntiles) return;  // padding workgroups (grid rounded up to 8) take part in nothing
  if (tc.probe) {
    region_probe(st, w.mbox, tc.ntiles);
    return;
  }
  __shared__ double zx[257], zf[257];
  if (D == 3) stage_zig(zx, zf);  // (read after region_stage's barriers)
  apply_tile_run<D, S, 2>(g, st, B, C, w, tc, tile, &w.acc_slots[b & (kAccSlots - 1)], zx, zf);
}

// The persistent applies of every replica of a batch in one launch.  The batch's regions are packed, whole replicas at a time, into
// rounds of at most one region per workgroup (round k: regions rt0[k] ..
// rt0[k] + rn[k] - 1 of the batch; trep: a region's replica, toff: the
// replicas' first regions).  Workgroup b runs its region of round 0 through
// every cycle of its replica, then its region of round 1, and so on, each
// with its replica's geometry, region shape, state, spaces and mailboxes.
// A region waits only on regions of its own replica, which are all in the
// same round and each run by another resident workgroup that has finished
// the earlier rounds' regions, none of which waits on a later round: every
// round completes.  probe: only check that every workgroup of the launch is
// resident (counter: word 2 of the first region's mailbox; nwg workgroups).
template <int D>
__global__ void __launch_bounds__(kTileThreads, 2) k_bapply_tile(const BatchRep* reps, const TileCfg* tcs,
                                                              const uint32_t* toff, const uint32_t* trep,
                                                              ApplyState* sts, const uint32_t* rt0,
                                                              const uint32_t* rn, uint32_t nrounds, uint32_t nwg,
                                                              uint32_t xcd_chunk, uint32_t probe, uint32_t tag,
                                                              Bodies B, Cells C, Work w) {
  __shared__ Geometry sg;
  __shared__ TileCfg stc;
  const uint32_t b = blockIdx.x;
  const uint32_t t = (b & 7u) * xcd_chunk + (b >> 3);
  if (t >= nwg) return;  // uniform over the block
  if (probe) {
    region_probe(sts + trep[0], w.mbox, nwg);
    return;
  }
  for (uint32_t k = 0; k < nrounds; ++k) {
    if (t >= rn[k]) continue;  // uniform over the block
    const uint32_t gt = rt0[k] + t, r = trep[gt];
    const uint32_t* gsrc = (const uint32_t*)&reps[r].g;
    for (uint32_t i = threadIdx.x; i < sizeof(Geometry) / 4; i += blockDim.x) ((uint32_t*)&sg)[i] = gsrc[i];
    const uint32_t* tsrc = (const uint32_t*)&tcs[r];
    for (uint32_t i = threadIdx.x; i < sizeof(TileCfg) / 4; i += blockDim.x)
      ((uint32_t*)&stc)[i] = i == offsetof(TileCfg, tag) / 4 ? tag : tsrc[i];
    __syncthreads();
    Work wr = w;
    wr.start = w.start + reps[r].space_off;
    wr.mbox = w.mbox + (size_t)toff[r] * kMailboxStride;
    wr.tracing = 0;
    // the ziggurat layers from the constant tables: the LDS they would take
    // is worth more as region entries here (more regions per CU)
    apply_tile_run<D, float, 1>(sg, sts + r, B, C, wr, stc, gt - toff[r], &w.acc_slots[r], kZigX, kZigF);
    __syncthreads();  // sg and stc are rewritten for the next round
  }
}

// explicit instantiations (launched from the host translation units)
template __global__ void k_apply_tile<2, float>(Geometry g, ApplyState* st, Bodies B, Cells C, Work w, TileCfg tc);
template __global__ void k_apply_tile<2, double>(Geometry g, ApplyState* st, Bodies B, Cells C, Work w, TileCfg tc);
template __global__ void k_apply_tile<3, float>(Geometry g, ApplyState* st, Bodies B, Cells C, Work w, TileCfg tc);
template __global__ void k_apply_tile<3, double>(Geometry g, ApplyState* st, Bodies B, Cells C, Work w, TileCfg tc);
template __global__ void k_bapply_tile<3>(const BatchRep*, const TileCfg*, const uint32_t*, const uint32_t*,
                                          ApplyState*, const uint32_t*, const uint32_t*, uint32_t, uint32_t, uint32_t,
                                          uint32_t, uint32_t, Bodies, Cells, Work);

}  // namespace hmc
