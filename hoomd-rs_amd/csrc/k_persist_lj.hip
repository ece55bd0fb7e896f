// The persistent apply for isotropic pair energies (LJ and shifted LJ, mixed
// precision): one launch runs every cycle and colour of an apply,
// as k_apply_tile does for hard shapes.  A region's 4 to 12 trials of a pass share
// out all lanes of the workgroup, whole quads to each; quads' sums are combined in
// LDS and decided together by wavefront 0, four lanes to a trial, which stores
// the accepted moves and publishes the pass.  The last wavefront meanwhile
// draws the next pass's proposals.  Workgroups have 1, 2 or 4 wavefronts, so that
// the wavefronts of the workgroups sharing a CU spread evenly over its four SIMDs.
//
// Bound by the chain of a pass: of 29,000 cycles the pair terms are 8,500 (two
// wavefronts per SIMD, 57 operations per candidate), the decision and its publish
// 5,500, the wait for the neighbours 6,000, the reload of the halo 6,000.
// 524,288 bodies at density 0.8 (490 regions of nine trials, 120 passes): 2232 us
// per apply with half-wavefronts as the trials' lanes, where the ninth trial ran
// after the other eight and took as long; 1734 with all lanes shared out and the
// proposals beside the decision; 1624 with the candidates by planes of rows; 1487
// with the re-takes' sites loaded together; 1460 with the last wavefront's
// proposals off the wait and the reload.
//
// A trial's candidates are the staged sites of its 3^D neighbour cells in
// LDS (box-relative FP32, body index in w).  For each candidate the final
// and initial FP32 displacements give r^2; membership r^2 < r_cut^2 is
// decided in FP32 only outside a band around r_cut^2 that bounds the FP32
// error of r^2 against the reference's FP64 value, and the pair energies are
// FP32 (s2 = sigma^2 rcp(r^2) and its powers, as in lj_energy32).  The decision stands when the FP32 dH, with a
// rigorous bound on its distance to the reference's FP64 dH, decides the
// Metropolis test; otherwise (a candidate in the membership band, a site
// without images, or a bound that straddles the decision) the trial is
// re-taken exactly in FP64 from the FP64 sites with the reference's image
// rules (lj_r2), with the same random draws.  Decisions therefore equal the
// per-colour FP64 path's bit for bit.
//
// Bound of one FP32 pair term against the reference's FP64 term, for the
// per-axis displacement error E (tc.perr: the roundings of the FP64 sites
// to box-relative FP32 on both sides, and the reference's own roundings of
// the displacement and image shift), with u = 2^-24:
//   |r2_32 - r2_ref| <= beta = E (2 sum|d_a| + D E) + (5 u + 2^-50) r2_32
//     (the FP32 difference, squares and sums; the reference's r^2), and for
//     every pair counted (r2_32 < band_hi) beta <= tc.beta_max;
//   |e_32 - e(r2_32)| <= 48 u A   (A = 4 eps (s12 + s6) + |shift|; the FP32
//     powers s12 and s6 are summed separately and combined in FP64),
//   |e(r2_32) - e(r2_ref)| <= |de/dr2| beta <= 4 eps (6 s12 + 3 s6) / r2 x
//     beta_max x 1.02 (de/dr2 varies by less than 2% over the interval when
//     beta <= r2 / 1024, i.e. r2_32 >= tc.r2_open; closer pairs are left
//     open).  W = (6 s12 + 3 s6) / r2 is summed in FP32 and the bound taken
//     as 1.03 (1 + 2^-16) 4 eps beta_max sum W, the extra factors covering
//     W's own roundings and its sum.
// The energy sums over a quad add gamma_(rounds + 2) (A_f + A_i), the quads are
// added in FP64; the reference's FP64 terms and sum differ from exact by less than
// 2^-40 (A_f + A_i).  A trial the FP32 values leave open is re-taken in FP64
// over the candidates whose FP32 r^2 (final or initial) lies below the top
// of the membership band -- every term the reference sums is among them.
#include "persist.hpp"

namespace hmc {

constexpr int kLjRegionThreads = 256;  // upper bound of the workgroup size
constexpr int kLjList = kLjRegionThreads / 4 * 12;  // listed bodies of an FP64 re-take (LjPart's words)
constexpr int kLjMaxTrials = 12;       // trials of a region per pass

// The proposal of a trial of the next pass, kept in LDS across the wait for
// the neighbour regions.  Lane k of the workgroup draws trial k's, and with
// it everything of the trial that depends on the proposal alone: the trial
// position, its space test, the FP32 images of the trial and initial sites,
// and the site and LDS entry an acceptance writes.
struct LjProp {
  Sfc64 rng;     // the trial's stream after the proposal (Metropolis draws)
  double t[3];   // trial body position wrap(wrap(x + v)) (the site before wrap(.. + 0))
  double4 sp;    // the accepted site: wrap(t + 0) with its ghost flags
  float4 ent;    // its LDS entry
  float tr[3];   // FP32 box-relative trial site
  float xr[3];   // FP32 box-relative initial site (the body's LDS entry)
  uint32_t s, self, body, go, in_space, pad;
};

static_assert(sizeof(LjProp) == 160, "proposal size counted in the host's LDS budget");

// A quad's sums over its candidates, as wavefront 0 reads them.
struct LjPart {
  float4 f;  // final: s12, s6, n; open candidates
  float4 i;  // initial: s12, s6, n; the lanes' rounds of summation (the trial's first quad)
  float4 t;  // t12 and t6 of both sites
};

struct Lj32 {
  // over the pairs within r_cut: the sums of s^12 and s^6 (s = sigma / r), of
  // s^12 / r^2 and s^6 / r^2, and their count
  float s12, s6, t12, t6, n;
};

// One candidate q (box-relative FP32 entry) against the FP32 site p: adds
// its powers to acc when within r_cut (r^2 < lo).  *near: the smallest r^2, and
// *edge: its least distance to the middle of the membership band; the trial is
// left open where they show a candidate within the band, or closer than the
// error bound allows.  Selects, not branches: some lane is nearly always
// within r_cut.
// The energy sum is 4 eps (S12 - S6) - n shift, its magnitude sum
// 4 eps (S12 + S6) + n |shift|, and W = 6 T12 + 3 T6.
template <int D>
__device__ __forceinline__ void lj_pair32(const float* p, float4 q, float lo, float mid, float sig2, Lj32& acc,
                                          float& near, float& edge) {
  const float dx = q.x - p[0], dy = q.y - p[1];
  float r2;
  if (D == 3) {
    const float dz = q.z - p[2];
    r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
  } else {
    r2 = fmaf(dx, dx, dy * dy);
  }
  const bool in = r2 < lo;
  near = fminf(near, r2);
  edge = fminf(edge, fabsf(r2 - mid));
  const float rr = in ? __builtin_amdgcn_rcpf(r2) : 0.0f;
  const float s2 = sig2 * rr;
  const float s4 = s2 * s2, s8 = s4 * s4;
  const float s12 = s4 * s8, s6 = s2 * s4;
  acc.s12 += s12;
  acc.s6 += s6;
  acc.t12 = fmaf(s12, rr, acc.t12);
  acc.t6 = fmaf(s6, rr, acc.t6);
  acc.n += in ? 1.0f : 0.0f;
}

// A DPP move of v within quads (quad_perm).
template <int CTRL>
__device__ __forceinline__ float dpp_f32(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
__device__ __forceinline__ float quad_sum(float v) {
  v += dpp_f32<0xb1>(v);  // quad_perm [1, 0, 3, 2]
  return v + dpp_f32<0x4e>(v);  // quad_perm [2, 3, 0, 1]
}
// Lane J's value of a quad, in its four lanes.
template <int J>
__device__ __forceinline__ double quad_lane(double v) {
  constexpr int P = J * 0x55;
  return __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(v), P, 0xf, 0xf, false),
                          __builtin_amdgcn_update_dpp(0, __double2loint(v), P, 0xf, 0xf, false));
}
__device__ __forceinline__ double half_sum(double v) {
#pragma unroll
  for (int d = 16; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
  return v;
}
__device__ __forceinline__ uint32_t half_sum(uint32_t v) {
#pragma unroll
  for (int d = 16; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
  return v;
}
// FP64 sums of one trial over candidate bodies, exactly as the per-colour
// FP64 path forms each term (lj_r2: the reference's image and cell-edge
// rules), from the FP64 sites read with device-scope loads; lj_reduce64 adds
// the half-wave's lanes.
struct Lj64 {
  double ef, af, ei, ai;
  uint32_t nf, ni;
};
template <int D>
__device__ __forceinline__ void lj_term64(const Geometry& g, const double4* spos, const double* t, const double* xi,
                                          uint32_t body, Lj64& s) {
  const double4 sj = ld_dev_d4(&spos[body]);
  const double r2f = lj_r2<D>(g, t, sj);
  if (r2f < g.lj_rc2) {
    const double e = lj_energy(g, r2f);
    s.ef += e;
    s.af += fabs(e);
    s.nf += 1;
  }
  const double r2i = lj_r2<D>(g, xi, sj);
  if (r2i < g.lj_rc2) {
    const double e = lj_energy(g, r2i);
    s.ei += e;
    s.ai += fabs(e);
    s.ni += 1;
  }
}
__device__ __forceinline__ void lj_reduce64(Lj64& s) {
  s.ef = half_sum(s.ef);
  s.af = half_sum(s.af);
  s.ei = half_sum(s.ei);
  s.ai = half_sum(s.ai);
  s.nf = half_sum(s.nf);
  s.ni = half_sum(s.ni);
}

// The FP64 decision of the per-colour path (trial_lj): infinite final energy
// rejects, infinite initial energy accepts, else Metropolis with the
// summation-order bound (*amb when it cannot settle the decision).
__device__ __forceinline__ bool lj_decide64(Sfc64& rng, const Lj64& s, double kT, bool* amb) {
  *amb = false;
  if (s.ef == INFINITY) return false;
  if (s.ei == INFINITY) return true;
  const double dH = s.ef - s.ei;
  const double nmax = (double)max(max(s.nf, s.ni), 1u);
  const double gam = nmax * 0x1p-53 / (1.0 - nmax * 0x1p-53);
  const double delta = (2.0 * gam * (s.af + s.ai) + 0x1p-52 * fabs(dH)) * (1.0 + 0x1p-20) + 0x1p-1070;
  return lj_metropolis(rng, dH, delta, kT, amb) != 0;
}

template <int D>
__global__ void __launch_bounds__(kLjRegionThreads, 2) k_apply_lj(Geometry g, ApplyState* st, Bodies B, Cells C, Work w,
                                                             TileCfg tc) {
  constexpr int AL = D - 1;  // the row axis (stride 1)
  constexpr uint32_t NCOL = 1u << D;
    const uint32_t b = blockIdx.x;
  const uint32_t tile = (b & 7u) * tc.xcd_chunk + (b >> 3);  // XCD-aware region order
  if (tile >= tc.ntiles) return;  // padding workgroups (grid rounded up to 8) take part in nothing
  if (tc.probe) {
    region_probe(st, w.mbox, tc.ntiles);
    return;
  }
  extern __shared__ __align__(16) unsigned char smem[];
  const RegionLds<float> l = region_lds<D, float>(smem, tc);
  const uint32_t CW = tc.E[AL] + 1;
  const uint16_t* coff = l.coff;
  float4* lb = l.lb;
  __shared__ double zx[257], zf[257];
  __shared__ unsigned blk_acc;
  __shared__ uint32_t hcnt[kHaloLists];
  __shared__ LjProp props[2][kLjMaxTrials];  // pass i's in props[i & 1]
  __shared__ LjPart part[kLjRegionThreads / 4];
  uint32_t* list = (uint32_t*)part;  // a re-take's bodies (wavefront 0 has read the sums by then)
  const uint32_t tid = threadIdx.x, wid = tid >> 6, lane = tid & 63u, last = (blockDim.x >> 6) - 1u;
  const uint32_t hw = tid >> 5, hl = tid & 31u, G = blockDim.x >> 5;  // half-waves (regions that overflow)
  const uint32_t cycles = st->cycles, substep0 = st->substep0;
  const uint64_t step = st->step;
  const uint32_t seed = st->seed;
  const double max_move = st->max_move, kT = st->kT;
  const double stamp = move_stamp(st->epoch);
  double origin[3] = {0.0, 0.0, 0.0};
  for (int a = 0; a < D; ++a) origin[a] = st->origin[a];
  const Region rg = region_of<D>(g, tc, origin, tile);
  const float sig2 = (float)(g.lj_sigma * g.lj_sigma), eps4 = (float)g.lj_eps4, shift = (float)g.lj_shift;
  const float blo = tc.band_lo, bhi = tc.band_hi, r2_open = tc.r2_open;
  // |r2 - bmid| <= bhalf holds for every r2 in the band (both roundings covered)
  const float bmid = 0.5f * (blo + bhi), bhalf = 0.5f * (bhi - blo) + 0x1p-21f * bhi;
  const uint32_t ntr = tc.trials;
  // trial tk of a pass: lanes tk lpt .. of the workgroup
  const uint32_t quads = (blockDim.x >> 2) / ntr, lpt = 4u * quads, tk = tid / lpt, tl = tid % lpt;

  if (D == 3) stage_zig(zx, zf);
  if (tid == 0) blk_acc = 0;
  if (tid < (uint32_t)kHaloLists) hcnt[tid] = 0;
  __shared__ uint32_t odd;  // a site without images (its entry is NaN): the FP64 re-take for every trial
  if (tid == 0) odd = 0;
  const bool overflow = region_stage<D, float, 0>(g, tc, rg, B, C, w, l, &odd);

  unsigned retests = 0, ambiguous = 0;
  // The proposals of pass i, drawn while the neighbour regions finish pass
  // i - 1 (they read only static cell data and this region's own bodies),
  // one lane per trial; trial k's waits in props.  Trial k of colour c is
  // the space with digits 2 h + c_a of the region (h the digits of k in T).
  auto trial_space = [&](uint32_t colour, uint32_t k, uint32_t* cb, bool* active) {
    uint32_t s = 0, hh[3] = {0, 0, 0};
    for (int a = D - 1; a >= 0; --a) {
      hh[a] = k % tc.T[a];
      k /= tc.T[a];
    }
    *active = true;
    for (int a = 0; a < D; ++a) {
      const uint32_t lc = 2 * hh[a] + ((colour >> (D - 1 - a)) & 1u);
      if ((int32_t)lc >= rg.rl[a]) *active = false;
      s += (uint32_t)(rg.org[a] + (int32_t)lc) * g.stride[a];
      cb[a] = lc + 1;
    }
    return s;
  };
  auto propose = [&](uint32_t i, uint32_t k) {
    const uint32_t colour = i & (NCOL - 1), substep = substep0 + (i >> D);
    uint32_t cb[3] = {0, 0, 0};
    bool active = false;
    const uint32_t s = trial_space(colour, k, cb, &active);
    LjProp& pr = props[i & 1][k];
    pr.s = s;
    pr.go = 0;
    if (active && !overflow) {
      const uint32_t crow = D == 3 ? cb[0] * tc.E[1] + cb[1] : cb[0];
      const uint32_t e0 = coff[crow * CW + cb[AL]];
      const uint32_t n = coff[crow * CW + cb[AL] + 1] - e0;
      if (n) {
        Sfc64 rng = counter_rng<true>(step, substep, seed, s);
        const uint32_t self = e0 + choose_index(rng, n);
        const float4 se = lb[self];
        const uint32_t body = (uint32_t)__float_as_int(se.w);
        const double4 bp = B.bpos[body];
        double v[3] = {0.0, 0.0, 0.0};
        ball_sample<D>(rng, max_move, zx, zf, v);
        const double x[3] = {bp.x + v[0], bp.y + v[1], bp.z + v[2]};
        const uint32_t own[3] = {(uint32_t)(rg.org[0] + (int32_t)cb[0] - 1), (uint32_t)(rg.org[1] + (int32_t)cb[1] - 1),
                                 D == 3 ? (uint32_t)(rg.org[2] + (int32_t)cb[2] - 1) : 0u};
        const TrialSite<D> ts = trial_site<D>(geo_ptr(g.self), st, origin, x, own, s);
        const double* t = ts.t;
        const double4 sp = pack_site(ts.n, ts.flags);
        float te[3] = {0.0f, 0.0f, 0.0f};
        box_relative64<D>(g, rg.c64, t, te);
        pr.rng = rng;
        for (int a = 0; a < 3; ++a) pr.t[a] = t[a];
        pr.sp = sp;
        pr.ent = stage_entry64<D, float>(g, rg.c64, ts.n, body);
        pr.tr[0] = te[0];
        pr.tr[1] = te[1];
        pr.tr[2] = te[2];
        pr.xr[0] = se.x;
        pr.xr[1] = se.y;
        pr.xr[2] = se.z;
        pr.self = self;
        pr.body = body;
        pr.in_space = ts.in ? 1u : 0u;
        pr.go = 1;
      }
    }
  };

  // A trial's candidates in LDS, for lane gl of the GS that share them: the
  // rows of three cells around its cell a plane of three rows at a time (in 2D the
  // only one), f(entry index, entry) for every third row's runs.  Returns the
  // rounds.  (A candidate's index from two compares; with all nine rows in one
  // run it took 27 operations of the 100 of a round.)
  //
  // Rows and row ends whose nearest point to both sites is the cutoff away hold
  // no candidate: cut by the squared distances to the faces of the cell, with a
  // margin of 10^-4 for the FP32 roundings.
  const float cut = bhi * (1.0f + 1e-4f);
  auto candidates = [&](const LjProp& pr, uint32_t colour, uint32_t k, uint32_t gl, uint32_t GS, auto&& f) -> uint32_t {
    uint32_t pcb[3] = {0, 0, 0};
    bool act = false;
    (void)trial_space(colour, k, pcb, &act);
    float flo[3], fhi[3];
#pragma unroll
    for (int a = 0; a < D; ++a) {
      const float wd = (float)g.width[a], face = ((float)pcb[a] - 0.5f * (float)tc.E[a]) * wd;
      const float ut = pr.tr[a] - face, ux = pr.xr[a] - face;
      const float dl = fmaxf(fminf(ut, ux), 0.0f), dh = fmaxf(wd - fmaxf(ut, ux), 0.0f);
      flo[a] = dl * dl;
      fhi[a] = dh * dh;
    }
    const uint32_t self = pr.self;
    uint32_t rounds = 0;
#pragma unroll 1
    for (int i0 = 0; i0 < (D == 3 ? 3 : 1); ++i0) {
      const float d0 = D == 3 ? (i0 == 0 ? flo[0] : i0 == 2 ? fhi[0] : 0.0f) : 0.0f;
      uint32_t off[3], pre[4];
      pre[0] = 0;
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        const float d = d0 + (r == 0 ? flo[AL - 1] : r == 2 ? fhi[AL - 1] : 0.0f);
        const uint32_t row = D == 3 ? (pcb[0] + i0 - 1u) * tc.E[1] + (pcb[1] + r - 1u) : pcb[0] + r - 1u;
        const uint32_t c0 = row * CW + pcb[AL] - 1u;
        const uint32_t ca = c0 + (d + flo[AL] < cut ? 0u : 1u);
        const uint32_t cz = d < cut ? c0 + (d + fhi[AL] < cut ? 3u : 2u) : ca;
        const uint32_t first = coff[ca];
        off[r] = first - pre[r];
        pre[r + 1] = pre[r] + (coff[cz] - first);
      }
      const uint32_t total = pre[3];
      // (offsets summed from masks: selected, the compiler puts them in memory)
      const uint32_t o0 = off[0], d1 = off[1] - off[0], d2 = off[2] - off[1], p1 = pre[1], p2 = pre[2];
      auto slot_of = [&](uint32_t c) {
        return c + o0 + (d1 & (0u - (uint32_t)(c >= p1))) + (d2 & (0u - (uint32_t)(c >= p2)));
      };
      // two at a time, for their loads' latency (past the end the body's own
      // entry, which is skipped)
      for (uint32_t c = gl; c < total; c += 2 * GS) {
        const uint32_t q0 = slot_of(c), x = slot_of(c + GS), q1 = c + GS < total ? x : self;
        const float4 e0 = lb[q0], e1 = lb[q1];
        f(q0 == self, e0);
        f(q1 == self, e1);
      }
      rounds += (total + GS - 1) / GS;
    }
    return rounds;
  };
  // The exact FP64 re-take by wavefront 0, with the same draws.  The bodies that
  // may be within r_cut are listed first, and their FP64 sites then loaded
  // together: one load from the device's memory after another, as the candidates
  // come, took as long as a pass (30,000 cycles), and one trial in 400 is re-taken,
  // 12 in the device per pass, which all other regions came to wait for.
  auto retake64 = [&](const LjProp& pr, uint32_t colour, uint32_t k, Sfc64& rng, bool* amb) {
    const double4 sp = ld_dev_d4(&B.spos[pr.body]);
    const double xi[3] = {sp.x, sp.y, sp.z}, t[3] = {pr.t[0], pr.t[1], pr.t[2]};
    const float tr[3] = {pr.tr[0], pr.tr[1], pr.tr[2]}, xr[3] = {pr.xr[0], pr.xr[1], pr.xr[2]};
    Lj64 s64{0.0, 0.0, 0.0, 0.0, 0u, 0u};
    uint32_t cnt = 0;  // (lane 0 takes part in every round, so its count is right)
    candidates(pr, colour, k, lane, 64u, [&](bool own, const float4& e) {
      float dfx = e.x - tr[0], dfy = e.y - tr[1], dix = e.x - xr[0], diy = e.y - xr[1];
      float r2f = fmaf(dfx, dfx, dfy * dfy), r2i = fmaf(dix, dix, diy * diy);
      if (D == 3) {
        const float dfz = e.z - tr[2], diz = e.z - xr[2];
        r2f = fmaf(dfz, dfz, r2f);
        r2i = fmaf(diz, diz, r2i);
      }
      // both far beyond r_cut in FP32: no term of the reference's sums
      const bool term = !own && !(r2f >= bhi && r2i >= bhi);
      const unsigned long long m = __ballot(term);
      const uint32_t base = __builtin_amdgcn_readfirstlane(cnt);
      const uint32_t at = base + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
      cnt = base + (uint32_t)__popcll(m);
      if (!term) return;
      const uint32_t body = (uint32_t)__float_as_int(e.w);
      if (at < (uint32_t)kLjList)
        list[at] = body;
      else
        lj_term64<D>(g, B.spos, t, xi, body, s64);
    });
    wave_lds_order();
    const uint32_t n = min((uint32_t)__builtin_amdgcn_readfirstlane(cnt), (uint32_t)kLjList);
    for (uint32_t q = lane; q < n; q += 64u) lj_term64<D>(g, B.spos, t, xi, list[q], s64);
    wave_lds_order();  // (the list is free for the next re-take)
    s64.ef = wave_sum_dpp(s64.ef);
    s64.af = wave_sum_dpp(s64.af);
    s64.ei = wave_sum_dpp(s64.ei);
    s64.ai = wave_sum_dpp(s64.ai);
    s64.nf = wave_sum(s64.nf);
    s64.ni = wave_sum(s64.ni);
    return lj_decide64(rng, s64, kT, amb);
  };
  // update_body_properties (microstate.rs:985-1034) of an accepted trial
  auto accept_move = [&](const LjProp& pr) {
    B.bpos[pr.body] = make_double4(pr.t[0], pr.t[1], pr.t[2], stamp);
    st_dev_d4(&B.spos[pr.body], pr.sp);
    lb[pr.self] = pr.ent;
    if (!(pr.ent.x == pr.ent.x)) odd = 1;
  };
  auto trace_trial = [&](uint32_t colour, uint32_t substep, uint32_t k, uint32_t body, bool accepted) {
    unsigned long long ti = atomicAdd((unsigned long long*)&st->trace_n, 1ull);
    if (ti < w.trace_cap) {
      uint32_t cbt[3] = {0, 0, 0};
      bool act = false;
      hmc_trace_record rec;
      rec.substep = substep;
      rec.color = colour;
      rec.space = trial_space(colour, k, cbt, &act);
      rec.body = (int64_t)body;
      rec.status = accepted ? 1 : 0;
      rec.pad = 0;
      w.trace[ti] = rec;
    }
  };

  const uint32_t npass = cycles * NCOL;
  if (npass && wid == last && lane < ntr) propose(0, lane);
  region_halo_lists<D, float>(tc, rg, l, hcnt);
  __syncthreads();
  unsigned nacc = 0;  // accepted trials (one lane each)
  for (uint32_t i = 0; i < npass; ++i) {
    const uint32_t colour = i & (NCOL - 1), substep = substep0 + (i >> D);
    const LjProp* prop = props[i & 1];
    // a region whose box exceeds its LDS capacity (rare): the trials from the
    // cell lists in global memory, exactly in FP64, a half-wave each
    for (uint32_t k = hw; overflow && k < ntr; k += G) {
      bool accepted = false, traced = false;
      uint32_t tbody = 0;
      bool active = true;
      uint32_t s = 0;
      int32_t m[3] = {0, 0, 0};
      {
        uint32_t cb[3] = {0, 0, 0};
        s = trial_space(colour, k, cb, &active);
        for (int a = 0; a < D; ++a) m[a] = rg.org[a] + (int32_t)cb[a] - 1;
      }
      const uint32_t s0 = active ? w.start[s] : 0u, n = active ? w.start[s + 1] - s0 : 0u;
      if (active && n) {
        Sfc64 rng = counter_rng(step, substep, seed, s);
        const uint32_t pick = choose_index(rng, n);
        const uint32_t slot = s0 + pick, body = C.body[slot];
        double v[3] = {0.0, 0.0, 0.0};
        ball_sample<D>(rng, max_move, zx, zf, v);
        const double4 bp = B.bpos[body];
        double x[3] = {bp.x, bp.y, bp.z};
        for (int a = 0; a < D; ++a) x[a] = wrap1(g, a, x[a] + v[a]);
        traced = true;
        tbody = body;
        if (space_of<D>(g, origin, x) == s) {
          double t[3] = {0.0, 0.0, 0.0};
          for (int a = 0; a < D; ++a) t[a] = wrap1(g, a, x[a]);
          const double4 sp = ld_dev_d4(&B.spos[body]);
          const double xi[3] = {sp.x, sp.y, sp.z};
          // candidates: the slots of the 3^D neighbour spaces in order, their
          // first slots and prefix in this half-wave's share of the LDS site
          // buffer (unused when the region overflows)
          constexpr uint32_t NS = D == 3 ? 27u : 9u;
          uint32_t* seg0 = (uint32_t*)lb + hw * 64u;
          uint32_t* segp = seg0 + 32u;
          if (hl < NS) {
            uint32_t q = hl, ns = 0;
            for (int a = D - 1; a >= 0; --a) {
              const int32_t sh = g.shape[a];
              int32_t mm = m[a] + (int32_t)(q % 3u) - 1;
              q /= 3u;
              mm = mm < 0 ? mm + sh : (mm >= sh ? mm - sh : mm);
              ns += (uint32_t)mm * g.stride[a];
            }
            seg0[hl] = w.start[ns];
            segp[hl + 1] = w.start[ns + 1] - w.start[ns];
          }
          if (hl == 0) segp[0] = 0;
          wave_lds_order();
          if (hl == 0)
            for (uint32_t k = 1; k <= NS; ++k) segp[k] += segp[k - 1];
          wave_lds_order();
          const uint32_t total = segp[NS];
          Lj64 s64{0.0, 0.0, 0.0, 0.0, 0u, 0u};
          for (uint32_t c = hl; c < total; c += 32u) {
            uint32_t lo = 0, hi = NS;  // the last k with segp[k] <= c
            while (hi - lo > 1) {
              const uint32_t mid = (lo + hi) >> 1;
              if (segp[mid] <= c)
                lo = mid;
              else
                hi = mid;
            }
            const uint32_t q = seg0[lo] + (c - segp[lo]);
            if (q != slot) lj_term64<D>(g, B.spos, t, xi, C.body[q], s64);
          }
          lj_reduce64(s64);
          bool amb = false;
          accepted = lj_decide64(rng, s64, kT, &amb);
          ambiguous += (amb && hl == 0) ? 1u : 0u;
          if (accepted && hl == 0) {
            double nsp[3] = {0.0, 0.0, 0.0};
            for (int a = 0; a < D; ++a) nsp[a] = wrap1(g, a, t[a] + 0.0);
            B.bpos[body] = make_double4(t[0], t[1], t[2], stamp);
            st_dev_d4(&B.spos[body], pack_site(nsp, ghost_flags<D>(g, nsp)));
          }
        }
      }
      if (traced && hl == 0 && w.tracing) trace_trial(colour, substep, k, tbody, accepted);
      nacc += (accepted && hl == 0) ? 1u : 0u;
    }
    if (!overflow) {
      // ---- the trials of this pass from LDS
      Lj32 af{0.0f, 0.0f, 0.0f, 0.0f, 0.0f}, ai{0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
      bool open = false;
      float rounds = 0.0f;
      if (tk < ntr && prop[tk].go && prop[tk].in_space) {
        const LjProp& pr = prop[tk];
        const float tr[3] = {pr.tr[0], pr.tr[1], pr.tr[2]}, xr[3] = {pr.xr[0], pr.xr[1], pr.xr[2]};
        float near = INFINITY, edge = INFINITY;
        const uint32_t n = candidates(pr, colour, tk, tl, lpt, [&](bool own, float4 e) {
          e.x = own ? 0x1p60f : e.x;  // (out of range)
          lj_pair32<D>(tr, e, blo, bmid, sig2, af, near, edge);
          lj_pair32<D>(xr, e, blo, bmid, sig2, ai, near, edge);
        });
        open = near < r2_open || !(edge > bhalf) || odd;
        if (tl == 0) rounds = (float)n;
      }
      const LjPart p = {make_float4(quad_sum(af.s12), quad_sum(af.s6), quad_sum(af.n), quad_sum(open ? 1.0f : 0.0f)),
                        make_float4(quad_sum(ai.s12), quad_sum(ai.s6), quad_sum(ai.n), rounds),
                        make_float4(quad_sum(af.t12), quad_sum(ai.t12), quad_sum(af.t6), quad_sum(ai.t6))};
      if ((tid & 3u) == 0) part[tid >> 2] = p;
      __syncthreads();
      if (wid == 0) {
        // lane j of quad k: trial k's final (0) or initial (1) sums, or both
        // sites' t12 and t6 (2)
        const uint32_t k = lane >> 2, j = lane & 3u;
        const bool live = k < ntr && prop[k < ntr ? k : 0].go, run = live && prop[k].in_space;
        bool accepted = false, decided = true;
        if (run) {
          const LjProp& pr = prop[k];
          const float4* src = (const float4*)&part[k * quads] + min(j, 2u);
          double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
          for (uint32_t q = 0; q < quads; q += 4) {  // four loads in flight
            float4 v[4];
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) v[u] = src[3 * min(q + u, quads - 1u)];
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) {
              const bool in = q + u < quads;
              a0 += in ? (double)v[u].x : 0.0;
              a1 += in ? (double)v[u].y : 0.0;
              a2 += in ? (double)v[u].z : 0.0;
              a3 += in ? (double)v[u].w : 0.0;
            }
          }
          const double e4 = (double)eps4, sh = (double)shift;
          // energy and magnitude (lanes 0 and 1), W (lane 2)
          const double e = e4 * (a0 - a1) - a2 * sh, mag = e4 * (a0 + a1) + a2 * fabs(sh);
          const double wsum = 6.0 * (a0 + a1) + 3.0 * (a2 + a3);
          const double dH32 = quad_lane<0>(e) - quad_lane<1>(e), sa = quad_lane<0>(mag) + quad_lane<1>(mag);
          const double sb = 1.03 * (1.0 + 0x1p-16) * e4 * (double)tc.beta_max * quad_lane<2>(wsum);
          const double rounds = quad_lane<1>(a3);
          const double delta = (((48.0 + rounds + 8.0) * 0x1p-24 + 0x1p-40) * sa + sb) * (1.0 + 0x1p-10) + 0x1p-1070;
          decided = false;
          if (quad_lane<0>(a3) == 0.0 && isfinite(dH32) && isfinite(delta)) {
            Sfc64 rng = pr.rng;
            bool amb32 = false;
            accepted = lj_metropolis(rng, dH32, delta, kT, &amb32) != 0;
            decided = !amb32;
            accepted = accepted && decided;
          }
        }
        // trials left open, one at a time
        unsigned long long todo = __ballot(j == 0 && !decided);
        while (todo) {
          const uint32_t kr = (uint32_t)__builtin_ctzll(todo) >> 2;
          todo &= todo - 1ull;
          Sfc64 rng = prop[kr].rng;  // the FP64 decision draws the same u
          bool amb = false;
          const bool acc = retake64(prop[kr], colour, kr, rng, &amb);
          if (k == kr) accepted = acc;
          retests += lane == 0 ? 1u : 0u;
          ambiguous += (amb && lane == 0) ? 1u : 0u;
        }
        if (j == 0 && live) {
          if (accepted) accept_move(prop[k]);
          if (w.tracing) trace_trial(colour, substep, k, prop[k].body, accepted);
          nacc += accepted ? 1u : 0u;
        }
        if (i + 1 < npass) {
          __builtin_amdgcn_s_waitcnt(0);  // the moves' stores have completed
          wave_publish(w.mbox, tile, tc.tag, i + 1);
        }
      }
    } else if (i + 1 < npass) {
      region_publish(w.mbox, tile, tc.tag, i + 1);
    }
    if (i + 1 == npass) break;  // no later pass reads the halo
    // The last wavefront draws the next proposals, the others reload (a single
    // one does both).
    if (wid == last && lane < ntr) propose(i + 1, lane);
    const uint32_t loaders = last ? 64u * last : 64u;
    if (tid < loaders) region_wait<D>(st, w.mbox, tc, rg, tile, i + 1);
    // (cells of about 15 entries: 16 lanes each)
    if (!overflow) {
      RegionReload<D, float, 16, 2, 2> reload(g, tc, rg, B, l, hcnt, i + 1, loaders);
      reload.issue();
      __syncthreads();  // (a re-take reads the halo of this pass)
      reload.commit(&odd);
    }
    __syncthreads();
  }
  lane_add(&st->band_retests, retests);
  lane_add(&st->ambiguous, ambiguous);
  if (tid == 0 && overflow) atomicAdd(&st->tile_overflows, 1ull);
  if (nacc) atomicAdd(&blk_acc, nacc);
  __syncthreads();
  if (tid == 0 && blk_acc) atomicAdd(&w.acc_slots[b & (kAccSlots - 1)], (unsigned long long)blk_acc);
}

template __global__ void k_apply_lj<2>(Geometry g, ApplyState* st, Bodies B, Cells C, Work w, TileCfg tc);
template __global__ void k_apply_lj<3>(Geometry g, ApplyState* st, Bodies B, Cells C, Work w, TileCfg tc);

}  // namespace hmc
