// Measurements over the current state: total energy, insertion energies of
// candidate bodies, and the scale distribution function.
#include "sweep_device.hpp"

namespace hmc {

// ------------------------------------------------ lanes sharing one query --
// A site's neighbour query on G lanes: lane gl takes the neighbour spaces gl,
// gl + G, ... of the 3^D (5^D) around the site's space, each space once.  One
// lane per site ran all its candidates in a chain of dependent loads on few
// wavefronts (864 LJ bodies: 4 workgroups, 317 us; on half-waves 22 us).
// The setup every lane of a group repeats costs more than it gives once one lane
// per query fills the device: energy_lanes and insert_lanes on the host.
struct Neighbours {
  uint32_t n[3], first[3];  // spaces visited along each axis, the first of them
};
template <int D>
__device__ __forceinline__ Neighbours neighbours_of(const Geometry& g, uint32_t s) {
  Neighbours q;
#pragma unroll
  for (int a = 0; a < 3; ++a) q.n[a] = 1, q.first[a] = 0;
#pragma unroll
  for (int a = 0; a < D; ++a) {
    const uint32_t sh = (uint32_t)g.shape[a], r = (uint32_t)g.reach[a], m = (s / g.stride[a]) % sh;
    const bool all = 2u * r + 1u >= sh;  // the whole axis
    q.n[a] = all ? sh : 2u * r + 1u;
    q.first[a] = all ? 0u : (m >= r ? m - r : m + sh - r);
  }
  return q;
}
template <int D>
__device__ __forceinline__ uint32_t neighbour_space(const Geometry& g, const Neighbours& q, uint32_t j) {
  uint32_t s = 0;
#pragma unroll
  for (int a = D - 1; a >= 0; --a) {
    const uint32_t d = j % q.n[a], sh = (uint32_t)g.shape[a];
    j /= q.n[a];
    const uint32_t m = q.first[a] + d;
    s += (m >= sh ? m - sh : m) * g.stride[a];
  }
  return s;
}
template <int G>
__device__ __forceinline__ double group_sum(double v) {
#pragma unroll
  for (int d = G / 2; d >= 1; d >>= 1) v += __shfl_xor(v, d, G);
  return v;
}

// ------------------------------------------------------------- total energy --
// PairwiseCutoff::total_energy (pairwise_cutoff.rs:720-745): the sum over
// sites i and neighbours j with site_tag_i < site_tag_j (body index = site
// tag for single-site bodies) of the pair energy, infinite on any hard
// overlap.  Per block of `per` consecutive sites to each group of G lanes: the
// partial sum, the sum of |terms|, the number of non-zero terms and an overlap
// flag, reduced in a fixed order.
template <int D, int G>
__global__ void __launch_bounds__(kEnergyBlock) k_energy(Geometry g, const ApplyState* st, Bodies B, Work w,
                                                         uint32_t per, double* part) {
  __shared__ double vx[3 * kMaxVertices];
  constexpr int kGroups = kEnergyBlock / G;
  __shared__ double red[kGroups][3];
  __shared__ int any_inf;
  if (threadIdx.x == 0) any_inf = 0;
  if (g.model == HMC_CONVEX_POLYHEDRON) stage_verts(g, vx);
  __syncthreads();
  const uint32_t gr = threadIdx.x / G, gl = threadIdx.x % G;
  const uint32_t i0 = (blockIdx.x * kGroups + gr) * per;
  double e = 0.0, a = 0.0, cnt = 0.0;
  bool inf = false;
  for (uint32_t i = i0; i < min(i0 + per, g.n_bodies); ++i) {
    const double4 si = B.spos[i];
    const double t[3] = {si.x, si.y, si.z};
    const double4 bp = B.bpos[i];
    const double x[3] = {bp.x, bp.y, bp.z};
    uint32_t s = space_of<D>(g, st->origin, x);
    if (s == UINT32_MAX) s = 0;  // outside the checkerboard: reported as an error by the host
    const Neighbours nq = neighbours_of<D>(g, s);
    const uint32_t NS = nq.n[0] * nq.n[1] * nq.n[2];
    quat qi = {1.0, {0.0, 0.0, 0.0}};
    if (g.model == HMC_CONVEX_POLYHEDRON) {
      const double4 q4 = B.squat[i];
      qi = {q4.x, {q4.y, q4.z, q4.w}};
    }
    for (uint32_t k = gl; k < NS; k += G) {
      const uint32_t ns = neighbour_space<D>(g, nq, k);
      const uint32_t q1 = w.start[ns + 1];
      for (uint32_t q = w.start[ns]; q < q1 && !inf; ++q) {
        const uint32_t j = w.tmp_body[q];
        if (j <= i) continue;
        const double4 sj = B.spos[j];
        if (g.model == HMC_HARD_SPHERE) {
          inf = overlap64<D>(g, t, sj);
        } else if (g.model == HMC_CONVEX_POLYHEDRON) {
          v3 rj;
          const double d2 = convex_image(g, t, sj, &rj);
          if (d2 < g.cv_rcut2) {
            const double4 q4 = B.squat[j];
            inf = convex_overlap(vx, g.nverts, g.cv_rcut2, d2, v3{t[0], t[1], t[2]}, qi, rj,
                                 quat{q4.x, {q4.y, q4.z, q4.w}});
          }
        } else {
          const double r2 = lj_r2<D>(g, t, sj);
          if (r2 < g.lj_rc2) {
            const double one = lj_energy(g, r2);
            if (one == INFINITY) {  // pairwise_cutoff.rs:720-745 returns at once
              inf = true;
              break;
            }
            e += one;
            a += fabs(one);
            cnt += 1.0;
          }
        }
      }
    }
  }
  if (inf) any_inf = 1;
  e = group_sum<G>(e);
  a = group_sum<G>(a);
  cnt = group_sum<G>(cnt);
  if (gl == 0) {
    red[gr][0] = e;
    red[gr][1] = a;
    red[gr][2] = cnt;
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    double v = 0.0;
    for (int h = 0; h < kGroups; ++h) v += red[h][threadIdx.x];
    part[4 * blockIdx.x + threadIdx.x] = v;
  }
  if (threadIdx.x == 3) part[4 * blockIdx.x + 3] = any_inf ? 1.0 : 0.0;
}

// Sum of the block partials by one workgroup of kEnergyFinal threads: thread t
// adds partials t, t + kEnergyFinal, ... in order, then a fixed tree in LDS
// (a deterministic order; the energy's bound holds for any order of its terms).
__global__ void __launch_bounds__(kEnergyFinal) k_energy_final(const double* part, uint32_t nblocks, double* out) {
  __shared__ double r[4][kEnergyFinal];
  double e = 0.0, a = 0.0, n = 0.0, inf = 0.0;
  for (uint32_t b = threadIdx.x; b < nblocks; b += kEnergyFinal) {
    e += part[4 * b];
    a += part[4 * b + 1];
    n += part[4 * b + 2];
    inf = fmax(inf, part[4 * b + 3]);
  }
  r[0][threadIdx.x] = e;
  r[1][threadIdx.x] = a;
  r[2][threadIdx.x] = n;
  r[3][threadIdx.x] = inf;
  __syncthreads();
  for (int h = kEnergyFinal / 2; h >= 1; h >>= 1) {
    if ((int)threadIdx.x < h) {
      r[0][threadIdx.x] += r[0][threadIdx.x + h];
      r[1][threadIdx.x] += r[1][threadIdx.x + h];
      r[2][threadIdx.x] += r[2][threadIdx.x + h];
      r[3][threadIdx.x] = fmax(r[3][threadIdx.x], r[3][threadIdx.x + h]);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    out[0] = r[0][0];
    out[1] = r[1][0];
    out[2] = r[2][0];
    out[3] = r[3][0];
  }
}

// PairwiseCutoff::delta_energy_insert (pairwise_cutoff.rs:1017-1025 with
// :420-488): the energy of a new body's site wrap(body + 0) with every site of
// the microstate (the new body has no tag yet, so nothing is filtered),
// infinite on a hard overlap or an infinite pair term.  G lanes per
// candidate over the 3^D (or 5^D) neighbour spaces of the current cells;
// out[2 k] is the energy, out[2 k + 1] the bound 2 gamma_n sum |terms| on its
// difference from the reference's summation order.
template <int D, int G>
__global__ void __launch_bounds__(kEnergyBlock) k_insert_energy(Geometry g, const ApplyState* st, Bodies B, Work w,
                                                                const double* __restrict__ cand, uint32_t n,
                                                                double* __restrict__ out, uint32_t* outside) {
  const uint32_t k = blockIdx.x * (kEnergyBlock / G) + threadIdx.x / G, gl = threadIdx.x % G;
  if (k >= n) return;  // (a whole group)
  double t[3] = {0.0, 0.0, 0.0};
  for (int a = 0; a < D; ++a) t[a] = wrap1(g, a, cand[(size_t)k * D + a] + 0.0);
  const uint32_t s = space_of<D>(g, st->origin, t);
  if (s == UINT32_MAX) {  // outside the checkerboard: reported as an error by the host
    if (gl == 0) {
      atomicOr(outside, 1u);
      out[2 * (size_t)k] = 0.0;
      out[2 * (size_t)k + 1] = 0.0;
    }
    return;
  }
  const Neighbours nq = neighbours_of<D>(g, s);
  const uint32_t NS = nq.n[0] * nq.n[1] * nq.n[2];
  double e = 0.0, a = 0.0, cnt = 0.0;
  bool inf = false;
  for (uint32_t j = gl; j < NS; j += G) {
    const uint32_t ns = neighbour_space<D>(g, nq, j);
    const uint32_t q1 = w.start[ns + 1];
    for (uint32_t q = w.start[ns]; q < q1 && !inf; ++q) {
      const double4 sj = B.spos[w.tmp_body[q]];
      if (g.model == HMC_HARD_SPHERE) {
        inf = overlap64<D>(g, t, sj);
      } else {
        const double r2 = lj_r2<D>(g, t, sj);
        if (r2 < g.lj_rc2) {
          const double one = lj_energy(g, r2);
          if (one == INFINITY) {
            inf = true;
            break;
          }
          e += one;
          a += fabs(one);
          cnt += 1.0;
        }
      }
    }
  }
  e = group_sum<G>(e);
  a = group_sum<G>(a);
  cnt = group_sum<G>(cnt);
  inf = group_sum<G>(inf ? 1.0 : 0.0) > 0.0;
  if (gl != 0) return;
  const double nt = fmax(cnt, 1.0);
  const double gam = nt * 0x1p-53 / (1.0 - nt * 0x1p-53);
  out[2 * (size_t)k] = inf ? INFINITY : e;
  out[2 * (size_t)k + 1] = inf ? 0.0 : 2.0 * gam * a;
}

// ------------------------------------------------ scale distribution function --
// The SDF of hard spheres/disks as HOOMD-blue's hpmc compute.SDF defines it
// (no counterpart in the reference): for each body, the smallest compression
// x = 1 - sigma / r over the other bodies (r the minimum-image distance
// between sites) at which the scaled system would first overlap, counted in
// bin floor(x / dx) when 0 <= x < xmax and the bin is below nbins; x < 0 (an
// overlap) is counted apart.  x is monotone in r^2, so the minimum is taken
// over r^2 = (d_x^2 + d_y^2) + d_z^2 and x is formed once.  Bodies within
// r_max = sigma / (1 - xmax) of a body lie in its neighbour spaces: one space
// on each side when the space width is at least r_max (1 + 2^-30), else two
// (the width is at least sigma and xmax < 1/2).  reps/boff describe one or
// several systems laid out as in a batch.
//
// A lane per body, in slot order (neighbouring lanes read the same spaces), blocks
// to XCDs in slabs.  With three or more spaces along every axis the neighbours are
// rows of three spaces, two loads of slots a row (four at the periodic face), and
// rows and row ends farther than r_max from the site are left out: 27 spaces
// become 20.  1,000,188 spheres at packing fraction 0.5: 735 us in body order from 27
// spaces, 611 so, 215 with the counts summed in LDS. (Bound by the dependent loads
// of a candidate, slot to body to site.)
//
// Returns the bin of slot p's body (replica r): nbins for an overlap, UINT32_MAX
// for none.
template <int D>
__device__ __forceinline__ uint32_t sdf_bin(const Geometry& g, const double* origin, uint32_t soff, uint32_t p,
                                            uint32_t b, const Bodies& B, const Work& w, double xmax, double dx,
                                            uint32_t nbins) {
  constexpr int AL = D - 1;
  const uint32_t s = w.elem_space[b] - soff;
  const double4 si = B.spos[b];
  const double t[3] = {si.x, si.y, si.z};
  const double rmax = g.sigma / (1.0 - xmax);
  int32_t m[3] = {0, 0, 0}, reach[3] = {0, 0, 0};
  bool plain = true;
  {
    uint32_t q = s;
#pragma unroll
    for (int a = 0; a < D; ++a) {
      m[a] = (int32_t)(q / g.stride[a]);
      q -= (uint32_t)m[a] * g.stride[a];
      reach[a] = g.width[a] >= rmax * (1.0 + 0x1p-30) ? 1 : 2;
      plain = plain && reach[a] == 1 && g.shape[a] >= 3;
    }
  }
  double best = __builtin_inf();
  auto test = [&](uint32_t q) {
    const double4 sj = B.spos[w.tmp_body[q]];
    const double u[3] = {sj.x, sj.y, sj.z};
    double r2 = 0.0;
#pragma unroll
    for (int a = 0; a < D; ++a) {
      double d = t[a] - u[a];
      d = d > g.half[a] ? d - g.L[a] : d < -g.half[a] ? d + g.L[a] : d;
      r2 = r2 + d * d;
    }
    if (q != p) best = fmin(best, r2);
  };
  if (plain) {
    // squared distances to the faces of the space
    const float cut = g.row_cut2;
    float flo[3], fhi[3];
#pragma unroll
    for (int a = 0; a < D; ++a)
      face_gap2(t[a] - origin[a], (double)m[a], g.width[a], g.L[a], &flo[a], &fhi[a]);
    const int32_t sh = g.shape[AL], ml = m[AL];
    const bool wlo = ml == 0, whi = ml + 1 == sh;  // the lower / upper space lies across the face
    constexpr int NR = D == 3 ? 9 : 3;
    uint32_t lo[NR], hi[NR];
#pragma unroll
    for (int k = 0; k < NR; ++k) {
      const int i0 = D == 3 ? k / 3 : k, i1 = D == 3 ? k % 3 : 0;
      float d = i0 == 0 ? flo[0] : i0 == 2 ? fhi[0] : 0.0f;
      int32_t y0 = m[0] + i0 - 1;
      y0 = y0 < 0 ? y0 + g.shape[0] : y0 == g.shape[0] ? 0 : y0;
      uint32_t sb = soff + (uint32_t)y0 * g.stride[0];
      if constexpr (D == 3) {
        d += i1 == 0 ? flo[1] : i1 == 2 ? fhi[1] : 0.0f;
        int32_t y1 = m[1] + i1 - 1;
        y1 = y1 < 0 ? y1 + g.shape[1] : y1 == g.shape[1] ? 0 : y1;
        sb += (uint32_t)y1 * g.stride[1];
      }
      const bool lower = !(d + flo[AL] >= cut), upper = !(d + fhi[AL] >= cut);
      const uint32_t ca = sb + (uint32_t)ml - (lower && !wlo ? 1u : 0u), cz = sb + (uint32_t)ml + (upper && !whi ? 2u : 1u);
      lo[k] = hi[k] = 0;
      if (!(d >= cut)) {
        lo[k] = w.start[ca];
        hi[k] = w.start[cz];
        if ((wlo && lower) || (whi && upper)) {  // across the face
          const uint32_t c = sb + (wlo ? (uint32_t)(sh - 1) : 0u);
          const uint32_t q1 = w.start[c + 1u];
          for (uint32_t q = w.start[c]; q < q1; ++q) test(q);
        }
      }
    }
#pragma unroll
    for (int k = 0; k < NR; ++k)
      for (uint32_t q = lo[k]; q < hi[k]; ++q) test(q);
  } else {
    uint32_t nb[3][5];
    int nn[3] = {1, 1, 1};
    for (int a = 0; a < D; ++a) {
      const int32_t sh = g.shape[a];
      int k = 0;
      for (int off = -reach[a]; off <= reach[a]; ++off) {
        const int32_t mm = ((m[a] + off) % sh + sh) % sh;
        bool seen = false;
        for (int j = 0; j < k; ++j) seen |= nb[a][j] == (uint32_t)mm * g.stride[a];
        if (!seen) nb[a][k++] = (uint32_t)mm * g.stride[a];
      }
      nn[a] = k;
    }
    for (int i0 = 0; i0 < nn[0]; ++i0)
      for (int i1 = 0; i1 < nn[1]; ++i1)
        for (int i2 = 0; i2 < (D == 3 ? nn[2] : 1); ++i2) {
          const uint32_t ns = soff + nb[0][i0] + nb[1][i1] + (D == 3 ? nb[2][i2] : 0u);
          const uint32_t q1 = w.start[ns + 1];
          for (uint32_t q = w.start[ns]; q < q1; ++q) test(q);
        }
  }
  if (!(best < __builtin_inf())) return UINT32_MAX;  // no other body nearby
  const double x = 1.0 - g.sigma / sqrt(best);
  if (x < 0.0) return nbins;
  const double bin = floor(x / dx);
  return x < xmax && bin < (double)nbins ? (uint32_t)bin : UINT32_MAX;
}

// Blocks of kSdfThreads take runs of `per` slots; the blocks of an XCD take a
// slab.  The counts of the run's first system (most runs lie in one) are summed in
// LDS first (`lds`: nbins + 1 words of it): with an atomic operation per body on a
// few hundred counters the kernel took 611 us.
template <int D>
__global__ void __launch_bounds__(kSdfThreads) k_sdf(const BatchRep* reps, const ApplyState* sts,
                                                     const uint32_t* boff, uint32_t R, uint32_t n_total,
                                                     uint32_t xcd_chunk, uint32_t per, int lds, Bodies B, Work w,
                                                     double xmax, double dx, uint32_t nbins, uint32_t* hist,
                                                     uint32_t* ovl) {
  extern __shared__ uint32_t lh[];
  const uint32_t lb = (blockIdx.x & 7u) * xcd_chunk + (blockIdx.x >> 3);
  const uint64_t begin = (uint64_t)lb * per, end = min(begin + per, (uint64_t)n_total);
  if (begin >= end) return;  // uniform
  if (lds) {
    for (uint32_t i = threadIdx.x; i <= nbins; i += kSdfThreads) lh[i] = 0;
    __syncthreads();
  }
  const uint32_t r0 = R > 1 ? find_replica(boff, R, (uint32_t)begin) : 0u;
  uint32_t r = r0;
  for (uint64_t q = begin + threadIdx.x; q < end; q += kSdfThreads) {
    const uint32_t p = (uint32_t)q, b = w.tmp_body[p];
    while (r + 1u < R && p >= boff[r + 1u]) ++r;
    uint32_t k = UINT32_MAX;
    for (bool done = false; !done;) {  // one system of the wavefront at a time: its constants are scalars
      const uint32_t ru = __builtin_amdgcn_readfirstlane(r);
      if (r != ru) continue;
      k = sdf_bin<D>(reps[ru].g, sts[ru].origin, reps[ru].space_off, p, b, B, w, xmax, dx, nbins);
      done = true;
    }
    if (k == UINT32_MAX) continue;
    if (lds && r == r0)
      atomicAdd(&lh[k], 1u);
    else
      atomicAdd(k < nbins ? &hist[(size_t)r * nbins + k] : &ovl[r], 1u);
  }
  if (!lds) return;
  __syncthreads();
  // (blocks begin at different counters)
  const uint32_t n = nbins + 1u, first = (lb * 37u) % n;
  for (uint32_t i = threadIdx.x; i < n; i += kSdfThreads) {
    const uint32_t k = i + first < n ? i + first : i + first - n;
    if (lh[k]) atomicAdd(k < nbins ? &hist[(size_t)r0 * nbins + k] : &ovl[r0], lh[k]);
  }
}

// explicit instantiations (launched from the host translation units)
template __global__ void k_energy<2, 1>(Geometry g, const ApplyState* st, Bodies B, Work w, uint32_t per, double* part);
template __global__ void k_energy<2, 2>(Geometry g, const ApplyState* st, Bodies B, Work w, uint32_t per, double* part);
template __global__ void k_energy<3, 1>(Geometry g, const ApplyState* st, Bodies B, Work w, uint32_t per, double* part);
template __global__ void k_energy<3, 2>(Geometry g, const ApplyState* st, Bodies B, Work w, uint32_t per, double* part);
template __global__ void k_energy<2, 8>(Geometry g, const ApplyState* st, Bodies B, Work w, uint32_t per, double* part);
template __global__ void k_energy<2, 32>(Geometry g, const ApplyState* st, Bodies B, Work w, uint32_t per, double* part);
template __global__ void k_energy<3, 8>(Geometry g, const ApplyState* st, Bodies B, Work w, uint32_t per, double* part);
template __global__ void k_energy<3, 32>(Geometry g, const ApplyState* st, Bodies B, Work w, uint32_t per, double* part);
template __global__ void k_insert_energy<2, 8>(Geometry g, const ApplyState* st, Bodies B, Work w, const double* __restrict__ cand, uint32_t n, double* __restrict__ out, uint32_t* outside);
template __global__ void k_insert_energy<2, 32>(Geometry g, const ApplyState* st, Bodies B, Work w, const double* __restrict__ cand, uint32_t n, double* __restrict__ out, uint32_t* outside);
template __global__ void k_insert_energy<3, 8>(Geometry g, const ApplyState* st, Bodies B, Work w, const double* __restrict__ cand, uint32_t n, double* __restrict__ out, uint32_t* outside);
template __global__ void k_insert_energy<3, 32>(Geometry g, const ApplyState* st, Bodies B, Work w, const double* __restrict__ cand, uint32_t n, double* __restrict__ out, uint32_t* outside);
template __global__ void k_sdf<2>(const BatchRep* reps, const ApplyState* sts, const uint32_t* boff, uint32_t R, uint32_t n_total, uint32_t xcd_chunk, uint32_t per, int lds, Bodies B, Work w, double xmax, double dx, uint32_t nbins, uint32_t* hist, uint32_t* ovl);
template __global__ void k_sdf<3>(const BatchRep* reps, const ApplyState* sts, const uint32_t* boff, uint32_t R, uint32_t n_total, uint32_t xcd_chunk, uint32_t per, int lds, Bodies B, Work w, double xmax, double dx, uint32_t nbins, uint32_t* hist, uint32_t* ovl);

}  // namespace hmc
