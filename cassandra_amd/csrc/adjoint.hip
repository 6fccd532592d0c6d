// adjoint.hip -- derivatives of a box's nonbonded energy with respect to the
// per-type LJ parameters, the per-site-kind charges and the coordinates, for
// the box's own coordinates (cass_adjoint) or for a batch of coordinate
// frames of the box kept in device memory (cass_adjoint_set_frames,
// cass_adjoint_frames).
//
// No counterpart exists in the reference; the energy being differentiated is
// exactly the one Compute_System_Total_Energy assembles
// (energy_routines.f90:2648-2953): intermolecular LJ + real-space q-q (with
// the A&S erfc of :2143-2163, differentiated as written), the intramolecular
// scaled terms and the periodic image part of intramolecular pairs, the
// reciprocal sum, the self energy and the LJ tail correction.  Lorentz-
// Berthelot mixing (create_nonbond_table.f90:370-392) carries the pair
// derivatives to the per-type parameters.
//
// Kernels (FP64 throughout), per launch over F frames:
//   k_adj_pairs<NI>  one wavefront per (molecule i, frame).  The molecules j
//                    inside the molecule cutoff are compacted into an LDS
//                    queue and scored 64 at a time, one j per lane, every
//                    site pair of (i, j); then i's intramolecular pairs, one
//                    per lane.  Writes per site of i (dE/d eps of its type,
//                    dE/d sigma, dE/d q, force) and the energy of i's pairs
//                    (intermolecular halved: each pair is visited from both
//                    sides).
//   k_adj_prep       per (site, frame): coordinates and charge, fractional
//                    coordinates and the charge of live sites.
//   k_adj_sk         structure factors: one lane per (n_x, |n_z|) column and
//                    four n_y, summing over a share of a frame's sites the
//                    eight products of the cosines and sines per axis, from
//                    which k_adj_weights forms the four k vectors (+-n_y,
//                    +-n_z), the frame's reciprocal energy and the weights
//                    of k_adj_recip.
//   k_adj_recip      one lane per (site, frame): dE/dq of the site and its
//                    reciprocal force, from the weights along the columns.
//   k_adj_frame      one workgroup per frame: the per-type and per-kind sums,
//                    the energy and the forces, in a fixed order.
// Frame-independent terms (self energy, tail correction) are added on the
// host.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "engine.h"
#include "kernels.h"

using namespace cass;

namespace {

constexpr int kAdjTypes = 8;     // atom types
constexpr int kAdjKinds = 16;    // species-atom kinds (charges)
constexpr int kAdjSites = 8;     // sites per molecule
constexpr int kAdjOut = 1 + 2 * kAdjTypes + kAdjKinds;  // per frame: E, dE/d eps_t, dE/d sig_t, dE/d q_k
constexpr int kNyC = 4;          // n_y values per step of the reciprocal kernels
constexpr int kSkWaves = 8;      // waves per workgroup of k_adj_sk
constexpr int kSkSites = 64;     // sites per tile of k_adj_sk, fewer where the tables of powers are long

// d/dx of the A&S erfc as computed (t = 1/(1+p x), erfc = t*poly(t)*exp(-x^2)).
__host__ __device__ inline void erfc_as_d(double x, double &f, double &df) {
  const double A1 = 0.254829592, A2 = -0.284496736, A3 = 1.421413741, A4 = -1.453152027, A5 = 1.061405429,
               P = 0.3275911;
  const double t = 1.0 / (1.0 + P * x);
  const double poly = A1 + t * (A2 + t * (A3 + t * (A4 + t * A5)));
  const double dpoly = A2 + t * (2.0 * A3 + t * (3.0 * A4 + t * 4.0 * A5));
  const double e = exp(-x * x);
  const double tp = t * poly;
  f = tp * e;
  const double dtp_dt = poly + t * dpoly;
  const double dt_dx = -P * t * t;
  df = dtp_dt * dt_dx * e + tp * (-2.0 * x) * e;
}

struct AdjParams {
  int ntypes, q_style, vdw_sum;
  double rc2_vdw, inv_rc2_vdw, rc2_coul, rc_coul, alpha, alpha_dsf, dsf1, dsf2;
};

// LJ pair: energy, dU/d eps_ij, dU/d sig_ij, dU/dr / r.
__host__ __device__ inline void lj_pair(const AdjParams &a, double r2, double eps, double sig, double &u,
                                        double &de, double &ds, double &dr_over_r) {
  const double s2 = sig * sig / r2, s6 = s2 * s2 * s2, s12 = s6 * s6;
  u = 4.0 * eps * (s12 - s6);
  de = 4.0 * (s12 - s6);
  ds = sig > 0.0 ? 4.0 * eps * (12.0 * s12 - 6.0 * s6) / sig : 0.0;
  dr_over_r = 4.0 * eps * (-12.0 * s12 + 6.0 * s6) / r2;
  if (a.vdw_sum == CASS_SUM_CUT_SHIFT) {
    const double c2 = sig * sig / a.rc2_vdw, c6 = c2 * c2 * c2, c12 = c6 * c6;
    u -= 4.0 * eps * (c12 - c6);
    de -= 4.0 * (c12 - c6);
    if (sig > 0.0) ds -= 4.0 * eps * (12.0 * c12 - 6.0 * c6) / sig;
  }
}

// q-q pair with charges factored out: E = qi qj g(r); returns g and dg/dr / r.
// intra: the scaled minimum-image part plus the periodic part (Ewald), or
// the DSF pair less (1 - qscale) of the bare Coulomb term.
__host__ __device__ inline void qq_pair(const AdjParams &a, double r2, bool intra, double qscale, double &g,
                                        double &dg_over_r) {
  const double r = sqrt(r2);
  if (a.q_style == CASS_Q_EWALD) {
    double f, df;
    erfc_as_d(a.alpha * r, f, df);
    const double base = intra ? (qscale - 1.0 + f) : f;
    g = kChargeFactor * base / r;
    const double dbase = df * a.alpha;
    dg_over_r = kChargeFactor * (dbase / r - base / r2) / r;
  } else if (a.q_style == CASS_Q_DSF) {
    const double ec = erfc(a.alpha_dsf * r);
    const double sub = intra ? (1.0 - qscale) : 0.0;
    const double v = a.dsf2 * (r - a.rc_coul) - a.dsf1 + ec / r - sub / r;
    g = kChargeFactor * v;
    const double dv = a.dsf2 - 2.0 * a.alpha_dsf / 1.7724538509055159 * exp(-a.alpha_dsf * a.alpha_dsf * r2) / r -
                      ec / r2 + sub / r2;
    dg_over_r = kChargeFactor * dv / r;
  } else if (a.q_style == CASS_Q_CUT || a.q_style == CASS_Q_MINIMUM) {
    const double s = intra ? qscale : 1.0;
    g = kChargeFactor * s / r;
    dg_over_r = -kChargeFactor * s / (r2 * r);
  } else {
    g = 0.0;
    dg_over_r = 0.0;
  }
}

// Frames on the device: frame f's site coordinates at x + f*stride, y + ...,
// z + ..., its molecules' (COM, max_dcom) at (double*)com + f*stride.
struct AdjFrameView {
  const double *x, *y, *z;
  const double4 *com;
  int64_t stride;
};

// 1/x for the pair distances and the erfc argument (x in [1e-3, 1e4]): the
// hardware reciprocal seed refined by two Newton steps, within an ulp or two
// of the quotient.
__device__ inline double rcp_nr(double x) {
  double y = __builtin_amdgcn_rcp(x);
  y = fma(y, fma(-x, y, 1.0), y);
  return fma(y, fma(-x, y, 1.0), y);
}

__device__ inline double wave_sum_x(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// The minimum image of a site pair's displacement.
__device__ __forceinline__ void adj_image(const BoxDev &b, double &rx, double &ry, double &rz) {
  if (b.cubic) {
    // one image shift per axis without branches: equal to the cubic
    // if/else form for |d| < 1.5 L (sites of whole molecules in the box)
    rx = fma(-rint(rx * b.Li[0]), b.L[0], rx);
    ry = fma(-rint(ry * b.Li[4]), b.L[1], ry);
    rz = fma(-rint(rz * b.Li[8]), b.L[2], rz);
  } else {
    min_image(b, rx, ry, rz);
  }
}

// a * b + c with a constant c in scalar registers: left to itself the compiler
// copies it to vector registers for the two-address form, two moves for each
// multiply-add (45 of the 245 instructions of a pair).
__device__ __forceinline__ double fma_c(double a, double b, double c) {
  double d;
  asm("v_fma_f64 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "s"(c));
  return d;
}

// exp(x) for x <= 0 (exp(-(alpha r)^2) of a pair within its cutoff): x = n ln
// 2 + r with |r| <= ln 2 / 2, the Taylor series of exp(r) to r^13 (remainder
// below 5e-18), and the exponent.  Within one ulp of exp over [-700, 0].
__device__ __forceinline__ double exp_neg(double x) {
  const double n = rint(x * 1.4426950408889634074);
  double r = fma(n, -0.6931471803691238, x);  // ln 2: 32 leading bits, then the rest
  r = fma(n, -1.9082149292705877e-10, r);
  double p = fma_c(r, 1.0 / 6227020800.0, 1.0 / 479001600.0);
  p = fma_c(p, r, 1.0 / 39916800.0);
  p = fma_c(p, r, 1.0 / 3628800.0);
  p = fma_c(p, r, 1.0 / 362880.0);
  p = fma_c(p, r, 1.0 / 40320.0);
  p = fma_c(p, r, 1.0 / 5040.0);
  p = fma_c(p, r, 1.0 / 720.0);
  p = fma_c(p, r, 1.0 / 120.0);
  p = fma_c(p, r, 1.0 / 24.0);
  p = fma_c(p, r, 1.0 / 6.0);
  p = fma(p, r, 0.5);
  p = fma(p, r, 1.0);
  p = fma(p, r, 1.0);
  return ldexp(p, (int)n);
}

// One site of molecule i against a site of another molecule at displacement
// (rx, ry, rz), of type tj and charge qj: adds the pair energies (halved: each
// intermolecular pair is visited from both sides) and i's side of every
// derivative to acc = (E, dE/d eps of the site's type, dE/d sigma, dE/d q,
// force x, y, z).  ptab[ti * ntypes + tj] = (eps_ij, sigma_ij^2, 1/sigma_ij,
// 0); heps = 1 / (2 eps of the site's type), 0 for eps = 0.
template <bool EW>
__device__ __forceinline__ void adj_pair(const AdjParams &a, const double4 *ptab, double rx, double ry, double rz,
                                         int tj, double qj, int ti, double qi, double heps, double (&acc)[7]) {
  const double r2 = rx * rx + ry * ry + rz * rz;
  const double inv_r2 = rcp_nr(r2);
  double fr = 0.0;  // -dE/dr / r on site ia
  if (r2 <= a.rc2_vdw && ti >= 0 && tj >= 0) {
    const double4 pt = ptab[ti * a.ntypes + tj];
    const double s2 = pt.y * inv_r2, s6 = s2 * s2 * s2, s12 = s6 * s6;
    double lj = s12 - s6, dl = 12.0 * s12 - 6.0 * s6;
    const double e4 = 4.0 * pt.x;
    fr = e4 * dl * inv_r2;
    if (a.vdw_sum == CASS_SUM_CUT_SHIFT) {
      const double c2 = pt.y * a.inv_rc2_vdw, c6 = c2 * c2 * c2, c12 = c6 * c6;
      lj -= c12 - c6;
      dl -= 12.0 * c12 - 6.0 * c6;
    }
    acc[0] += 0.5 * e4 * lj;
    acc[1] += 4.0 * lj * pt.x * heps;
    acc[2] += 0.5 * e4 * dl * pt.z;
  }
  if (r2 <= a.rc2_coul && (EW || a.q_style != CASS_Q_NONE)) {
    double g, dg;  // E = qi qj g, dg = (dg/dr) / r
    if (EW) {
      const double A1 = 0.254829592, A2 = -0.284496736, A3 = 1.421413741, A4 = -1.453152027,
                   A5 = 1.061405429, P = 0.3275911;
      const double r = sqrt(r2), inv_r = r * inv_r2;
      const double x = a.alpha * r;
      const double tt = rcp_nr(1.0 + P * x);
      const double poly = fma_c(tt, fma_c(tt, fma_c(tt, fma_c(tt, A5, A4), A3), A2), A1);
      const double dpoly = fma_c(tt, fma_c(tt, fma_c(tt, 4.0 * A5, 3.0 * A4), 2.0 * A3), A2);
      const double ex = exp_neg(-x * x);
      const double f = tt * poly * ex;
      const double df = ((poly + tt * dpoly) * (-P * tt * tt) - 2.0 * x * tt * poly) * ex;
      g = kChargeFactor * f * inv_r;
      dg = kChargeFactor * (df * a.alpha * inv_r - f * inv_r2) * inv_r;
    } else {
      qq_pair(a, r2, false, 1.0, g, dg);
    }
    acc[0] += 0.5 * qi * qj * g;
    acc[3] += qj * g;
    fr -= qi * qj * dg;
  }
  acc[4] += fr * rx;
  acc[5] += fr * ry;
  acc[6] += fr * rz;
}

constexpr int kAdjRing = 128;   // site pairs waiting per site of i
constexpr int kAdjList = 512;  // molecule indices held in LDS per pass

// One wavefront (64 lanes) per (molecule i, frame).  The molecules j inside
// the molecule cutoff of i are listed in LDS by ballot compaction (up to
// kAdjList per pass).  Their sites are then walked for the squared distances
// to NI sites of i at a time, and the pairs within the cutoff compacted again,
// one ring per site of i, so that the pair terms run on full waves: of the
// listed molecules' pairs four in ten lie outside the cutoff, and with three
// sites a molecule a walk of one j per lane left a fifth of the lanes idle.
// The vector unit's issue rate bounds the kernel (busy three cycles in four):
// 200 frames of 800 three-site molecules took 2.23 ms with one j per lane and
// shuffle trees per sum, and take 1.61.  The wave sums are added to LDS slots
// per site.  Then i's intramolecular pairs, one per lane.  Writes site_out[f][site][6] = (dE/d eps of the site's type,
// dE/d sigma, dE/d q, force) and emol[f][i], the energy of i's pairs.  vs/qs:
// per species the intramolecular scale tables (pair_off + ia*n + ja); nj_max:
// the largest molecule.
template <bool EW, int NI>
__global__ void __launch_bounds__(64) k_adj_pairs(BoxDev b, TopoDev tp, AdjParams a, AdjFrameView fv,
                                                  const double4 *__restrict__ xq, const int *__restrict__ stype,
                                                  const double4 *__restrict__ ptab_g,
                                                  const double *__restrict__ vscale,
                                                  const double *__restrict__ qscale,
                                                  const int *__restrict__ pair_off, const int *__restrict__ mcode, int nsites,
                                                  int nj_max,
                                                  double *__restrict__ site_out, double *__restrict__ emol) {
  __shared__ int list[kAdjList];
  __shared__ int ring[NI][kAdjRing];
  __shared__ double sacc[kAdjSites][7];
  __shared__ double trans[7 * 65];  // lanes' parts of one site's sums, then the intramolecular pairs' terms
  double (*pval)[9] = (double (*)[9])trans;
  static_assert(kAdjSites * (kAdjSites - 1) / 2 * 9 <= 7 * 65, "pair terms");
  __shared__ double4 ptab[kAdjTypes * kAdjTypes];
  const int i = blockIdx.x, f = blockIdx.y, lane = threadIdx.x;
  const double *X = fv.x + f * fv.stride, *Y = fv.y + f * fv.stride, *Z = fv.z + f * fv.stride;
  const double4 *COM = (const double4 *)((const double *)fv.com + f * fv.stride);
  double *so = site_out + (int64_t)f * nsites * 6;
  const int si = b.species[i], fi = b.first[i];
  const int ni = tp.sp_natoms[si], oi = tp.sp_atom_off[si];
  if (!b.live[i]) {
    for (int t = lane; t < ni * 6; t += 64) so[(int64_t)fi * 6 + t] = 0.0;
    if (lane == 0) emol[(int64_t)f * b.nmols + i] = 0.0;
    return;
  }
  if (lane < kAdjSites * 7) sacc[lane / 7][lane % 7] = 0.0;
  for (int k = lane; k < a.ntypes * a.ntypes; k += 64) ptab[k] = ptab_g[k];
  const double4 *XQ = xq + (int64_t)f * nsites;
  const double4 ci = COM[i];
  // this lane's place among the sites of `per` molecules at a time
  const int per = 64 / nj_max, pe = lane / nj_max, pj = lane - pe * nj_max;
  const double rc2 = EW || a.q_style != CASS_Q_NONE ? fmax(a.rc2_vdw, a.rc2_coul) : a.rc2_vdw;
  int base = 0;  // wave-uniform
  while (base < b.nmols) {
    int n = 0;  // wave-uniform list length
    while (n <= kAdjList - 64 && base < b.nmols) {
      const int j = base + lane;
      bool cand = false;
      int code = -1;
      if (j < b.nmols) {
        // (squared distances: the reference's root differs at the prefilter
        // distance alone, where no site pair is within its cutoff; and its one
        // image shift of centres, whatever their distance)
        code = mcode[j];
        const double4 cj = COM[j];
        double dx = ci.x - cj.x, dy = ci.y - cj.y, dz = ci.z - cj.z;
        min_image(b, dx, dy, dz);
        const double rint = b.rcut_max + ci.w + cj.w;
        cand = code >= 0 && j != i && (b.vdw_minimum || dx * dx + dy * dy + dz * dz <= rint * rint);
      }
      const uint64_t m = __builtin_amdgcn_ballot_w64(cand);
      const int before =
          __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
      if (cand) list[n + before] = code;
      n += __popcll(m);
      base += 64;
    }
    __syncthreads();
    for (int ia0 = 0; ia0 < ni; ia0 += NI) {
      double xi[NI], yi[NI], zi[NI], qi[NI], heps[NI], acc[NI][7];
      int ti[NI];
#pragma unroll
      for (int u = 0; u < NI; ++u) {
        const int ia = min(ia0 + u, ni - 1);
        xi[u] = X[fi + ia];
        yi[u] = Y[fi + ia];
        zi[u] = Z[fi + ia];
        ti[u] = tp.atom_type[oi + ia];
        qi[u] = tp.atom_charge[oi + ia];
        const double epsd = ti[u] >= 0 ? tp.eps[ti[u] * (tp.ntypes + 1)] : 0.0;
        heps[u] = epsd > 0.0 ? 0.5 / epsd : 0.0;
#pragma unroll
        for (int k = 0; k < 7; ++k) acc[u][k] = 0.0;
      }
      int head[NI], cnt[NI];
#pragma unroll
      for (int u = 0; u < NI; ++u) head[u] = cnt[u] = 0;
      for (int c0 = 0;; c0 += per) {
        const bool last = c0 >= n;
        if (!last) {
          int site = -1;
          double4 sj = make_double4(0.0, 0.0, 0.0, 0.0);
          if (pe < per && c0 + pe < n) {
            const int code = list[c0 + pe];
            if (pj < (code & 15)) site = (code >> 4) + pj;
          }
          if (site >= 0) sj = XQ[site];
#pragma unroll
          for (int u = 0; u < NI; ++u) {
            double rx = xi[u] - sj.x, ry = yi[u] - sj.y, rz = zi[u] - sj.z;
            adj_image(b, rx, ry, rz);
            const bool close = site >= 0 && (NI == 1 || ia0 + u < ni) && rx * rx + ry * ry + rz * rz <= rc2;
            const uint64_t m = __builtin_amdgcn_ballot_w64(close);
            const int before =
                __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
            if (close) ring[u][(head[u] + cnt[u] + before) & (kAdjRing - 1)] = site;
            cnt[u] += __popcll(m);
          }
          __syncthreads();
        }
#pragma unroll
        for (int u = 0; u < NI; ++u)
          if (cnt[u] >= 64 || (last && cnt[u] > 0)) {
            const int take = min(cnt[u], 64);
            if (lane < take) {
              const int sb = ring[u][(head[u] + lane) & (kAdjRing - 1)];
              const double4 so2 = XQ[sb];
              double rx = xi[u] - so2.x, ry = yi[u] - so2.y, rz = zi[u] - so2.z;
              adj_image(b, rx, ry, rz);
              adj_pair<EW>(a, ptab, rx, ry, rz, stype[sb], so2.w, ti[u], qi[u], heps[u], acc[u]);
            }
            head[u] += take;
            cnt[u] -= take;
            __syncthreads();
          }
        if (last) break;
      }
      // the wave sums: eight lanes per value add eight lanes' parts each
#pragma unroll
      for (int u = 0; u < NI; ++u)
        if (NI == 1 || ia0 + u < ni) {
#pragma unroll
          for (int k = 0; k < 7; ++k) trans[k * 65 + lane] = acc[u][k];
          __syncthreads();
          const int k = min(lane >> 3, 6);
          double v = 0.0;
#pragma unroll
          for (int h = 0; h < 8; ++h) v += trans[k * 65 + (lane & 7) * 8 + h];
          v = dpp_add<0x111, 0xf>(v);
          v = dpp_add<0x112, 0xf>(v);
          v = dpp_add<0x114, 0xf>(v);
          if ((lane & 7) == 7 && lane < 56) sacc[ia0 + u][k] += v;
          __syncthreads();
        }
    }
    __syncthreads();
  }
  // intramolecular pairs of i (no minimum image, as
  // Compute_Molecule_Nonbond_Intra_Energy), pair p on lane p; each site's
  // terms are summed below
  const int po = pair_off[si];
  const int npair = ni * (ni - 1) / 2;
  int ia = 0, ja = 1;
  {
    int rem = lane;
    while (ia < ni - 1 && rem >= ni - 1 - ia) {
      rem -= ni - 1 - ia;
      ++ia;
    }
    ja = ia + 1 + rem;
  }
  double e = 0.0, fr = 0.0, rx = 0.0, ry = 0.0, rz = 0.0;
  double dea = 0.0, deb = 0.0, dsa = 0.0, dsb = 0.0, dqa = 0.0, dqb = 0.0;
  if (lane < npair) {
    rx = X[fi + ia] - X[fi + ja];
    ry = Y[fi + ia] - Y[fi + ja];
    rz = Z[fi + ia] - Z[fi + ja];
    const double r2 = rx * rx + ry * ry + rz * rz;
    const int ta = tp.atom_type[oi + ia], tb = tp.atom_type[oi + ja];
    const double qa = tp.atom_charge[oi + ia], qb = tp.atom_charge[oi + ja];
    const double vs = vscale[po + ia * ni + ja], qs = qscale[po + ia * ni + ja];
    if (r2 <= a.rc2_vdw && ta >= 0 && tb >= 0 && vs != 0.0) {
      const int k = ta * tp.ntypes + tb;
      const double eps0 = tp.eps[k], sig = tp.sig[k];
      double u, de, ds, dr;
      lj_pair(a, r2, eps0 * vs, sig, u, de, ds, dr);
      e += u;
      if (eps0 > 0.0) {
        dea = de * vs * eps0 * 0.5 / tp.eps[ta * (tp.ntypes + 1)];
        deb = de * vs * eps0 * 0.5 / tp.eps[tb * (tp.ntypes + 1)];
      }
      if (sig > 0.0) {
        dsa = ds * 0.5;
        dsb = ds * 0.5;
      }
      fr -= dr;
    }
    if (r2 <= a.rc2_coul && a.q_style != CASS_Q_NONE) {
      double g, dg;
      qq_pair(a, r2, true, qs, g, dg);
      e += qa * qb * g;
      dqa = qb * g;
      dqb = qa * g;
      fr -= qa * qb * dg;
    }
  }
  // per site s and derivative k: the sum over the pairs (s, ja) and (ia, s),
  // one (s, k) per lane
  e = wave_total(e);
  if (lane < npair) {
    double *o = pval[lane];
    o[0] = dea;
    o[1] = dsa;
    o[2] = dqa;
    o[3] = fr * rx;
    o[4] = fr * ry;
    o[5] = fr * rz;
    o[6] = deb;
    o[7] = dsb;
    o[8] = dqb;
  }
  __syncthreads();
  if (lane < ni * 6) {
    const int s = lane / 6, k = lane - 6 * s;
    double v = sacc[s][1 + k];
    int p = 0;
    for (int pa = 0; pa < ni; ++pa)
      for (int pb = pa + 1; pb < ni; ++pb, ++p)
        v += pa == s ? pval[p][k] : pb == s ? (k < 3 ? pval[p][6 + k] : -pval[p][k]) : 0.0;
    so[(int64_t)(fi + s) * 6 + k] = v;
  }
  if (lane == 0) {
    double ei = e;
    for (int s = 0; s < ni; ++s) ei += sacc[s][0];
    emol[(int64_t)f * b.nmols + i] = ei;
  }
}

// Per (site, frame): xq = (x, y, z, q); with Ewald also ph = (s_x, s_y,
// s_z, q) with q = 0 for sites of dead molecules.
__global__ void k_adj_prep(BoxDev b, TopoDev tp, AdjFrameView fv, const int *__restrict__ site_mol,
                           const int *__restrict__ site_spa, int nsites, double4 *__restrict__ xq,
                           double4 *__restrict__ ph) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x, f = blockIdx.y;
  if (s >= nsites) return;
  const double x = fv.x[f * fv.stride + s], y = fv.y[f * fv.stride + s], z = fv.z[f * fv.stride + s];
  const double qs = tp.atom_charge[site_spa[s]];
  xq[(int64_t)f * nsites + s] = make_double4(x, y, z, qs);
  if (!ph) return;
  const double sx = b.Li[0] * x + b.Li[3] * y + b.Li[6] * z;
  const double sy = b.Li[1] * x + b.Li[4] * y + b.Li[7] * z;
  const double sz = b.Li[2] * x + b.Li[5] * y + b.Li[8] * z;
  const double q = b.live[site_mol[s]] ? qs : 0.0;
  ph[(int64_t)f * nsites + s] = make_double4(sx, sy, sz, q);
}

// The k set as columns (n_x, |n_z|) of steps of kNyC n_y values; a step's
// place t stands for n_y = kNyC step + t and its four sign choices, kidx =
// the k index of (+n_z, +n_y), (+, -), (-, +), (-, -), or -1 where the set has
// none (also for the second sign of a zero).  Tasks: one wave of k_adj_sk
// each, 64 columns (or -1) at one step.
struct AdjCols {
  int ncols, ntasks, nslots, nw;  // nw: weights per frame
  int tx, ty, tz;                 // powers kept per axis (ty a multiple of kNyC)
  const int4 *col;                // n_x, |n_z|, steps, first weight
  const int *slot0;               // first place of the column in kidx
  const int4 *kidx;
  const int *lane_col;            // [ntasks][64]
  const int *task_step;
};

// Structure factors.  exp(i k.r) summed over a frame's sites is a contraction
// of three factors per axis: with the products of the x and z factors held
// once per site, each n_y costs eight multiply-adds for the four sign choices,
// two per k vector and site, against the sine and cosine per run and site and
// the six operations per vector of a walk along the runs (0.65 ms against 2.35
// ms for 200 frames of 2400 sites and 4117 k vectors).  The y factors are LDS
// broadcasts, which two signs of n_z share, and bound the kernel.
// part[f][split][task][32][lane]: the sums over a share of the sites, so that
// few frames fill the chip too.
__global__ void __launch_bounds__(64 * kSkWaves)
    k_adj_sk(AdjCols A, const double4 *__restrict__ ph, int nsites, int tile, int nsplit, double *__restrict__ part) {
  extern __shared__ cplx tab[];
  cplx *TX = tab, *TY = TX + tile * A.tx, *TZ = TY + tile * A.ty;
  const int tid = threadIdx.x, lane = tid & 63, nthr = blockDim.x;
  const int split = blockIdx.y, f = blockIdx.z;
  const int task = blockIdx.x * (nthr >> 6) + __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool on = task < A.ntasks;
  const int c = on ? A.lane_col[task * 64 + lane] : -1;
  const int step = on ? A.task_step[task] : 0;
  const int4 col = A.col[c < 0 ? 0 : c];
  const double4 *P = ph + (int64_t)f * nsites;
  // the sites of this split: whole tiles dealt out in order
  const int ntile = (nsites + tile - 1) / tile;
  const int t0 = (int)((int64_t)ntile * split / nsplit), t1 = (int)((int64_t)ntile * (split + 1) / nsplit);
  double acc[kNyC][8];
#pragma unroll
  for (int t = 0; t < kNyC; ++t)
#pragma unroll
    for (int k = 0; k < 8; ++k) acc[t][k] = 0.0;
  for (int tl = t0; tl < t1; ++tl) {
    __syncthreads();
    // the powers of the unit phases, one (site, axis) per thread; the charge
    // goes with the x factor
    for (int u = tid; u < 3 * tile; u += nthr) {
      const int d = u / tile, sl = u - d * tile, s = tl * tile + sl;
      const double4 p = s < nsites ? P[s] : make_double4(0.0, 0.0, 0.0, 0.0);
      cplx E;
      sincos(kTwoPi * (d == 0 ? p.x : d == 1 ? p.y : p.z), &E.im, &E.re);
      const int np = d == 0 ? A.tx : d == 1 ? A.ty : A.tz;
      cplx *T = d == 0 ? TX + sl * A.tx : d == 1 ? TY + sl * A.ty : TZ + sl * A.tz;
      cplx v = {d == 0 ? p.w : 1.0, 0.0};
      for (int k = 0; k < np; ++k) {
        T[k] = v;
        v = cmul(v, E);
      }
    }
    __syncthreads();
    if (on) {
      const cplx *px = TX + col.x, *pz = TZ + col.y, *py = TY + step * kNyC;
#pragma unroll 2
      for (int sl = 0; sl < tile; ++sl) {
        const cplx x = px[sl * A.tx], z = pz[sl * A.tz];
        const double p0 = x.re * z.re, p1 = x.im * z.im, p2 = x.re * z.im, p3 = x.im * z.re;
#pragma unroll
        for (int t = 0; t < kNyC; ++t) {
          const cplx y = py[sl * A.ty + t];
          acc[t][0] = fma(p0, y.re, acc[t][0]);
          acc[t][1] = fma(p1, y.re, acc[t][1]);
          acc[t][2] = fma(p2, y.re, acc[t][2]);
          acc[t][3] = fma(p3, y.re, acc[t][3]);
          acc[t][4] = fma(p0, y.im, acc[t][4]);
          acc[t][5] = fma(p1, y.im, acc[t][5]);
          acc[t][6] = fma(p2, y.im, acc[t][6]);
          acc[t][7] = fma(p3, y.im, acc[t][7]);
        }
      }
    }
  }
  if (!on) return;
  double *o = part + (((int64_t)f * nsplit + split) * A.ntasks + task) * (8 * kNyC * 64) + lane;
#pragma unroll
  for (int t = 0; t < kNyC; ++t)
#pragma unroll
    for (int k = 0; k < 8; ++k) o[(t * 8 + k) * 64] = acc[t][k];
}

// The structure factors from the sums: with A = exp(i (n_x a +- n_z c)) and
// (c, s) of n_y, S(+-n_y) = sum A (c +- i s).  we = the lane's reciprocal
// energy sum Cn |S|^2; per column sign and n_y the weights of k_adj_recip
// from (X, Y) = 2 Cn (Re S, Im S) of the two n_y signs: (X+ + X-, Y+ - Y-,
// Y+ + Y-, X+ - X-).
__global__ void __launch_bounds__(64) k_adj_weights(AdjCols A, EwaldDev ew, int nsplit,
                                                    const double *__restrict__ part, double4 *__restrict__ wk,
                                                    double *__restrict__ we) {
  const int task = blockIdx.x, f = blockIdx.y, lane = threadIdx.x;
  const int c = A.lane_col[task * 64 + lane], step = A.task_step[task];
  double e = 0.0;
  if (c >= 0) {
    const int4 col = A.col[c];
    double4 *W = wk + (int64_t)f * A.nw + col.w + step * kNyC;
    for (int t = 0; t < kNyC; ++t) {
      double R[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) R[k] = 0.0;
      for (int sp = 0; sp < nsplit; ++sp) {
        const double *o = part + (((int64_t)f * nsplit + sp) * A.ntasks + task) * (8 * kNyC * 64) + t * 512 + lane;
#pragma unroll
        for (int k = 0; k < 8; ++k) R[k] += o[k * 64];
      }
      const int4 ki = A.kidx[A.slot0[c] + step * kNyC + t];
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        if (g == 1 && col.y == 0) continue;
        const double sg = g ? -1.0 : 1.0;
        const double cc = R[0] - sg * R[1], sc = R[3] + sg * R[2], cs = R[4] - sg * R[5], ss = R[7] + sg * R[6];
        const int kp = g ? ki.z : ki.x, km = g ? ki.w : ki.y;
        const double cp = kp < 0 ? 0.0 : ew.cn[kp], cm = km < 0 ? 0.0 : ew.cn[km];
        const double Cp = cc - ss, Sp = sc + cs, Cm = cc + ss, Sm = sc - cs;
        e += cp * (Cp * Cp + Sp * Sp) + cm * (Cm * Cm + Sm * Sm);
        const double xp = 2.0 * cp * Cp, xm = 2.0 * cm * Cm, yp = 2.0 * cp * Sp, ym = 2.0 * cm * Sm;
        W[g * col.z * kNyC + t] = make_double4(xp + xm, yp - ym, yp + ym, xp - xm);
      }
    }
  }
  we[((int64_t)f * A.ntasks + task) * 64 + lane] = e;
}

// One lane per (site, frame): dE/dq (per unit charge) and the reciprocal
// force.  Along a column, A = a + i b at its n_x and n_z and (c, s) of n_y,
// the two n_y signs together give
//   dE/dq += a u + b v,  u = sum c W.x + s W.y,  v = sum c W.z - s W.w,
//   dE/d(x, z phase) += (n_x, n_z) (a v - b u),
//   dE/d(y phase) += sum n_y (c F + s G),  F += a W.y - b W.w, G -= a W.x + b W.z,
// eight multiply-adds per two k vectors with the sines and cosines of the
// lane's n_y and F, G in registers (NCH steps of kNyC; NCH 0: any number of
// n_y, the factors by products on the way), against the eight and the row
// bases per k vector of a walk along the runs (0.64 ms against 1.33 ms for
// 200 frames of 2400 sites and 4117 k vectors).  The weights are uniform over
// the wave and come in as one stream.
template <int NCH>
__global__ void __launch_bounds__(64) k_adj_recip(BoxDev b, TopoDev tp, AdjCols A, const int *__restrict__ site_mol,
                                                  const int *__restrict__ site_spa, const double4 *__restrict__ ph,
                                                  int nsites, const double4 *__restrict__ wk,
                                                  double4 *__restrict__ srec) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x, f = blockIdx.y;
  const double4 p = ph[(int64_t)f * nsites + min(s, nsites - 1)];
  cplx Ea, Eb, Ec;
  sincos(kTwoPi * p.x, &Ea.im, &Ea.re);
  sincos(kTwoPi * p.y, &Eb.im, &Eb.re);
  sincos(kTwoPi * p.z, &Ec.im, &Ec.re);
  constexpr int NY = NCH > 0 ? NCH * kNyC : 1;
  double yc[NY], ys[NY], F[NY], G[NY];
  {
    cplx v = {1.0, 0.0};
#pragma unroll
    for (int t = 0; t < NY; ++t) {
      yc[t] = v.re;
      ys[t] = v.im;
      F[t] = G[t] = 0.0;
      v = cmul(v, Eb);
    }
  }
  const double4 *W = wk + (int64_t)f * A.nw;
  double4 nxt[kNyC];
#pragma unroll
  for (int t = 0; t < kNyC; ++t) nxt[t] = W[t];
  cplx X = {1.0, 0.0}, Z = {1.0, 0.0};
  int cx = 0, cz = 0;  // the powers X and Z hold
  double dq = 0.0, gx = 0.0, gy = 0.0, gz = 0.0;
  for (int r = 0; r < A.ncols; ++r) {
    const int4 col = A.col[r];
    if (col.y != cz) {
      Z = col.y == cz + 1 ? cmul(Z, Ec) : cpow_int(Ec, col.y);
      cz = col.y;
    }
    if (col.x != cx) {
      X = col.x == cx + 1 ? cmul(X, Ea) : cpow_int(Ea, col.x);
      cx = col.x;
    }
    const double p0 = X.re * Z.re, p1 = X.im * Z.im, p2 = X.re * Z.im, p3 = X.im * Z.re;
    for (int g = 0; g < (col.y ? 2 : 1); ++g) {
      const double a = g ? p0 + p1 : p0 - p1, bb = g ? p3 - p2 : p3 + p2;
      double u = 0.0, v = 0.0;
      if (NCH > 0) {
#pragma unroll
        for (int h = 0; h < NCH; ++h) {
          if (h >= col.z) break;
          // this step's weights came in during the last one
          double4 cur[kNyC];
#pragma unroll
          for (int t = 0; t < kNyC; ++t) cur[t] = nxt[t];
          W += kNyC;
#pragma unroll
          for (int t = 0; t < kNyC; ++t) nxt[t] = W[t];
#pragma unroll
          for (int t = 0; t < kNyC; ++t) {
            const int n = h * kNyC + t;
            const double4 w = cur[t];
            u = fma(yc[n], w.x, fma(ys[n], w.y, u));
            v = fma(yc[n], w.z, fma(-ys[n], w.w, v));
            F[n] = fma(a, w.y, fma(-bb, w.w, F[n]));
            G[n] = fma(-a, w.x, fma(-bb, w.z, G[n]));
          }
        }
      } else {
        cplx y = {1.0, 0.0};
        double du = 0.0, dv = 0.0;
        for (int n = 0; n < col.z * kNyC; ++n) {
          const double4 w = W[n];
          u = fma(y.re, w.x, fma(y.im, w.y, u));
          v = fma(y.re, w.z, fma(-y.im, w.w, v));
          du = fma((double)n, fma(y.re, w.y, -y.im * w.x), du);
          dv = fma((double)n, fma(y.im, w.z, y.re * w.w), dv);
          y = cmul(y, Eb);
        }
        gy += a * du - bb * dv;
        W += col.z * kNyC;
      }
      dq = fma(a, u, fma(bb, v, dq));
      const double gr = a * v - bb * u;
      gx = fma(gr, (double)col.x, gx);
      gz = fma(gr, (double)(g ? -col.y : col.y), gz);
    }
  }
  if (NCH > 0) {
#pragma unroll
    for (int n = 1; n < NY; ++n) gy = fma((double)n, fma(yc[n], F[n], ys[n] * G[n]), gy);
  }
  if (s >= nsites) return;
  const bool live = b.live[site_mol[s]] != 0;
  const double q = live ? tp.atom_charge[site_spa[s]] : 0.0;
  // F_e = -q cf 2 pi sum_d G_d dS_d/dr_e, dS_d/dr_e = Li[d + 3e]
  const double w = -q * kChargeFactor * kTwoPi;
  const double fx = w * (gx * b.Li[0] + gy * b.Li[1] + gz * b.Li[2]);
  const double fy = w * (gx * b.Li[3] + gy * b.Li[4] + gz * b.Li[5]);
  const double fz = w * (gx * b.Li[6] + gy * b.Li[7] + gz * b.Li[8]);
  srec[(int64_t)f * nsites + s] = live ? make_double4(dq * kChargeFactor, fx, fy, fz) : make_double4(0, 0, 0, 0);
}

template <int NV>
__device__ inline void block_sum(double (&v)[NV], double (*red)[4]) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const double sv = wave_sum_x(v[k]);
    if (lane == 0) red[k][wid] = sv;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NV; ++k) v[k] = (red[k][0] + red[k][1]) + (red[k][2] + red[k][3]);
}

// One workgroup (256 lanes) per frame: fout[f] = (E, dE/d eps_t, dE/d sig_t,
// dE/d q_k) without the frame-independent terms; forces[f][site] if asked.
__global__ void __launch_bounds__(256) k_adj_frame(BoxDev b, TopoDev tp, int nsites, int nwe,
                                                   const int *__restrict__ site_spa,
                                                   const double *__restrict__ site_out,
                                                   const double *__restrict__ emol, const double *__restrict__ we,
                                                   const double4 *__restrict__ srec, double *__restrict__ fout,
                                                   double *__restrict__ forces) {
  __shared__ double red[kAdjOut][4];
  const int f = blockIdx.x;
  double v[kAdjOut];
#pragma unroll
  for (int k = 0; k < kAdjOut; ++k) v[k] = 0.0;
  for (int i = threadIdx.x; i < b.nmols; i += 256) v[0] += emol[(int64_t)f * b.nmols + i];
  if (srec) {
    double er = 0.0;
    for (int k = threadIdx.x; k < nwe; k += 256) er += we[(int64_t)f * nwe + k];
    v[0] += er * kChargeFactor;
  }
  const double *so = site_out + (int64_t)f * nsites * 6;
  for (int s = threadIdx.x; s < nsites; s += 256) {
    const int spa = site_spa[s], t = tp.atom_type[spa];
    const double de = so[6 * s], ds = so[6 * s + 1];
    double dq = so[6 * s + 2];
    double fx = so[6 * s + 3], fy = so[6 * s + 4], fz = so[6 * s + 5];
    if (srec) {
      const double4 r = srec[(int64_t)f * nsites + s];
      dq += r.x;
      fx += r.y;
      fy += r.z;
      fz += r.w;
    }
#pragma unroll
    for (int k = 0; k < kAdjTypes; ++k) {
      v[1 + k] += (t == k) ? de : 0.0;
      v[1 + kAdjTypes + k] += (t == k) ? ds : 0.0;
    }
#pragma unroll
    for (int k = 0; k < kAdjKinds; ++k) v[1 + 2 * kAdjTypes + k] += (spa == k) ? dq : 0.0;
    if (forces) {
      double *fo = forces + ((int64_t)f * nsites + s) * 3;
      fo[0] = fx;
      fo[1] = fy;
      fo[2] = fz;
    }
  }
  block_sum<kAdjOut>(v, red);
  if (threadIdx.x < kAdjOut) {
    double r = v[0];
#pragma unroll
    for (int k = 1; k < kAdjOut; ++k) r = (threadIdx.x == k) ? v[k] : r;
    fout[(int64_t)f * kAdjOut + threadIdx.x] = r;
  }
}

typedef void (*pairs_kernel_t)(BoxDev, TopoDev, AdjParams, AdjFrameView, const double4 *, const int *,
                               const double4 *, const double *, const double *, const int *, const int *, int, int, double *,
                               double *);

// The pair kernel for the charge style (Ewald inline, the other styles
// through qq_pair).
pairs_kernel_t pairs_kernel(bool ewald) { return ewald ? k_adj_pairs<true, 3> : k_adj_pairs<false, 3>; }

// The reciprocal kernel for n_y up to ny (n_y factors in registers up to 15).
typedef void (*recip_kernel_t)(BoxDev, TopoDev, AdjCols, const int *, const int *, const double4 *, int,
                               const double4 *, double4 *);
recip_kernel_t recip_kernel(int ny) {
  return ny < 2 * kNyC   ? k_adj_recip<2>
         : ny < 3 * kNyC ? k_adj_recip<3>
         : ny < 4 * kNyC ? k_adj_recip<4>
                         : k_adj_recip<0>;
}

size_t up256(size_t x) { return (x + 255) & ~(size_t)255; }

// The columns of a k set (AdjCols) as one table: col, kidx, slot0, lane_col,
// task_step.
struct ColTable {
  AdjCols A{};
  std::vector<int32_t> words;
  size_t o_col = 0, o_kidx = 0, o_slot0 = 0, o_lane = 0, o_step = 0;
};

void build_columns(const std::vector<int32_t> &kn, const int32_t *kmax, ColTable &T) {
  const int nxs = kmax[0] + 1, nzs = kmax[2] + 1, K = (int)kn.size() / 3;
  // the largest |n_y| of every (|n_z|, n_x), -1 for none
  std::vector<int> top((size_t)nxs * nzs, -1), id((size_t)nxs * nzs, -1);
  for (int k = 0; k < K; ++k) {
    int &t = top[(size_t)std::abs(kn[3 * k + 2]) * nxs + kn[3 * k]];
    t = std::max(t, std::abs(kn[3 * k + 1]));
  }
  AdjCols &A = T.A;
  std::vector<int32_t> col, slot0;
  for (int g = 0; g < nxs * nzs; ++g)
    if (top[g] >= 0) {
      const int steps = top[g] / kNyC + 1, nz = g / nxs;
      id[g] = A.ncols++;
      col.insert(col.end(), {g % nxs, nz, steps, A.nw});
      slot0.push_back(A.nslots);
      A.nslots += steps * kNyC;
      A.nw += (nz ? 2 : 1) * steps * kNyC;
    }
  std::vector<int32_t> kidx((size_t)4 * A.nslots, -1);
  for (int k = 0; k < K; ++k) {
    const int nx = kn[3 * k], ny = kn[3 * k + 1], nz = kn[3 * k + 2];
    const int c = id[(size_t)std::abs(nz) * nxs + nx];
    kidx[4 * (size_t)(slot0[c] + std::abs(ny)) + (nz < 0 ? 2 : 0) + (ny < 0 ? 1 : 0)] = k;
  }
  // tasks: per step the columns that reach it, 64 at a time
  std::vector<int32_t> lane, step;
  const int most = kmax[1] / kNyC + 1;
  for (int h = 0; h < most; ++h) {
    int n = 0;
    for (int c = 0; c < A.ncols; ++c)
      if (col[4 * c + 2] > h) {
        if (n++ % 64 == 0) step.push_back(h);
        lane.push_back(c);
      }
    while (lane.size() % 64) lane.push_back(-1);
  }
  A.nw += kNyC;  // (the stream is read one step ahead)
  A.ntasks = (int)step.size();
  A.tx = nxs;
  A.ty = most * kNyC;
  A.tz = nzs;
  auto put = [&](const std::vector<int32_t> &v) {
    const size_t o = T.words.size();
    T.words.insert(T.words.end(), v.begin(), v.end());
    T.words.resize((T.words.size() + 3) & ~(size_t)3);
    return o;
  };
  T.o_col = put(col);
  T.o_kidx = put(kidx);
  T.o_slot0 = put(slot0);
  T.o_lane = put(lane);
  T.o_step = put(step);
}

}  // namespace

BoxDev cass_box_view(const cass_engine *e, const cass_box_state &b);
TopoDev cass_topo_view(const cass_engine *e);
EwaldDev cass_ewald_view(const cass_box_state &b);
double4 cass_host_com(const cass_engine *e, int s, const double *xyz);

// ------------------------------------------------------------------ host

// The styles, sizes and mixing the adjoint supports; fills the pair
// parameters.
static int adjoint_check(cass_engine *e, const cass_box_state &b, AdjParams &a) {
  const cass_params &p = b.p;
  if (p.vdw_style == CASS_VDW_MIE) return cass_fail(e, CASS_ERR_ARG, "adjoint supports LJ only");
  if (p.vdw_style == CASS_VDW_LJ &&
      !(p.vdw_sum_style == CASS_SUM_CUT || p.vdw_sum_style == CASS_SUM_CUT_TAIL ||
        p.vdw_sum_style == CASS_SUM_CUT_SHIFT))
    return cass_fail(e, CASS_ERR_ARG, "adjoint supports cut, cut_tail and cut_shift");
  if (e->ntypes > kAdjTypes || e->natoms_total > kAdjKinds) return cass_fail(e, CASS_ERR_ARG, "adjoint size limits");
  for (int s = 0; s < e->nspecies; ++s)
    if (e->sp_natoms[s] > kAdjSites) return cass_fail(e, CASS_ERR_ARG, "adjoint: molecule too large");
  if (b.nsites >= (1 << 27)) return cass_fail(e, CASS_ERR_ARG, "adjoint: too many sites");
  // the derivatives go through Lorentz-Berthelot mixing of the diagonal
  const int nt = e->ntypes;
  for (int i = 0; i < nt; ++i)
    for (int j = 0; j < nt; ++j) {
      const double ei = e->eps[i * nt + i], ej = e->eps[j * nt + j];
      const double si = e->sig[i * nt + i], sj = e->sig[j * nt + j];
      const double em = (i == j) ? ei : ((ei <= 1e-7 || ej <= 1e-7) ? 0.0 : std::sqrt(ei * ej));
      const double sm = (i == j) ? si : ((si <= 1e-7 || sj <= 1e-7) ? 0.0 : (si + sj) * 0.5);
      if (std::fabs(e->eps[i * nt + j] - em) > 1e-12 * std::max(1.0, std::fabs(em)) ||
          std::fabs(e->sig[i * nt + j] - sm) > 1e-12 * std::max(1.0, std::fabs(sm)))
        return cass_fail(e, CASS_ERR_ARG, "adjoint needs Lorentz-Berthelot mixing of the per-type parameters");
    }
  std::memset(&a, 0, sizeof(a));
  a.ntypes = nt;
  a.q_style = p.charge_style;
  a.vdw_sum = p.vdw_sum_style;
  a.rc2_vdw = p.vdw_style == CASS_VDW_NONE ? -1.0 : p.rcut_vdwsq;
  a.inv_rc2_vdw = p.rcut_vdwsq > 0.0 ? 1.0 / p.rcut_vdwsq : 0.0;
  a.rc2_coul = p.charge_style == CASS_Q_MINIMUM ? 1e300 : p.rcut_coulsq;
  a.rc_coul = p.rcut_coul;
  a.alpha = p.alpha_ewald;
  a.alpha_dsf = p.alpha_dsf;
  a.dsf1 = p.dsf_factor1;
  a.dsf2 = p.dsf_factor2;
  return CASS_OK;
}

// Frame-independent terms: the self energy (Ewald, DSF) and the LJ tail
// correction (energy_routines.f90:2956-3023) with their derivatives, added
// to out[kAdjOut].
static void adjoint_constants(const cass_engine *e, const cass_box_state &b, double *out) {
  const cass_params &p = b.p;
  const int nt = e->ntypes;
  double selfc = 0.0;
  if (p.charge_style == CASS_Q_EWALD) selfc = kChargeFactor * p.alpha_ewald / kRootPi;
  else if (p.charge_style == CASS_Q_DSF) selfc = (p.alpha_dsf / kRootPi + p.dsf_factor1 / 2.0) * kChargeFactor;
  std::vector<double> nb(nt, 0.0);
  for (int m = 0; m < b.nmols; ++m) {
    if (!b.live[m]) continue;
    const int sp = b.mol_species[m];
    for (int aa = 0; aa < e->sp_natoms[sp]; ++aa) {
      const int k = e->sp_atom_off[sp] + aa;
      const double q = e->atom_charge[k];
      out[0] += -q * q * selfc;
      out[1 + 2 * kAdjTypes + k] += -2.0 * q * selfc;
      const int t = e->atom_type[k];
      if (t >= 0) nb[t] += 1.0;
    }
  }
  if (p.vdw_sum_style == CASS_SUM_CUT_TAIL && p.vdw_style == CASS_VDW_LJ) {
    const double pre = 2.0 * kPi / p.volume;
    for (int i = 0; i < nt; ++i)
      for (int j = 0; j < nt; ++j) {
        const double eps = e->eps[i * nt + j], sig = e->sig[i * nt + j];
        const double s2 = sig * sig, s6 = s2 * s2 * s2, s12 = s6 * s6;
        const double w = pre * nb[i] * nb[j];
        const double f = s12 / (9.0 * p.rcut9) - s6 / (3.0 * p.rcut3);
        out[0] += w * 4.0 * eps * f;
        if (eps > 0.0) {
          out[1 + i] += w * 4.0 * f * eps / (2.0 * e->eps[i * nt + i]);
          out[1 + j] += w * 4.0 * f * eps / (2.0 * e->eps[j * nt + j]);
        }
        if (sig > 0.0) {
          const double dfs = (12.0 * s12 / (9.0 * p.rcut9) - 6.0 * s6 / (3.0 * p.rcut3)) / sig;
          out[1 + kAdjTypes + i] += w * 4.0 * eps * dfs * 0.5;
          out[1 + kAdjTypes + j] += w * 4.0 * eps * dfs * 0.5;
        }
      }
  }
}

// The kernels over count frames of fv; fout (count x kAdjOut) and, if
// forces is not null, forces (count x nsites x 3) receive the results on the
// host.
static int adjoint_run(cass_engine *e, int box, const AdjParams &a, const AdjFrameView &fv, int count,
                       double *fout_h, double *forces_h) {
  cass_box_state &b = e->boxes[box];
  const int ns = b.nsites, nm = b.nmols;
  const bool ewald = b.p.charge_style == CASS_Q_EWALD;
  int rc;
  if (ewald && !b.ewald_ready) {
    int32_t nv;
    if ((rc = cass_ewald_setup(e, box, &nv))) return rc;
  }
  // the reciprocal part: the k columns, and over how many shares of the sites
  // the structure factors are split (a share's sums are 16 KB a task; four
  // waves per SIMD where the frames alone give fewer)
  ColTable ct;
  const bool recip = ewald && b.nvecs > 0 && ns > 0;
  int tile = kSkSites, nsplit = 1;
  size_t sk_lds = 0;
  if (recip) {
    build_columns(b.kn_h, b.kmax, ct);
    const size_t per_site = sizeof(cplx) * (ct.A.tx + ct.A.ty + ct.A.tz);
    while (tile > 1 && per_site * tile > 48 * 1024) tile /= 2;
    sk_lds = per_site * tile;
    const int64_t waves = (int64_t)count * ct.A.ntasks;
    nsplit = (int)std::max<int64_t>(1, std::min<int64_t>((ns + tile - 1) / tile, (4096 + waves - 1) / waves));
  }
  const size_t part_bytes = recip ? sizeof(double) * 8 * kNyC * 64 * (size_t)ct.A.ntasks * nsplit : 0;
  // site tables and intramolecular scale tables
  std::vector<int32_t> site_mol(ns), site_spa(ns);
  for (int m = 0; m < nm; ++m)
    for (int aa = 0; aa < e->sp_natoms[b.mol_species[m]]; ++aa) {
      site_mol[b.mol_first[m] + aa] = m;
      site_spa[b.mol_first[m] + aa] = e->sp_atom_off[b.mol_species[m]] + aa;
    }
  const size_t npair_tab = e->vdw_scale.size();
  const size_t o_mol = 0, o_spa = up256(o_mol + 4 * (size_t)ns), o_poff = up256(o_spa + 4 * (size_t)ns),
               o_vs = up256(o_poff + 4 * (size_t)e->nspecies), o_qs = up256(o_vs + 8 * std::max<size_t>(1, npair_tab)),
               o_ptab = up256(o_qs + 8 * std::max<size_t>(1, npair_tab)),
               o_stype = up256(o_ptab + 32 * (size_t)e->ntypes * e->ntypes + 32),
               o_mcode = up256(o_stype + 4 * (size_t)ns), o_col = up256(o_mcode + 4 * (size_t)nm),
               o_var = up256(o_col + 4 * ct.words.size());
  // per-frame buffers: site_out (6 ns), emol (nm), xq and ph (4 ns), wk (4
  // nw), we, the structure factors' parts, srec (4 ns), fout (kAdjOut), forces
  // (3 ns)
  const size_t per_frame = up256(48 * (size_t)ns) + up256(8 * (size_t)nm) + up256(32 * (size_t)ns) +
                           (recip ? up256(32 * (size_t)ns) + up256(32 * (size_t)ct.A.nw) +
                                        up256(512 * (size_t)ct.A.ntasks) + up256(part_bytes) + up256(32 * (size_t)ns)
                                  : 0) +
                           up256(8 * kAdjOut) + (forces_h ? up256(24 * (size_t)ns) : 0);
  const size_t budget = (size_t)1 << 30;
  const int chunk = (int)std::max<size_t>(1, std::min<size_t>((size_t)count, budget / per_frame));
  char *s0 = (char *)cass_scratch(e, o_var + per_frame * chunk);
  if (!s0) return cass_fail(e, CASS_ERR_NOMEM, "adjoint scratch");
  int32_t *d_mol = (int32_t *)(s0 + o_mol), *d_spa = (int32_t *)(s0 + o_spa), *d_poff = (int32_t *)(s0 + o_poff);
  double *d_vs = (double *)(s0 + o_vs), *d_qs = (double *)(s0 + o_qs);
  double4 *d_ptab = (double4 *)(s0 + o_ptab);
  int32_t *d_stype = (int32_t *)(s0 + o_stype);
  const int32_t *d_mcode = (const int32_t *)(s0 + o_mcode);
  {
    // site types; per molecule (first site) << 4 | sites, -1 for a dead one
    std::vector<int32_t> st((o_col - o_stype) / 4);
    for (int s = 0; s < ns; ++s) st[s] = e->atom_type[site_spa[s]];
    for (int m = 0; m < nm; ++m)
      st[(o_mcode - o_stype) / 4 + m] = b.live[m] ? (b.mol_first[m] << 4) | e->sp_natoms[b.mol_species[m]] : -1;
    HIP_TRY(e, hipMemcpyAsync(d_stype, st.data(), 4 * st.size(), hipMemcpyHostToDevice, e->stream));
    HIP_TRY(e, hipStreamSynchronize(e->stream));  // st goes out of scope
  }
  {
    // per type pair (eps, sigma^2, 1/sigma, 0) of the engine's table
    const int nt = e->ntypes;
    std::vector<double4> pt((size_t)nt * nt + 1);
    for (int k = 0; k < nt * nt; ++k) {
      const double sg = e->sig[k];
      pt[k] = make_double4(e->eps[k], sg * sg, sg > 0.0 ? 1.0 / sg : 0.0, 0.0);
    }
    HIP_TRY(e, hipMemcpyAsync(d_ptab, pt.data(), sizeof(double4) * pt.size(), hipMemcpyHostToDevice, e->stream));
  }
  HIP_TRY(e, hipMemcpyAsync(d_mol, site_mol.data(), 4 * (size_t)ns, hipMemcpyHostToDevice, e->stream));
  HIP_TRY(e, hipMemcpyAsync(d_spa, site_spa.data(), 4 * (size_t)ns, hipMemcpyHostToDevice, e->stream));
  HIP_TRY(e, hipMemcpyAsync(d_poff, e->sp_pair_off.data(), 4 * (size_t)e->nspecies, hipMemcpyHostToDevice,
                            e->stream));
  if (npair_tab) {
    HIP_TRY(e, hipMemcpyAsync(d_vs, e->vdw_scale.data(), 8 * npair_tab, hipMemcpyHostToDevice, e->stream));
    HIP_TRY(e, hipMemcpyAsync(d_qs, e->q_scale.data(), 8 * npair_tab, hipMemcpyHostToDevice, e->stream));
  }
  if (recip) {
    HIP_TRY(e, hipMemcpyAsync(s0 + o_col, ct.words.data(), 4 * ct.words.size(), hipMemcpyHostToDevice, e->stream));
    const int32_t *w = (const int32_t *)(s0 + o_col);
    ct.A.col = (const int4 *)(w + ct.o_col);
    ct.A.kidx = (const int4 *)(w + ct.o_kidx);
    ct.A.slot0 = w + ct.o_slot0;
    ct.A.lane_col = w + ct.o_lane;
    ct.A.task_step = w + ct.o_step;
  }
  char *v0 = s0 + o_var;
  size_t o = 0;
  auto take = [&](size_t bytes) {
    char *p = v0 + o;
    o += up256(bytes);
    return p;
  };
  double *site_out = (double *)take(48 * (size_t)ns * chunk);
  double *emol = (double *)take(8 * (size_t)nm * chunk);
  double4 *xq = (double4 *)take(32 * (size_t)ns * chunk);
  double4 *ph = nullptr, *wk = nullptr, *srec = nullptr;
  double *we = nullptr, *part = nullptr;
  if (recip) {
    ph = (double4 *)take(32 * (size_t)ns * chunk);
    wk = (double4 *)take(32 * (size_t)ct.A.nw * chunk);
    we = (double *)take(512 * (size_t)ct.A.ntasks * chunk);
    part = (double *)take(part_bytes * chunk);
    srec = (double4 *)take(32 * (size_t)ns * chunk);
  }
  double *fout = (double *)take(8 * kAdjOut * (size_t)chunk);
  double *fdev = forces_h ? (double *)take(24 * (size_t)ns * chunk) : nullptr;
  const BoxDev bv = cass_box_view(e, b);
  const TopoDev tv = cass_topo_view(e);
  const EwaldDev ew = ewald ? cass_ewald_view(b) : EwaldDev{};
  const pairs_kernel_t pk = pairs_kernel(ewald);
  int nj_max = 1;
  for (int m = 0; m < nm; ++m) nj_max = std::max(nj_max, e->sp_natoms[b.mol_species[m]]);
  HIP_TRY(e, hipEventRecord(e->ev0, e->stream));
  for (int c0 = 0; c0 < count; c0 += chunk) {
    const int nf = std::min(chunk, count - c0);
    AdjFrameView v = fv;
    v.x += c0 * fv.stride;
    v.y += c0 * fv.stride;
    v.z += c0 * fv.stride;
    v.com = (const double4 *)((const double *)fv.com + c0 * fv.stride);
    if (ns > 0)
      hipLaunchKernelGGL(k_adj_prep, dim3((ns + 255) / 256, nf), dim3(256), 0, e->stream, bv, tv, v, d_mol, d_spa,
                         ns, xq, ph);
    if (nm > 0)
      hipLaunchKernelGGL(pk, dim3(nm, nf), dim3(64), 0, e->stream, bv, tv, a, v, xq, d_stype, d_ptab, d_vs, d_qs,
                         d_poff, d_mcode, ns, nj_max, site_out, emol);
    if (recip) {
      // the tasks in workgroups of equal size
      const int groups = (ct.A.ntasks + kSkWaves - 1) / kSkWaves, wpb = (ct.A.ntasks + groups - 1) / groups;
      if (sk_lds > 64 * 1024)
        HIP_TRY(e, hipFuncSetAttribute((const void *)k_adj_sk, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sk_lds));
      hipLaunchKernelGGL(k_adj_sk, dim3((ct.A.ntasks + wpb - 1) / wpb, nsplit, nf), dim3(64 * wpb), sk_lds, e->stream,
                         ct.A, ph, ns, tile, nsplit, part);
      hipLaunchKernelGGL(k_adj_weights, dim3(ct.A.ntasks, nf), dim3(64), 0, e->stream, ct.A, ew, nsplit, part, wk, we);
      hipLaunchKernelGGL(recip_kernel(b.kmax[1]), dim3((ns + 63) / 64, nf), dim3(64), 0, e->stream, bv, tv, ct.A,
                         d_mol, d_spa, ph, ns, wk, srec);
    }
    hipLaunchKernelGGL(k_adj_frame, dim3(nf), dim3(256), 0, e->stream, bv, tv, ns, ct.A.ntasks * 64, d_spa, site_out,
                       emol, we, srec, fout, fdev);
    if (hipGetLastError() != hipSuccess) return cass_fail(e, CASS_ERR_HIP, "adjoint launch");
    HIP_TRY(e, hipMemcpyAsync(fout_h + (size_t)c0 * kAdjOut, fout, 8 * kAdjOut * (size_t)nf, hipMemcpyDeviceToHost,
                              e->stream));
    if (forces_h)
      HIP_TRY(e, hipMemcpyAsync(forces_h + (size_t)c0 * 3 * ns, fdev, 24 * (size_t)ns * nf, hipMemcpyDeviceToHost,
                                e->stream));
  }
  HIP_TRY(e, hipEventRecord(e->ev1, e->stream));
  HIP_TRY(e, hipStreamSynchronize(e->stream));
  float ms = 0.0f;
  if (hipEventElapsedTime(&ms, e->ev0, e->ev1) == hipSuccess) e->last_kernel_ms = ms;
  return CASS_OK;
}

// Unpacks count frames of kAdjOut values (plus the constant terms) into the
// caller's arrays.
static void adjoint_unpack(const cass_engine *e, const cass_box_state &b, int count, const double *fout,
                           double *energy, double *de_deps, double *de_dsig, double *de_dq) {
  const int nt = e->ntypes, nk = e->natoms_total;
  std::vector<double> cst(kAdjOut, 0.0);
  adjoint_constants(e, b, cst.data());
  for (int f = 0; f < count; ++f) {
    const double *v = fout + (size_t)f * kAdjOut;
    if (energy) energy[f] = v[0] + cst[0];
    for (int t = 0; t < nt; ++t) {
      if (de_deps) de_deps[(size_t)f * nt + t] = v[1 + t] + cst[1 + t];
      if (de_dsig) de_dsig[(size_t)f * nt + t] = v[1 + kAdjTypes + t] + cst[1 + kAdjTypes + t];
    }
    if (de_dq)
      for (int k = 0; k < nk; ++k) de_dq[(size_t)f * nk + k] = v[1 + 2 * kAdjTypes + k] + cst[1 + 2 * kAdjTypes + k];
  }
}

extern "C" int cass_adjoint(cass_engine *e, int32_t box, double *energy, double *de_deps, double *de_dsig,
                            double *de_dq, double *forces) {
  if (!e || box < 0 || box >= (int)e->boxes.size()) return CASS_ERR_ARG;
  cass_box_state &b = e->boxes[box];
  AdjParams a;
  int rc = adjoint_check(e, b, a);
  if (rc) return rc;
  if (hipSetDevice(e->device) != hipSuccess) return CASS_ERR_HIP;
  AdjFrameView fv{b.x, b.y, b.z, b.comd, 0};
  double fout[kAdjOut];
  if ((rc = adjoint_run(e, box, a, fv, 1, fout, forces))) return rc;
  adjoint_unpack(e, b, 1, fout, energy, de_deps, de_dsig, de_dq);
  return CASS_OK;
}

extern "C" int cass_adjoint_set_frames(cass_engine *e, int32_t box, int32_t nframes, const double *xyz) {
  if (!e || box < 0 || box >= (int)e->boxes.size() || nframes < 0 || (nframes > 0 && !xyz)) return CASS_ERR_ARG;
  cass_box_state &b = e->boxes[box];
  if (hipSetDevice(e->device) != hipSuccess) return CASS_ERR_HIP;
  const int ns = b.nsites, nm = b.nmols;
  // per frame: x[ns], y[ns], z[ns], padded to 4 doubles, then comd[nm]
  const int64_t stride = (int64_t)((3 * (size_t)ns + 3) / 4 * 4) + 4 * (int64_t)nm;
  const size_t bytes = 8 * (size_t)stride * (size_t)nframes;
  for (size_t k = 0; k < 3 * (size_t)ns * (size_t)nframes; ++k)
    if (!std::isfinite(xyz[k])) return cass_fail(e, CASS_ERR_ARG, "non-finite coordinate in a frame");
  AdjFrames &fr = e->adjf;
  HIP_TRY(e, hipStreamSynchronize(e->stream));
  if (bytes > fr.cap) {
    if (fr.dev) (void)hipFree(fr.dev);
    fr.dev = nullptr;
    fr.cap = 0;
    if (hipMalloc((void **)&fr.dev, bytes) != hipSuccess) {
      fr.box = -1;
      fr.nframes = 0;
      return cass_fail(e, CASS_ERR_NOMEM, "adjoint frames");
    }
    fr.cap = bytes;
  }
  // staged through pinned memory one frame at a time
  double *h = (double *)cass_pinned(e, 8 * (size_t)stride);
  if (!h) return cass_fail(e, CASS_ERR_NOMEM, "pinned staging");
  for (int f = 0; f < nframes; ++f) {
    const double *src = xyz + 3 * (size_t)ns * f;
    for (int s = 0; s < ns; ++s) {
      h[s] = src[3 * s];
      h[ns + s] = src[3 * s + 1];
      h[2 * ns + s] = src[3 * s + 2];
    }
    double4 *com = (double4 *)(h + (stride - 4 * (int64_t)nm));
    for (int m = 0; m < nm; ++m) com[m] = cass_host_com(e, b.mol_species[m], src + 3 * (size_t)b.mol_first[m]);
    HIP_TRY(e, hipMemcpyAsync(fr.dev + (size_t)f * stride, h, 8 * (size_t)stride, hipMemcpyHostToDevice, e->stream));
    HIP_TRY(e, hipStreamSynchronize(e->stream));
  }
  fr.box = box;
  fr.nframes = nframes;
  fr.nsites = ns;
  fr.nmols = nm;
  fr.stride = stride;
  fr.mol_species = b.mol_species;
  fr.mol_first = b.mol_first;
  return CASS_OK;
}

extern "C" int cass_adjoint_frames(cass_engine *e, int32_t box, int32_t first, int32_t count, double *energy,
                                   double *de_deps, double *de_dsig, double *de_dq, double *forces) {
  if (!e || box < 0 || box >= (int)e->boxes.size()) return CASS_ERR_ARG;
  cass_box_state &b = e->boxes[box];
  const AdjFrames &fr = e->adjf;
  if (fr.box != box || !fr.dev) return cass_fail(e, CASS_ERR_STATE, "no frames stored for this box");
  if (fr.nsites != b.nsites || fr.nmols != b.nmols || fr.mol_species != b.mol_species || fr.mol_first != b.mol_first)
    return cass_fail(e, CASS_ERR_STATE, "the box's molecules changed since the frames were stored");
  if (first < 0 || count < 0 || (int64_t)first + count > fr.nframes) return cass_fail(e, CASS_ERR_ARG, "frame range");
  AdjParams a;
  int rc = adjoint_check(e, b, a);
  if (rc) return rc;
  if (count == 0) return CASS_OK;
  if (hipSetDevice(e->device) != hipSuccess) return CASS_ERR_HIP;
  const int ns = b.nsites;
  const double *base = fr.dev + (size_t)first * fr.stride;
  AdjFrameView fv{base, base + ns, base + 2 * (size_t)ns,
                  (const double4 *)(base + (fr.stride - 4 * (int64_t)b.nmols)), fr.stride};
  std::vector<double> fout((size_t)count * kAdjOut);
  if ((rc = adjoint_run(e, box, a, fv, count, fout.data(), forces))) return rc;
  adjoint_unpack(e, b, count, fout.data(), energy, de_deps, de_dsig, de_dq);
  return CASS_OK;
}
