// kernels.h -- device-side views, helpers and kernel declarations.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "pair.h"

namespace cass {

constexpr int kMaxBlock = 256;        // block size of the reduction kernels
constexpr int kMaxSites = 64;         // sites per molecule (trial kernels)
constexpr int kMaxWidomSites = 8;     // sites per Widom test molecule

// Box view (per-box constants are passed by value in the kernel arguments).
struct BoxDev {
  const double *x, *y, *z;
  const int *first, *species, *live;
  const double4 *comd;
  int nmols;
  int cubic, vdw_minimum;
  double L[3], hL[3];
  double Li[9], Lc[9];   // length_inv and length, column-major
  double rcut_max, rcut_cbmc;
  // tabulated CBMC pair energies (Create_Atompair_Nrg_table): vdW per
  // (type pair, bin) at apt[(ti * ntypes + tj) * apt_res + bin], the charge
  // factor f2 per bin at apt[ntypes^2 * apt_res + bin]; apt_res = 0: off
  const double *apt;
  int apt_res;
  double apt_step, apt_shift, apt_rcs;  // rsq_step, rsq_shifter, rcut_cbmcsq - rsq_shifter
};

// Topology view (nonbond tables and per species-atom data).
struct TopoDev {
  const double *eps, *sig, *mn, *mm;
  const int *atom_type;
  const double *atom_charge, *atom_mass;
  const int *sp_natoms, *sp_atom_off, *sp_coul_cbmc;
  int ntypes, nspecies, natoms_total;
};

// Ewald view.
// k vectors per segment of the move chains: 2354 vectors make 574 segments of
// five (82 % filled), about one per lane of eleven waves; four make 723.  us a
// move with 3 / 4 / 5 / 6 / 8: 512 waters and 2354 vectors 13.1 / 13.4 / 12.0 /
// 13.5 / 16.0, 1080 waters 23.7 / 23.2 / 23.2 / 24.7 / 28.0, 27 waters 7.6 / 7.6 /
// 7.7 / 8.2 / 10.7.  Boxes of many vectors take several rounds of segments
// either way and would gain from short ones: 17700 vectors 60 / 66 / 72 / 85 /
// 105, 56500 vectors 215 / 235 / 267 / 305 / 380.
constexpr int kKSeg = 5;

struct EwaldDev {
  int nvecs, nrows;
  const double *hx, *hy, *hz, *cn;
  double *cs, *sn, *cmol, *smol;
  double *cs_new, *sn_new, *cm_new, *sm_new;
  const int4 *rows;      // (nx, nz, ny0, +-count): a run of consecutive ny from ny0
  const int *row_k0;     // first traversal position of each row
  const int *kperm;      // k index of each traversal position
  const int4 *segs;      // runs of up to kKSeg vectors along nx: (k0 | len << 20, nx, ny, nz)
  int nsegs;
  int tx, ty, tz;        // powers of a site's unit phases per axis
};

struct WidomArgs {
  int64_t n_ins;
  uint64_t seed;
  int species, natoms, spa0, charged;
  double beta, e_const;
  double ref[kMaxWidomSites * 3];   // site offsets from the COM (reference geometry)
  double q[kMaxWidomSites];
  double mass[kMaxWidomSites];
  int type[kMaxWidomSites];         // atom type of each site (-1: none)
  int cutoff_only;                  // every pair term needs r <= rc_pair
  double rc_pair, rc_pair2;
  const double *place;              // explicit coordinates [n_ins][natoms][3] or null
};

__host__ __device__ inline double rint_away(double x) { return round(x); }

// Sum over the wave's 64 lanes, uniform, in a fixed order: row shifts within
// 16 lanes, then the row broadcasts, all on the vector unit's data-parallel
// moves (a step of about 20 cycles, against some 130 for a shuffle through
// the LDS hardware).  Every lane of the wave must be active.
template <int CTRL, int ROWS>
__device__ inline double dpp_add(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWS, 0xf, false);
  return v + __hiloint2double(hi, lo);
}
__device__ inline double wave_total(double v) {
  v = dpp_add<0x111, 0xf>(v);  // row_shr:1
  v = dpp_add<0x112, 0xf>(v);  // row_shr:2
  v = dpp_add<0x114, 0xf>(v);  // row_shr:4
  v = dpp_add<0x118, 0xf>(v);  // row_shr:8: lane 15 of each row has its sum
  v = dpp_add<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
  v = dpp_add<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), 63),
                          __builtin_amdgcn_readlane(__double2loint(v), 63));
}

// Zeroes the records [from, to) of one array (null: none), by the lanes of one
// wave: what a chain that stops leaves unwritten.
template <typename T>
__device__ inline void record_rest(T *p, int64_t from, int64_t to) {
  if (p)
    for (int64_t k = from + (threadIdx.x & 63); k < to; k += 64) p[k] = T(0);
}

// ------------------------------------------------------------- geometry
__device__ inline void min_image(const BoxDev &b, double &dx, double &dy, double &dz) {
  // minimum_image_separation.f90:35-112: cubic boxes shift by one box length
  // at most; other boxes round fractional coordinates.
  if (b.cubic) {
    if (dx > b.hL[0]) dx -= b.L[0]; else if (dx < -b.hL[0]) dx += b.L[0];
    if (dy > b.hL[1]) dy -= b.L[1]; else if (dy < -b.hL[1]) dy += b.L[1];
    if (dz > b.hL[2]) dz -= b.L[2]; else if (dz < -b.hL[2]) dz += b.L[2];
  } else {
    double sx = b.Li[0] * dx + b.Li[3] * dy + b.Li[6] * dz;
    double sy = b.Li[1] * dx + b.Li[4] * dy + b.Li[7] * dz;
    double sz = b.Li[2] * dx + b.Li[5] * dy + b.Li[8] * dz;
    sx -= rint_away(sx);
    sy -= rint_away(sy);
    sz -= rint_away(sz);
    dx = b.Lc[0] * sx + b.Lc[3] * sy + b.Lc[6] * sz;
    dy = b.Lc[1] * sx + b.Lc[4] * sy + b.Lc[7] * sz;
    dz = b.Lc[2] * sx + b.Lc[5] * sy + b.Lc[8] * sz;
  }
}

// Check_MoleculePair_Cutoff (energy_routines.f90:3027-3088).
__device__ inline bool molpair_in_range(const BoxDev &b, bool cbmc, double4 ci, double4 cj) {
  if (b.vdw_minimum) return true;
  double dx = ci.x - cj.x, dy = ci.y - cj.y, dz = ci.z - cj.z;
  min_image(b, dx, dy, dz);
  double rcom = sqrt(dx * dx + dy * dy + dz * dz);
  double rint = (cbmc ? b.rcut_cbmc : b.rcut_max) + ci.w + cj.w;
  return !(rcom > rint);
}

// Arithmetic of the two pair terms per precision mode: V for vdW, Q for the
// real-space q-q term, M for the operation sequence.
//   FP64:  the reference's operations in double (parity path).
//   Mixed: double arithmetic on FP32 hardware seeds (rcp, rsq) refined by one
//          Newton step, ~1e-14 relative per pair: plain FP32 pair terms lose
//          ~1e-7 per pair, which the cancellation of LJ s^12 - s^6 near
//          r = sigma and of the Coulomb sums amplifies to ~1e-5 of dE.
//   FP32:  single-precision pair terms on the hardware seeds.
// Pair geometry (minimum image, r^2, cutoff and overlap tests) is FP64 in
// every mode, so all modes see the same pair set.
struct PrecFP64 {
  using V = double;
  using Q = double;
  using M = MathRef;
};
struct PrecMixed {
  using V = double;
  using Q = double;
  using M = MathFast;
};
struct PrecFP32 {
  using V = float;
  using Q = float;
  using M = MathFast;
};

template <typename T>
__host__ __device__ inline const PairConst<T> &pconst(const PairConst<double> &cd, const PairConst<float> &cf);
template <>
__host__ __device__ inline const PairConst<double> &pconst<double>(const PairConst<double> &cd,
                                                                   const PairConst<float> &) {
  return cd;
}
template <>
__host__ __device__ inline const PairConst<float> &pconst<float>(const PairConst<double> &,
                                                                 const PairConst<float> &cf) {
  return cf;
}

// One probe molecule (sites px/py/pz with species-atom ids pspa) against
// stored molecule j: Compute_MoleculePair_Energy (energy_routines.f90:1589-1730).
// Accumulates vdW and q-q in FP64; returns true on overlap r^2 < rcut_low^2.
// Cutoff and overlap tests use the FP64 r^2 in every mode, so all modes see
// the same pair set.  With ecbmc the same pass also accumulates the
// CBMC-cutoff sum.
// Estimate_MoleculePair_Energy (energy_routines.f90:1528-1587): the CBMC
// energy of the probe against molecule j from the pair table, added to ev
// (the reference returns vdW and q-q together as the vdW term).  Each entry
// is vdW(bin) + f2(bin) (q_i kChargeFactor) q_j, the sum
// Create_Atompair_Nrg_table forms (atompair_nrg_table_routines.f90:244-256);
// the bin is INT((r^2 - rsq_shifter) / rsq_step), 1-based.  Unfused
// operations keep r^2 and the entry the reference's own roundings.  Returns
// true on overlap (shifted r^2 below one step: r^2 < rcut_low^2).
__device__ inline bool molpair_estimate(const BoxDev &b, const TopoDev &tp, int ni, const double *px,
                                        const double *py, const double *pz, const int *pspa, int j,
                                        double &ev) {
  const int sj = b.species[j], fj = b.first[j];
  const int nj = tp.sp_natoms[sj], oj = tp.sp_atom_off[sj];
  const int nt = tp.ntypes, res = b.apt_res;
  const double *f2 = b.apt + (size_t)nt * nt * res;
  double mp = 0.0;
  for (int ia = 0; ia < ni; ++ia) {
    const int ti = tp.atom_type[pspa[ia]];
    const double qf = __dmul_rn(tp.atom_charge[pspa[ia]], kChargeFactor);
    for (int ja = 0; ja < nj; ++ja) {
      double dx = px[ia] - b.x[fj + ja], dy = py[ia] - b.y[fj + ja], dz = pz[ia] - b.z[fj + ja];
      min_image(b, dx, dy, dz);
      const double r2s =
          __dsub_rn(__dadd_rn(__dadd_rn(__dmul_rn(dx, dx), __dmul_rn(dy, dy)), __dmul_rn(dz, dz)), b.apt_shift);
      if (!(r2s < b.apt_rcs)) continue;
      if (r2s < b.apt_step) return true;
      // 1 <= r2s / step < res + 1 here; the clamp guards the last edge
      const int bin = max(0, min(res, (int)(r2s / b.apt_step)) - 1);
      const int tj = tp.atom_type[oj + ja];
      const double v = (ti >= 0 && tj >= 0) ? b.apt[(size_t)(tj * nt + ti) * res + bin] : 0.0;
      const double e = __dadd_rn(v, __dmul_rn(f2[bin], __dmul_rn(qf, tp.atom_charge[oj + ja])));
      mp = __dadd_rn(mp, e);
    }
  }
  ev += mp;
  return false;
}

template <typename P>
__device__ inline bool molpair_energy(const BoxDev &b, const TopoDev &tp, const PairConst<double> &cd,
                                      const PairConst<float> &cf, bool cbmc, bool coul_cbmc, int ni,
                                      const double *px, const double *py, const double *pz,
                                      const int *pspa, int j, double &ev, double &eq, double *ecbmc) {
  // CBMC trials with the pair table (Compute_Molecule_Nonbond_Inter_Energy,
  // energy_routines.f90:1180-1182)
  if (cbmc && b.apt_res > 0 && !ecbmc) return molpair_estimate(b, tp, ni, px, py, pz, pspa, j, ev);
  using TV = typename P::V;
  using TQ = typename P::Q;
  const PairConst<TV> &cv = pconst<TV>(cd, cf);
  const PairConst<TQ> &cq = pconst<TQ>(cd, cf);
  const int sj = b.species[j], fj = b.first[j];
  const int nj = tp.sp_natoms[sj], oj = tp.sp_atom_off[sj];
  for (int ia = 0; ia < ni; ++ia) {
    const int ti = tp.atom_type[pspa[ia]];
    const double qi = tp.atom_charge[pspa[ia]];
    for (int ja = 0; ja < nj; ++ja) {
      double dx = px[ia] - b.x[fj + ja], dy = py[ia] - b.y[fj + ja], dz = pz[ia] - b.z[fj + ja];
      min_image(b, dx, dy, dz);
      const double r2d = dx * dx + dy * dy + dz * dz;
      if (r2d < cd.rc_low2) return true;
      bool gv, gq;
      pair_cutoff(cd, cbmc, r2d, gv, gq);
      if (cbmc && !coul_cbmc) gq = false;
      // the CBMC pass's own tests (Check_AtomPair_Cutoff with cbmc_flag)
      bool gvc = false, gqc = false;
      if (ecbmc) {
        pair_cutoff(cd, true, r2d, gvc, gqc);
        if (!coul_cbmc) gqc = false;
      }
      if (!(gv || gq || gvc || gqc)) continue;
      const int tj = tp.atom_type[oj + ja];
      TV e_v = (TV)0;
      TQ e_q = (TQ)0;
      if (ti >= 0 && tj >= 0 && (gv || gvc)) {
        const int k = ti * tp.ntypes + tj;
        e_v = vdw_inter<TV, typename P::M>(cv, (TV)r2d, (TV)tp.eps[k], (TV)tp.sig[k], (TV)tp.mn[k], (TV)tp.mm[k]);
      }
      const double qj = tp.atom_charge[oj + ja];
      const bool any_q = cd.q_style != CASS_Q_NONE && qi != 0.0 && qj != 0.0;
      if (any_q && (gq || gqc)) e_q = qq_inter<TQ, typename P::M>(cq, (TQ)r2d, (TQ)(qi * qj));
      if (gv) ev += (double)e_v;
      if (gq) eq += (double)e_q;
      if (gvc || gqc) {
        const bool cv = ti >= 0 && tj >= 0 && cd.vdw_style != CASS_VDW_NONE && gvc;
        *ecbmc += (cv ? (double)e_v : 0.0) + ((any_q && gqc) ? (double)e_q : 0.0);
      }
    }
  }
  return false;
}

// Get_COM and Compute_Max_Com_Distance (get_com.f90:45-121, 220-295);
// returns (xcom, ycom, zcom, max_dcom).
__host__ __device__ inline double4 molecule_com(const TopoDev &tp, int off, int n, const double *x,
                                                const double *y, const double *z) {
  double tm = 0.0, cx = 0.0, cy = 0.0, cz = 0.0;
  for (int a = 0; a < n; ++a) {
    const double m = tp.atom_mass[off + a];
    tm = tm + m;
    cx = cx + m * x[a];
    cy = cy + m * y[a];
    cz = cz + m * z[a];
  }
  cx = cx / tm;
  cy = cy / tm;
  cz = cz / tm;
  double dmax = 0.0;
  for (int a = 0; a < n; ++a) {
    const double dx = x[a] - cx, dy = y[a] - cy, dz = z[a] - cz;
    const double r2 = dx * dx + dy * dy + dz * dz;
    dmax = r2 > dmax ? r2 : dmax;
  }
  return make_double4(cx, cy, cz, sqrt(dmax));
}

// Counter-based uniform draws for batched placements (splitmix64 finaliser
// over (seed, insertion, draw)); u in [0, 1) with 53 random bits.
__host__ __device__ inline uint64_t mix64(uint64_t z) {
  z += 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}
__host__ __device__ inline double counter_uniform(uint64_t seed, uint64_t i, uint32_t d) {
  const uint64_t h = mix64(mix64(seed ^ (i * 0xD1B54A32D192ED03ull)) + d);
  return (double)(h >> 11) * (1.0 / 9007199254740992.0);
}

// Uniform COM in the box and uniform orientation (unit quaternion from three
// uniforms, Shoemake 1992) for insertion i.
__host__ __device__ inline void place_probe(const WidomArgs &w, const BoxDev &b, uint64_t i, double *px,
                                            double *py, double *pz) {
  const double u0 = counter_uniform(w.seed, i, 0), u1 = counter_uniform(w.seed, i, 1);
  const double u2 = counter_uniform(w.seed, i, 2), u3 = counter_uniform(w.seed, i, 3);
  const double u4 = counter_uniform(w.seed, i, 4), u5 = counter_uniform(w.seed, i, 5);
  const double fx = u0 - 0.5, fy = u1 - 0.5, fz = u2 - 0.5;
  const double cx = b.Lc[0] * fx + b.Lc[3] * fy + b.Lc[6] * fz;
  const double cy = b.Lc[1] * fx + b.Lc[4] * fy + b.Lc[7] * fz;
  const double cz = b.Lc[2] * fx + b.Lc[5] * fy + b.Lc[8] * fz;
  const double twopi = 6.283185307179586;
  const double r1 = sqrt(1.0 - u3), r2 = sqrt(u3);
  const double qx = r1 * sin(twopi * u4), qy = r1 * cos(twopi * u4);
  const double qz = r2 * sin(twopi * u5), qw = r2 * cos(twopi * u5);
  const double R00 = 1 - 2 * (qy * qy + qz * qz), R01 = 2 * (qx * qy - qz * qw), R02 = 2 * (qx * qz + qy * qw);
  const double R10 = 2 * (qx * qy + qz * qw), R11 = 1 - 2 * (qx * qx + qz * qz), R12 = 2 * (qy * qz - qx * qw);
  const double R20 = 2 * (qx * qz - qy * qw), R21 = 2 * (qy * qz + qx * qw), R22 = 1 - 2 * (qx * qx + qy * qy);
  for (int a = 0; a < w.natoms; ++a) {
    const double rx = w.ref[3 * a], ry = w.ref[3 * a + 1], rz = w.ref[3 * a + 2];
    px[a] = R00 * rx + R01 * ry + R02 * rz + cx;
    py[a] = R10 * rx + R11 * ry + R12 * rz + cy;
    pz[a] = R20 * rx + R21 * ry + R22 * rz + cz;
  }
}

// One box of a batched total-energy recompute (cass_total_energy_batch):
// its views, its pair blocks per molecule (nblk) and k blocks (kblk), and
// where its partials start.
struct RecomputeBox {
  BoxDev b;
  PairConst<double> cd;
  PairConst<float> cf;
  EwaldDev ew;
  int kblk, kparts, kdirect;  // k blocks; workgroups per molecule of the two ways
  int64_t part_off, kpart_off;
};

struct cplx {
  double re, im;
};
__host__ __device__ inline cplx cmul(cplx a, cplx b) {
  return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}
__host__ __device__ inline cplx cpow_int(cplx e, int n) {
  cplx base = n < 0 ? cplx{e.re, -e.im} : e;  // |e| = 1: e^-1 = conj(e)
  int k = n < 0 ? -n : n;
  cplx r = {1.0, 0.0};
  while (k) {
    if (k & 1) r = cmul(r, base);
    base = cmul(base, base);
    k >>= 1;
  }
  return r;
}

constexpr int kPairMols = 4;   // molecules per workgroup of the total pair sums, one wave each
constexpr int kBoxVecs = 64;   // k vectors per workgroup of the box sums,
constexpr int kBoxShare = 16;  // where a box has at least this many molecules, else kMaxBlock
inline int box_blocks(int nvecs, int nmols) {
  const int vecs = nmols >= kBoxShare ? kBoxVecs : kMaxBlock;
  return nvecs > vecs ? (nvecs + vecs - 1) / vecs : 1;
}
constexpr int kEwTab = 1024;   // phase powers held per molecule
// Whether a molecule of n sites takes a sine and cosine per site and k vector
// in the total energy's structure factors: its powers exceed the table, or the
// box has so few molecules that building the tables is what a call waits for
// (one water and 56000 vectors: the call takes 30.3 us by the table, 28.3
// without; four: 31.3 and 32.1).
__host__ __device__ inline bool ewald_direct(const EwaldDev &ew, int nmols, int n) {
  return nmols <= 2 || n * (ew.tx + ew.ty + ew.tz) > kEwTab;
}

// kernels (kernels.hip)
template <typename P>
__global__ void k_trials(BoxDev b, TopoDev tp, PairConst<double> cd, PairConst<float> cf, int species, int ni,
                         const double *txyz, int exclude, int cbmc, double *part, int *part_ov);
__global__ void k_finalize_trials(const double *part, const int *part_ov, int nblk, int ntrial, double *out,
                                  int *out_ov);
__global__ void k_sum(const double *in, size_t n, int stride, int comp, double *out);
template <typename P>
__global__ void k_total_pairs(BoxDev b, TopoDev tp, PairConst<double> cd, PairConst<float> cf, double *part,
                              int *part_ov);
__global__ void k_ewald_mol(BoxDev b, TopoDev tp, EwaldDev ew);
__global__ void k_ewald_direct(BoxDev b, TopoDev tp, EwaldDev ew);
__global__ void k_ewald_box(BoxDev b, EwaldDev ew, double *part);
template <typename P>
__global__ void k_total_pairs_multi(const RecomputeBox *boxes, TopoDev tp, const int2 *items, double *part,
                                    int *part_ov);
__global__ void k_ewald_mol_multi(const RecomputeBox *boxes, TopoDev tp, const int2 *items);
__global__ void k_ewald_direct_multi(const RecomputeBox *boxes, TopoDev tp, const int2 *items);
__global__ void k_ewald_box_multi(const RecomputeBox *boxes, const int2 *items, double *kpart);
__global__ void k_sum_multi(const RecomputeBox *boxes, const double *kpart, double *out);
__global__ void k_ewald_move(TopoDev tp, EwaldDev ew, int m, int species, int flag, int n, const double *nxyz,
                             double *part);
__global__ void k_ewald_commit(EwaldDev ew, int m);
__global__ void k_ewald_widom(TopoDev tp, EwaldDev ew, int species, int n, const double *txyz, double *part);
__global__ void k_sum_widom(const double *part, const int64_t *part_ov, int n, double *out, int64_t *out_ov);

}  // namespace cass
