// nvtdev.hip -- the NVT move loop of cass_nvt_run resident on the device.
//
// nvtmc_driver.f90:94-152 choosing between Translate (move_translate.f90:23-360)
// and Rotate (move_rotate.f90:23-520), with the same random-number draws
// (random_generators.f90:51-122), energy bookkeeping and accept_or_reject
// (accept_or_reject.f90:22-65) as the host-driven loop in nvt.cpp.  One
// workgroup of 512 threads runs the moves in sequence: thread 0 draws the
// move and builds the trial coordinates, all threads share the molecule-pair
// energies (old and new placements side by side) and the k vectors of the
// reciprocal update, and an accepted move is committed in device memory.  No
// host round trip per move: the host launches chunks of moves and reads the
// RNG state, energies and records back at the end.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <limits>
#include <type_traits>
#include <vector>

#include "engine.h"
#include "kernels.h"

namespace cass {

// 512 threads: two waves per SIMD leave 256 VGPRs per lane (1024 threads cap
// them at 128, and the move's state then spills to scratch)
constexpr int kNvtBlock = 512;
constexpr int kNvtWaves = kNvtBlock / 64;

struct NvtChainArgs {
  BoxDev b;
  TopoDev tp;
  PairConst<double> cd;
  PairConst<float> cf;
  EwaldDev ew;
  double *x, *y, *z;  // the box's site coordinates (the memory of b.x, b.y, b.z)
  double4 *comd;      // the box's (COM, max_dcom) (the memory of b.comd)
  const int *mols;    // mobile molecules in locate order
  int nm, species, n, spa0, charged, linear, coul_cbmc;
  int nj_uniform;  // the common site count of every molecule of the box, or 0
  double prob_translate, max_disp, max_rot, beta;
  int64_t nsteps, step0;  // moves of this launch; index of its first move
  int64_t *rng;           // 5 words, in/out
  double *en;             // total, inter, inter_vdw, inter_q, reciprocal; in/out
  uint8_t *kind, *accepted;  // records per move (index step0 + s), or null
  double *energy, *ln_pacc;
  int64_t *rng_state;
  int *status;  // set to 1 when a molecule overlaps before its move
  double *ctrav, *strav;  // molecule sums in k-traversal order (nvecs each)
  // the box held in LDS for the whole chain (offsets in bytes)
  int nsite, natoms_total, nspecies, ntypes;
  int o_x, o_y, o_z, o_comd, o_first, o_spec, o_live, o_atype, o_acharge, o_spn, o_spo, o_pt, o_pq, o_prow,
      o_mols, o_ent, o_eoff;
};

// One site pair of Compute_MoleculePair_Energy (energy_routines.f90:1589-1730):
// site ia of the moving molecule (px/py/pz, type pt, charge pq) against site
// (x, y, z, type tj, charge qj) of another molecule, full cutoffs, with the
// reference's FP64 operations (the arithmetic of molpair_energy<PrecFP64>);
// prow[ia * ntypes + tj] holds (eps, sigma, n, m) of the pair's types.
// Returns true on overlap r^2 < rcut_low^2, else adds the pair's terms.
// PM: 0 any style with the reference's FP64 operations (vdw_inter,
// qq_inter); 1 the common styles (LJ cut / cut_tail / cut_shift or none with
// Ewald, cut or no Coulomb), whose cutoff tests and pair terms are
// pair_cutoff, lj_cut, ewald_real and coul_cut directly (the branches
// vdw_inter and qq_inter take for them), FP64 operations; 2 the common
// styles in the mixed mode (hardware rcp/rsq seeds refined by Newton steps).
template <int PM>
__device__ inline bool nvt_pair(const BoxDev &b, const PairConst<double> &cd, double px, double py, double pz,
                                int ti, double qi, const double4 *prow_i, double x, double y, double z, int tj,
                                double qj, double &ev, double &eq) {
  double dx = px - x, dy = py - y, dz = pz - z;
  min_image(b, dx, dy, dz);
  const double r2d = dx * dx + dy * dy + dz * dz;
  if (r2d < cd.rc_low2) return true;
  bool gv, gq;
  constexpr bool COMMON = PM > 0;
  using M = typename std::conditional<PM == 2, MathFast, MathRef>::type;
  if (COMMON) {
    gv = cd.vdw_style == CASS_VDW_LJ && r2d <= cd.rc_vdw2;
    gq = cd.q_style != CASS_Q_NONE && r2d <= cd.rc_coul2;
  } else {
    pair_cutoff(cd, false, r2d, gv, gq);
  }
  if (!(gv || gq)) return false;
  double e_v = 0.0, e_q = 0.0;
  if (ti >= 0 && tj >= 0 && gv) {
    const double4 p = prow_i[tj];
    e_v = COMMON ? lj_cut<double, M>(cd, r2d, p.x, p.y) : vdw_inter<double, MathRef>(cd, r2d, p.x, p.y, p.z, p.w);
  }
  const bool any_q = cd.q_style != CASS_Q_NONE && qi != 0.0 && qj != 0.0;
  if (any_q && gq) {
    if (COMMON)
      e_q = cd.q_style == CASS_Q_EWALD ? ewald_real<double, M>(cd, r2d, qi * qj) : coul_cut<double, M>(r2d, qi * qj);
    else
      e_q = qq_inter<double, MathRef>(cd, r2d, qi * qj);
  }
  if (gv) ev += e_v;
  if (gq) eq += e_q;
  return false;
}

// The centre prefilter of Check_MoleculePair_Cutoff (energy_routines.f90:
// 3027-3088) on squared distances.  The reference compares the square root;
// the two can differ only at the prefilter distance itself, where every site
// pair lies beyond the cutoff and beyond rcut_low, so the energies and the
// overlap test do not depend on the choice.
__device__ inline bool nvt_in_range(const BoxDev &b, double4 ci, double4 cj) {
  if (b.vdw_minimum) return true;
  double dx = ci.x - cj.x, dy = ci.y - cj.y, dz = ci.z - cj.z;
  min_image(b, dx, dy, dz);
  const double rint = b.rcut_max + ci.w + cj.w;
  return dx * dx + dy * dy + dz * dz <= rint * rint;
}

// Exclusive workgroup scan of two counts (fixed order); also returns the
// totals.  sc/st: LDS scratch of kNvtWaves ints each.
__device__ inline void nvt_scan2(int c, int t, int &cpre, int &tpre, int &ctot, int &ttot, int *sc, int *st) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  int ci = c, ti = t;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int cu = __shfl_up(ci, o, 64), tu = __shfl_up(ti, o, 64);
    if (lane >= o) {
      ci += cu;
      ti += tu;
    }
  }
  if (lane == 63) {
    sc[wid] = ci;
    st[wid] = ti;
  }
  __syncthreads();
  int cw = 0, tw = 0, ca = 0, ta = 0;
  for (int w = 0; w < kNvtWaves; ++w) {
    if (w < wid) {
      cw += sc[w];
      tw += st[w];
    }
    ca += sc[w];
    ta += st[w];
  }
  cpre = cw + ci - c;
  tpre = tw + ti - t;
  ctot = ca;
  ttot = ta;
  __syncthreads();
}

__device__ inline int64_t nvt_lsl(int64_t v, int k) { return (int64_t)((uint64_t)v << k); }
__device__ inline int64_t nvt_lsr(int64_t v, int k) { return (int64_t)((uint64_t)v >> k); }

// rranf (random_generators.f90:51-122): five-component LFSR, u in (0, 1)
__device__ inline double nvt_uniform(int64_t *s) {
  int64_t b;
  b = nvt_lsr(nvt_lsl(s[0], 1) ^ s[0], 53);
  s[0] = nvt_lsl(s[0] & -2, 10) ^ b;
  b = nvt_lsr(nvt_lsl(s[1], 24) ^ s[1], 50);
  s[1] = nvt_lsl(s[1] & -512, 5) ^ b;
  b = nvt_lsr(nvt_lsl(s[2], 3) ^ s[2], 23);
  s[2] = nvt_lsl(s[2] & -4096, 29) ^ b;
  b = nvt_lsr(nvt_lsl(s[3], 5) ^ s[3], 24);
  s[3] = nvt_lsl(s[3] & -131072, 23) ^ b;
  b = nvt_lsr(nvt_lsl(s[4], 3) ^ s[4], 33);
  s[4] = nvt_lsl(s[4] & -8388608, 8) ^ b;
  return (double)(s[0] ^ s[1] ^ s[2] ^ s[3] ^ s[4]) * 5.4210108624275221E-20 + 0.5;
}

__device__ inline double nvt_wave_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  return v;
}

__device__ inline int nvt_wave_or(int v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v |= __shfl_down(v, o, 64);
  return v;
}

// Workgroup sum of NV doubles and an OR of flags in a fixed order (waves,
// then the waves in index order); every thread receives the result.
template <int NV>
__device__ inline void nvt_reduce(double (&v)[NV], int &flag, double (*sh)[kNvtWaves], int *shf, double *res,
                                  int *resf) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < NV; ++k) v[k] = nvt_wave_sum(v[k]);
  flag = nvt_wave_or(flag);
  if (lane == 0) {
#pragma unroll
    for (int k = 0; k < NV; ++k) sh[k][wid] = v[k];
    shf[wid] = flag;
  }
  __syncthreads();
  if (wid == 0) {
    // the wave partials on the first kNvtWaves lanes, summed by a fixed
    // shuffle tree
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      double s = lane < kNvtWaves ? sh[k][lane] : 0.0;
#pragma unroll
      for (int o = kNvtWaves / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
      if (lane == 0) res[k] = s;
    }
    int f = lane < kNvtWaves ? shf[lane] : 0;
#pragma unroll
    for (int o = kNvtWaves / 2; o > 0; o >>= 1) f |= __shfl_xor(f, o, 64);
    if (lane == 0) *resf = f;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NV; ++k) v[k] = res[k];
  flag = *resf;
}

// One axis of Fold_Molecule for a cubic box: the centre c and the sites q
// move by one box length when c leaves [-h, h].
__device__ inline void nvt_fold(double &c, double *q, int n, double L, double h) {
  if (c > h) {
    c = c - L;
    for (int i = 0; i < n; ++i) q[i] = q[i] - L;
  } else if (c < -h) {
    c = c + L;
    for (int i = 0; i < n; ++i) q[i] = q[i] + L;
  }
}

template <int PM, int NSE>
__device__ __forceinline__ void nvt_chain_run(const NvtChainArgs &a) {
  __shared__ double ox[kMaxSites], oy[kMaxSites], oz[kMaxSites];
  __shared__ double qx[kMaxSites], qy[kMaxSites], qz[kMaxSites];
  __shared__ int pspa[kMaxSites];
  __shared__ double4 com_old, com_new, cn_fold;
  __shared__ int s_m, s_rot, s_acc;
  __shared__ double sh[4][kNvtWaves];
  __shared__ int shf[kNvtWaves];
  __shared__ int scan_c[kNvtWaves], scan_t[kNvtWaves];
  __shared__ double eph[6 * kMaxSites];  // (cos, sin) of 2 pi s_x, s_y, s_z per new site
  __shared__ double res[4];
  __shared__ int resf;
  extern __shared__ char lds[];
  double *lx = (double *)(lds + a.o_x), *ly = (double *)(lds + a.o_y), *lz = (double *)(lds + a.o_z);
  double4 *lcomd = (double4 *)(lds + a.o_comd);
  int *lfirst = (int *)(lds + a.o_first), *lspec = (int *)(lds + a.o_spec), *llive = (int *)(lds + a.o_live);
  int *atype = (int *)(lds + a.o_atype);
  double *acharge = (double *)(lds + a.o_acharge);
  int *spn = (int *)(lds + a.o_spn), *spo = (int *)(lds + a.o_spo);
  int *pt = (int *)(lds + a.o_pt);
  double *pq = (double *)(lds + a.o_pq);
  double4 *prow = (double4 *)(lds + a.o_prow);
  int *lmols = (int *)(lds + a.o_mols);
  int *ent_j = (int *)(lds + a.o_ent), *ent_off = (int *)(lds + a.o_eoff);
  const int tid = threadIdx.x;
  const int n = a.n, K = a.ew.nvecs, nmols = a.b.nmols;
  for (int i = tid; i < a.nsite; i += kNvtBlock) {
    lx[i] = a.x[i];
    ly[i] = a.y[i];
    lz[i] = a.z[i];
  }
  for (int i = tid; i < nmols; i += kNvtBlock) {
    lcomd[i] = a.comd[i];
    lfirst[i] = a.b.first[i];
    lspec[i] = a.b.species[i];
    llive[i] = a.b.live[i];
  }
  for (int i = tid; i < a.natoms_total; i += kNvtBlock) {
    atype[i] = a.tp.atom_type[i];
    acharge[i] = a.tp.atom_charge[i];
  }
  for (int i = tid; i < a.nspecies; i += kNvtBlock) {
    spn[i] = a.tp.sp_natoms[i];
    spo[i] = a.tp.sp_atom_off[i];
  }
  for (int i = tid; i < a.nm; i += kNvtBlock) lmols[i] = a.mols[i];
  for (int i = tid; i < n * a.ntypes; i += kNvtBlock) {
    const int ia = i / a.ntypes, tj = i - ia * a.ntypes;
    const int ti = a.tp.atom_type[a.spa0 + ia];
    const int k = (ti < 0 ? 0 : ti) * a.ntypes + tj;
    prow[i] = make_double4(a.tp.eps[k], a.tp.sig[k], a.tp.mn[k], a.tp.mm[k]);
  }
  if (tid < n) {
    pspa[tid] = a.spa0 + tid;
    pt[tid] = a.tp.atom_type[a.spa0 + tid];
    pq[tid] = a.tp.atom_charge[a.spa0 + tid];
  }
  // RNG words and energies: used by thread 0 only, kept in LDS
  __shared__ int64_t rs[5];
  __shared__ double en[5];
  if (tid == 0) {
    for (int k = 0; k < 5; ++k) rs[k] = a.rng[k];
    for (int k = 0; k < 5; ++k) en[k] = a.en[k];
  }
  __syncthreads();
  for (int64_t st = 0; st < a.nsteps; ++st) {
    // --- the move (thread 0): draws in the order of nvtmc_driver / Translate / Rotate
    if (tid == 0) {
      const double rno = nvt_uniform(rs);
      const int rot = !(rno <= a.prob_translate);
      (void)nvt_uniform(rs);  // species pick (one mobile species)
      const int im = (int)(nvt_uniform(rs) * a.nm);
      const int m = lmols[im];
      const int f = lfirst[m];
      const double4 co = lcomd[m];
      double4 cn = co;
      for (int i = 0; i < n; ++i) {
        ox[i] = lx[f + i];
        oy[i] = ly[f + i];
        oz[i] = lz[f + i];
      }
      if (!rot) {
        const double dx = (2.0 * nvt_uniform(rs) - 1.0) * a.max_disp;
        const double dy = (2.0 * nvt_uniform(rs) - 1.0) * a.max_disp;
        const double dz = (2.0 * nvt_uniform(rs) - 1.0) * a.max_disp;
        for (int i = 0; i < n; ++i) {
          qx[i] = ox[i] + dx;
          qy[i] = oy[i] + dy;
          qz[i] = oz[i] + dz;
        }
        cn.x = co.x + dx;
        cn.y = co.y + dy;
        cn.z = co.z + dz;
        // Fold_Molecule (minimum_image_separation.f90:162-240), cubic boxes
        if (a.b.cubic) {
          nvt_fold(cn.x, qx, n, a.b.L[0], a.b.hL[0]);
          nvt_fold(cn.y, qy, n, a.b.L[1], a.b.hL[1]);
          nvt_fold(cn.z, qz, n, a.b.L[2], a.b.hL[2]);
        }
      } else {
        double r[9];
        if (a.linear) {
          // Rotate_Molecule_Eulerian (move_rotate.f90:468-520)
          const double th = acos(1.0 - 2.0 * nvt_uniform(rs));
          const double ph = (1.0 - 2.0 * nvt_uniform(rs)) * kPi;
          const double ps = (1.0 - 2.0 * nvt_uniform(rs)) * kPi;
          r[0] = cos(ps) * cos(ph) - cos(th) * sin(ph) * sin(ps);
          r[1] = cos(ps) * sin(ph) + cos(th) * cos(ph) * sin(ps);
          r[2] = sin(ps) * sin(th);
          r[3] = -sin(ps) * cos(ph) - cos(th) * sin(ph) * cos(ps);
          r[4] = -sin(ps) * sin(ph) + cos(th) * cos(ph) * cos(ps);
          r[5] = cos(ps) * sin(th);
          r[6] = sin(th) * sin(ph);
          r[7] = -sin(th) * cos(ph);
          r[8] = cos(th);
        } else {
          // Rotate_Molecule_Axis (move_rotate.f90:362-463)
          double p1 = 0.0, p2 = 0.0, p3 = 0.0;
          const int axis = (int)(3.0 * nvt_uniform(rs)) + 1;
          const double ang = (2.0 * nvt_uniform(rs) - 1.0) * a.max_rot;
          if (axis == 1)
            p1 = ang;
          else if (axis == 2)
            p2 = ang;
          else
            p3 = ang;
          // cos(0) = 1 and sin(0) = 0 exactly: only the drawn axis needs them
          const double ca = cos(ang), sa = sin(ang);
          const double c1 = axis == 1 ? ca : 1.0, c2 = axis == 2 ? ca : 1.0, c3 = axis == 3 ? ca : 1.0;
          const double s1 = axis == 1 ? sa : 0.0, s2 = axis == 2 ? sa : 0.0, s3 = axis == 3 ? sa : 0.0;
          (void)p1;
          (void)p2;
          (void)p3;
          r[0] = c1 * c3 - s1 * c2 * s3;
          r[1] = s1 * c3 + c1 * c2 * s3;
          r[2] = s2 * s3;
          r[3] = -c1 * s3 - s1 * c2 * c3;
          r[4] = -s1 * s3 + c1 * c2 * c3;
          r[5] = s2 * c3;
          r[6] = s1 * s2;
          r[7] = -c1 * s2;
          r[8] = c2;
        }
        for (int i = 0; i < n; ++i) {
          const double px = ox[i] - co.x, py = oy[i] - co.y, pz = oz[i] - co.z;
          qx[i] = (r[0] * px + r[1] * py + r[2] * pz) + co.x;
          qy[i] = (r[3] * px + r[4] * py + r[5] * pz) + co.y;
          qz[i] = (r[6] * px + r[7] * py + r[8] * pz) + co.z;
        }
      }
      s_m = m;
      s_rot = rot;
      cn_fold = cn;
    }
    __syncthreads();
    // the trial kernel's prefilter centres: Get_COM of each placement; and,
    // on a third wave, the unit phases exp(2 pi i s) of the new sites'
    // fractional coordinates for the reciprocal sums
    if (tid == 0) com_old = molecule_com(a.tp, a.spa0, n, ox, oy, oz);
    if (tid == 64) com_new = molecule_com(a.tp, a.spa0, n, qx, qy, qz);
    if (NSE > 0 && a.charged && tid >= 128 && tid < 128 + 3 * n) {
      const int t = tid - 128, i = t / 3, d = t - 3 * i;
      const double sd = a.b.Li[d] * qx[i] + a.b.Li[3 + d] * qy[i] + a.b.Li[6 + d] * qz[i];
      double sv, cv;
      sincos(kTwoPi * sd, &sv, &cv);
      eph[2 * t] = cv;
      eph[2 * t + 1] = sv;
    }
    __syncthreads();
    const int m = s_m;
    // --- inter energies of the old and the new placement (Compute_Molecule_Nonbond_Inter_Energy):
    // the molecules that pass the COM prefilter (Check_MoleculePair_Cutoff)
    // are listed in LDS, then every site pair of the list is one task
    int nent = 0, ntask = 0;
    for (int base = 0; base < 2 * nmols; base += kNvtBlock) {
      const int t = base + tid;
      int take = 0, tasks = 0, j = 0, which = 0;
      if (t < 2 * nmols) {
        which = t >= nmols ? 1 : 0;
        j = t - which * nmols;
        if (j != m && llive[j] && nvt_in_range(a.b, which ? com_new : com_old, lcomd[j])) {
          take = 1;
          tasks = n * spn[lspec[j]];
        }
      }
      int cpre, tpre, ctot, ttot;
      nvt_scan2(take, tasks, cpre, tpre, ctot, ttot, scan_c, scan_t);
      if (take) {
        ent_j[nent + cpre] = (j << 1) | which;
        ent_off[nent + cpre] = ntask + tpre;
      }
      nent += ctot;
      ntask += ttot;
    }
    if (tid == 0) ent_off[nent] = ntask;
    __syncthreads();
    double ev0 = 0.0, eq0 = 0.0, ev1 = 0.0, eq1 = 0.0;  // old / new placement
    int ov = 0;
    const int tpe = n * a.nj_uniform;  // tasks per listed molecule when all have nj_uniform sites
    for (int task = tid; task < ntask; task += kNvtBlock) {
      int lo;
      if (tpe > 0) {
        lo = task / tpe;
      } else {
        lo = 0;
        int hi = nent - 1;
        while (lo < hi) {
          const int mid = (lo + hi + 1) >> 1;
          if (ent_off[mid] <= task)
            lo = mid;
          else
            hi = mid - 1;
        }
      }
      const int code = ent_j[lo], which = code & 1, j = code >> 1;
      const int sj = lspec[j], nj = spn[sj], oj = spo[sj], fj = lfirst[j];
      const int local = task - ent_off[lo], ia = local / nj, ja = local - ia * nj;
      const double *px = which ? qx : ox, *py = which ? qy : oy, *pz = which ? qz : oz;
      double ev = 0.0, eq = 0.0;
      if (nvt_pair<PM>(a.b, a.cd, px[ia], py[ia], pz[ia], pt[ia], pq[ia], prow + ia * a.ntypes, lx[fj + ja], ly[fj + ja],
                   lz[fj + ja], atype[oj + ja], acharge[oj + ja], ev, eq)) {
        ov |= which ? 2 : 1;
      } else if (which) {
        ev1 += ev;
        eq1 += eq;
      } else {
        ev0 += ev;
        eq0 += eq;
      }
    }
    double v[4] = {ev0, eq0, ev1, eq1};
    nvt_reduce<4>(v, ov, sh, shf, res, &resf);
    if (ov & 1) {
      if (tid == 0) *a.status = 1;
      __syncthreads();
      break;
    }
    // --- reciprocal space: Update_System_Ewald_Reciprocal_Energy (staged)
    double erm = 0.0;
    const bool reach = !(ov & 2);
    if (reach && a.charged) {
      // from the unit phases computed beside the centres, each lane walks
      // k runs of the traversal (ny runs at fixed (nz, nx)) with the cosine
      // recurrence and stores the molecule sums at the run's k indices
      double e1[1] = {0.0};
      int f0 = 0;
      double *__restrict__ ctrav = a.ctrav, *__restrict__ strav = a.strav;
      const int *__restrict__ kperm = a.ew.kperm;
      const double *__restrict__ ecn = a.ew.cn;
      const double *__restrict__ ecs = a.ew.cs, *__restrict__ esn = a.ew.sn;
      const double *__restrict__ ecm = a.ew.cmol, *__restrict__ esm = a.ew.smol;
      double *__restrict__ cs_new = a.ew.cs_new, *__restrict__ sn_new = a.ew.sn_new;
      double *__restrict__ cm_new = a.ew.cm_new, *__restrict__ sm_new = a.ew.sm_new;
      if (NSE > 0) {
        // molecule sums along the runs, in traversal order
        const int4 *__restrict__ rows = a.ew.rows;
        const int *__restrict__ row_k0 = a.ew.row_k0;
        for (int r = tid; r < a.ew.nrows; r += kNvtBlock) {
          const int4 row = rows[r];
          const int nx = row.x, nz = row.y, ny0 = row.z, cnt = row.w;
          const int dir = cnt > 0 ? 1 : -1, len = cnt > 0 ? cnt : -cnt;
          const int j0 = row_k0[r];
          cplx t[NSE > 0 ? NSE : 1], u[NSE > 0 ? NSE : 1];
          double c2[NSE > 0 ? NSE : 1];
#pragma unroll
          for (int i = 0; i < NSE; ++i) {
            const cplx ea = {eph[6 * i], eph[6 * i + 1]}, eb = {eph[6 * i + 2], eph[6 * i + 3]};
            const cplx ec = {eph[6 * i + 4], eph[6 * i + 5]};
            const cplx p = cmul(cmul(cpow_int(ea, nx), cpow_int(ec, nz)), cpow_int(eb, ny0));
            t[i] = {pq[i] * p.re, pq[i] * p.im};
            u[i] = cmul(t[i], {eb.re, -dir * eb.im});
            c2[i] = 2.0 * eb.re;
          }
          for (int kk = 0; kk < len; ++kk) {
            double c = t[0].re, sv = t[0].im;
#pragma unroll
            for (int i = 1; i < NSE; ++i) {
              c = c + t[i].re;
              sv = sv + t[i].im;
            }
#pragma unroll
            for (int i = 0; i < NSE; ++i) {
              const cplx tn = {fma(c2[i], t[i].re, -u[i].re), fma(c2[i], t[i].im, -u[i].im)};
              u[i] = t[i];
              t[i] = tn;
            }
            ctrav[j0 + kk] = c;
            strav[j0 + kk] = sv;
          }
        }
        __threadfence_block();
        __syncthreads();
        // the staged box sums and the energy, one k per lane
        for (int jt = tid; jt < K; jt += kNvtBlock) {
          const int k = kperm[jt];
          const size_t mk = (size_t)m * K + k;
          const double c = ctrav[jt], sv = strav[jt];
          const double c1 = ecs[k] + (c - ecm[mk]), s1 = esn[k] + (sv - esm[mk]);
          cs_new[k] = c1;
          sn_new[k] = s1;
          cm_new[k] = c;
          sm_new[k] = sv;
          e1[0] += ecn[k] * (c1 * c1 + s1 * s1);
        }
      } else {
        for (int k = tid; k < K; k += kNvtBlock) {
          const size_t mk = (size_t)m * K + k;
          const double hx = a.ew.hx[k], hy = a.ew.hy[k], hz = a.ew.hz[k];
          double c = 0.0, sv = 0.0;
          for (int i = 0; i < n; ++i) {
            const double hr = hx * qx[i] + hy * qy[i] + hz * qz[i];
            double sn, cs;
            sincos(hr, &sn, &cs);
            c = c + pq[i] * cs;
            sv = sv + pq[i] * sn;
          }
          const double c1 = a.ew.cs[k] + (c - a.ew.cmol[mk]), s1 = a.ew.sn[k] + (sv - a.ew.smol[mk]);
          a.ew.cs_new[k] = c1;
          a.ew.sn_new[k] = s1;
          a.ew.cm_new[k] = c;
          a.ew.sm_new[k] = sv;
          e1[0] += a.ew.cn[k] * (c1 * c1 + s1 * s1);
        }
      }
      nvt_reduce<1>(e1, f0, sh, shf, res, &resf);
      erm = e1[0] * kChargeFactor;
    }
    // --- acceptance (thread 0)
    if (tid == 0) {
      double lnp = std::numeric_limits<double>::quiet_NaN();
      int acc = 0;
      if (reach) {
        double dE = 0.0;
        if (a.charged) dE = erm - en[4];
        if (!s_rot)
          dE = dE + (v[2] - v[0]) + (v[3] - v[1]);
        else
          dE = dE + v[2] - v[0] + v[3] - v[1];
        lnp = a.beta * dE;
        if (lnp <= 0.0) {
          acc = 1;
        } else if (lnp < kMaxKBT) {
          const double pacc = exp(-lnp);
          if (nvt_uniform(rs) <= pacc) acc = 1;
        }
        if (acc) {
          en[0] = en[0] + dE;
          en[1] = en[1] + dE;
          en[2] = en[2] + v[2] - v[0];
          en[3] = en[3] + v[3] - v[1];
          if (a.charged) en[4] = erm;
          // the stored centre: the folded one after a translation, Get_COM
          // after a rotation (move_rotate.f90:287); max_dcom unchanged
          double4 c = lcomd[m];
          if (!s_rot) {
            c.x = cn_fold.x;
            c.y = cn_fold.y;
            c.z = cn_fold.z;
          } else {
            // Get_COM of the rotated sites: the new placement's centre
            c.x = com_new.x;
            c.y = com_new.y;
            c.z = com_new.z;
          }
          lcomd[m] = c;
          a.comd[m] = c;
        }
      }
      s_acc = acc;
      const int64_t g = a.step0 + st;
      if (a.kind) a.kind[g] = (uint8_t)s_rot;
      if (a.accepted) a.accepted[g] = (uint8_t)acc;
      if (a.energy) a.energy[g] = en[0];
      if (a.ln_pacc) a.ln_pacc[g] = lnp;
      if (a.rng_state)
        for (int k = 0; k < 5; ++k) a.rng_state[5 * g + k] = rs[k];
    }
    __syncthreads();
    if (s_acc) {
      const int f = lfirst[m];
      if (tid < n) {
        lx[f + tid] = qx[tid];
        ly[f + tid] = qy[tid];
        lz[f + tid] = qz[tid];
        a.x[f + tid] = qx[tid];
        a.y[f + tid] = qy[tid];
        a.z[f + tid] = qz[tid];
      }
      if (a.charged)
        for (int k = tid; k < K; k += kNvtBlock) {
          const size_t mk = (size_t)m * K + k;
          a.ew.cs[k] = a.ew.cs_new[k];
          a.ew.sn[k] = a.ew.sn_new[k];
          a.ew.cmol[mk] = a.ew.cm_new[k];
          a.ew.smol[mk] = a.ew.sm_new[k];
        }
    }
    __threadfence_block();
    __syncthreads();
  }
  if (tid == 0) {
    for (int k = 0; k < 5; ++k) a.rng[k] = rs[k];
    for (int k = 0; k < 5; ++k) a.en[k] = en[k];
  }
}

// One chain per launch (the arguments in the kernel's argument segment).
template <int PM, int NSE>
__global__ void __launch_bounds__(kNvtBlock) k_nvt_chain(NvtChainArgs a) {
  nvt_chain_run<PM, NSE>(a);
}

// Independent chains of several boxes, one workgroup per box: replicas of a
// system, or boxes of different state points, each on its own generator.
template <int PM, int NSE>
__global__ void __launch_bounds__(kNvtBlock) k_nvt_chain_multi(const NvtChainArgs *__restrict__ args) {
  nvt_chain_run<PM, NSE>(args[blockIdx.x]);
}

}  // namespace cass

using namespace cass;

BoxDev cass_box_view(const cass_engine *e, const cass_box_state &b);  // engine.hip
extern "C" int cass_nvt_run(cass_engine *e, int32_t box, cass_rng *rng, const cass_nvt_options *opt,
                            int64_t nsteps, cass_energy *en, cass_nvt_record *rec);  // nvt.cpp
TopoDev cass_topo_view(const cass_engine *e);
EwaldDev cass_ewald_view(const cass_box_state &b);

namespace {

// One chain's launch state: its arguments, LDS size and kernel selection,
// and where its generator, energies, mobile list and records stand in the
// batch's buffers.
struct NvtLaunch {
  NvtChainArgs a;
  size_t lds = 0;
  int pm = 0, nse = 0;
  bool host_loop = false;  // the box's copy exceeds the LDS: the host-driven loop runs it
  int box = -1;
  cass_rng *rng = nullptr;
  const cass_nvt_options *opt = nullptr;
  cass_energy *en = nullptr;
  cass_nvt_record *rec = nullptr;
  bool charged = false;
  std::vector<int> mols;  // locate order of the mobile species
  size_t o_state = 0, o_kind = 0, o_acc = 0, o_energy = 0, o_lnp = 0, o_rs = 0, o_mols = 0;
};

typedef void (*nvt_kernel_t)(NvtChainArgs);
typedef void (*nvt_multi_kernel_t)(const NvtChainArgs *);

nvt_kernel_t nvt_kernel(int pm, int nse) {
  static nvt_kernel_t const kt[3][5] = {
      {k_nvt_chain<0, 0>, k_nvt_chain<0, 1>, k_nvt_chain<0, 2>, k_nvt_chain<0, 3>, k_nvt_chain<0, 4>},
      {k_nvt_chain<1, 0>, k_nvt_chain<1, 1>, k_nvt_chain<1, 2>, k_nvt_chain<1, 3>, k_nvt_chain<1, 4>},
      {k_nvt_chain<2, 0>, k_nvt_chain<2, 1>, k_nvt_chain<2, 2>, k_nvt_chain<2, 3>, k_nvt_chain<2, 4>}};
  return kt[pm][nse];
}

nvt_multi_kernel_t nvt_multi_kernel(int pm, int nse) {
  static nvt_multi_kernel_t const kt[3][5] = {
      {k_nvt_chain_multi<0, 0>, k_nvt_chain_multi<0, 1>, k_nvt_chain_multi<0, 2>, k_nvt_chain_multi<0, 3>,
       k_nvt_chain_multi<0, 4>},
      {k_nvt_chain_multi<1, 0>, k_nvt_chain_multi<1, 1>, k_nvt_chain_multi<1, 2>, k_nvt_chain_multi<1, 3>,
       k_nvt_chain_multi<1, 4>},
      {k_nvt_chain_multi<2, 0>, k_nvt_chain_multi<2, 1>, k_nvt_chain_multi<2, 2>, k_nvt_chain_multi<2, 3>,
       k_nvt_chain_multi<2, 4>}};
  return kt[pm][nse];
}

// Checks, the LDS layout of the box copy, the kernel choice and the arguments
// of one chain but for its buffers (nvt_buffers).  nsteps == 0 or a box
// beyond the LDS leaves L.a unset (host_loop / nothing to launch).
int nvt_prepare(cass_engine *e, int32_t box, cass_rng *rng, const cass_nvt_options *opt, int64_t nsteps,
                cass_energy *en, cass_nvt_record *rec, NvtLaunch &L) {
  if (!e || !rng || !opt || !en || nsteps < 0 || box < 0 || box >= (int)e->boxes.size()) return CASS_ERR_ARG;
  cass_box_state &b = e->boxes[box];
  L.box = box;
  L.rng = rng;
  L.opt = opt;
  L.en = en;
  L.rec = rec;
  const int sp = opt->species;
  if (sp < 0 || sp >= e->nspecies) return CASS_ERR_ARG;
  const int n = e->sp_natoms[sp];
  if (n > kMaxSites) return cass_fail(e, CASS_ERR_ARG, "molecule has more sites than the device chain holds");
  bool has_q = false;
  for (int a = 0; a < n; ++a) has_q = has_q || e->atom_charge[e->sp_atom_off[sp] + a] != 0.0;
  const bool charged = b.p.charge_style == CASS_Q_EWALD && has_q;
  L.charged = charged;
  if (charged && !b.ewald_ready) return cass_fail(e, CASS_ERR_STATE, "Ewald sums not set up");
  std::vector<int> &mols = L.mols;
  for (int m = 0; m < b.nmols; ++m)
    if (b.mol_species[m] == sp && b.live[m]) mols.push_back(m);
  const int nm = (int)mols.size();
  if (nm == 0) return cass_fail(e, CASS_ERR_STATE, "no molecules to move");
  if (nsteps == 0) return CASS_OK;
  HIP_TRY(e, hipSetDevice(e->device));
  // LDS layout of the box copy
  const int nsite = (int)(b.xyz_h.size() / 3), nt = std::max(e->ntypes, 1);
  size_t lds = 0;
  auto take = [&](size_t bytes) {
    const size_t o = lds;
    lds = (lds + bytes + 15) & ~(size_t)15;
    return (int)o;
  };
  NvtChainArgs &a = L.a;
  std::memset(&a, 0, sizeof(a));
  a.o_x = take(sizeof(double) * nsite);
  a.o_y = take(sizeof(double) * nsite);
  a.o_z = take(sizeof(double) * nsite);
  a.o_comd = take(sizeof(double4) * b.nmols);
  a.o_first = take(sizeof(int) * b.nmols);
  a.o_spec = take(sizeof(int) * b.nmols);
  a.o_live = take(sizeof(int) * b.nmols);
  a.o_atype = take(sizeof(int) * e->natoms_total);
  a.o_acharge = take(sizeof(double) * e->natoms_total);
  a.o_spn = take(sizeof(int) * e->nspecies);
  a.o_spo = take(sizeof(int) * e->nspecies);
  a.o_pt = take(sizeof(int) * n);
  a.o_pq = take(sizeof(double) * n);
  a.o_prow = take(sizeof(double4) * n * nt);
  a.o_mols = take(sizeof(int) * nm);
  a.o_ent = take(sizeof(int) * (2 * b.nmols + 1));
  a.o_eoff = take(sizeof(int) * (2 * b.nmols + 1));
  L.lds = lds;
  const bool common = (b.p.vdw_style == CASS_VDW_NONE ||
                       (b.p.vdw_style == CASS_VDW_LJ &&
                        (b.p.vdw_sum_style == CASS_SUM_CUT || b.p.vdw_sum_style == CASS_SUM_CUT_TAIL ||
                         b.p.vdw_sum_style == CASS_SUM_CUT_SHIFT))) &&
                      (b.p.charge_style == CASS_Q_NONE || b.p.charge_style == CASS_Q_EWALD ||
                       b.p.charge_style == CASS_Q_CUT);
  int lds_max = 0;
  HIP_TRY(e, hipDeviceGetAttribute(&lds_max, hipDeviceAttributeMaxSharedMemoryPerBlock, e->device));
  if (lds > (size_t)lds_max - 8192) {
    L.host_loop = true;
    return CASS_OK;
  }
  // the reciprocal sums of molecules up to 4 sites by phase recurrences
  // along the k runs, larger ones by sincos per k
  L.nse = (charged && n <= 4 && b.nrows > 0) ? n : 0;
  // the mixed and FP32 modes take the mixed pair arithmetic for the common
  // styles (FP64 accumulation, reciprocal space and acceptance in every mode)
  L.pm = common ? (e->prec == CASS_PREC_FP64 ? 1 : 2) : 0;
  a.b = cass_box_view(e, b);
  a.tp = cass_topo_view(e);
  a.cd = make_pair_const<double>(b.p, e->ntypes);
  a.cf = make_pair_const<float>(b.p, e->ntypes);
  a.ew = cass_ewald_view(b);
  if (!charged) a.ew.nvecs = 0;
  a.x = b.x;
  a.y = b.y;
  a.z = b.z;
  a.comd = b.comd;
  a.nm = nm;
  a.species = sp;
  a.n = n;
  a.spa0 = e->sp_atom_off[sp];
  a.charged = charged ? 1 : 0;
  a.linear = opt->linear;
  a.coul_cbmc = e->sp_coul_cbmc[sp];
  a.prob_translate = opt->prob_translate;
  a.max_disp = opt->max_disp;
  a.max_rot = opt->max_rot;
  a.beta = b.p.beta;
  a.nsite = nsite;
  a.nj_uniform = b.nmols > 0 ? e->sp_natoms[b.mol_species[0]] : 0;
  for (int mm = 0; mm < b.nmols; ++mm)
    if (e->sp_natoms[b.mol_species[mm]] != a.nj_uniform) a.nj_uniform = 0;
  a.natoms_total = e->natoms_total;
  a.nspecies = e->nspecies;
  a.ntypes = nt;
  return CASS_OK;
}

// The state of one chain in the batch's buffer.
struct NvtState {
  int64_t rng[5];
  double en[5];
  int status[2];
};

// The buffers of a batch, laid out over all its chains: first what comes back
// (states and records), then the mobile lists and argument tables, then the
// molecule sums.  One copy in, one copy out: with a set of copies per chain
// the calls themselves outlasted the chains.
struct NvtBuffers {
  char *dev = nullptr;
  size_t back = 0, in = 0;  // bytes copied back; bytes of back + lists + arguments
  size_t o_args = 0;
  std::vector<char> host;   // the first `in` bytes
};

int nvt_buffers(cass_engine *e, std::vector<NvtLaunch> &Ls, int64_t nsteps, NvtBuffers &B) {
  size_t off = 0;
  auto take = [&](size_t bytes) {
    const size_t o = off;
    off = (off + bytes + 255) & ~(size_t)255;
    return o;
  };
  const size_t ns = (size_t)nsteps;
  for (NvtLaunch &L : Ls) {
    if (L.host_loop) continue;
    const cass_nvt_record *rec = L.rec;
    L.o_state = take(sizeof(NvtState));
    if (rec && rec->kind) L.o_kind = take(ns);
    if (rec && rec->accepted) L.o_acc = take(ns);
    if (rec && rec->energy) L.o_energy = take(sizeof(double) * ns);
    if (rec && rec->ln_pacc) L.o_lnp = take(sizeof(double) * ns);
    if (rec && rec->rng_state) L.o_rs = take(sizeof(int64_t) * 5 * ns);
  }
  B.back = off;
  for (NvtLaunch &L : Ls)
    if (!L.host_loop) L.o_mols = take(sizeof(int) * L.mols.size());
  B.o_args = take(sizeof(NvtChainArgs) * std::max<size_t>(1, Ls.size()));
  B.in = off;
  std::vector<size_t> trav(Ls.size());
  for (size_t k = 0; k < Ls.size(); ++k)
    if (!Ls[k].host_loop) trav[k] = take(sizeof(double) * 2 * (size_t)Ls[k].a.ew.nvecs);
  B.dev = (char *)cass_scratch(e, off + 256);
  if (!B.dev) return cass_fail(e, CASS_ERR_NOMEM, "scratch");
  B.host.assign(B.in, 0);
  for (size_t k = 0; k < Ls.size(); ++k) {
    NvtLaunch &L = Ls[k];
    if (L.host_loop) continue;
    NvtState st{};
    std::memcpy(st.rng, L.rng->s, sizeof(st.rng));
    const double en_in[5] = {L.en->total, L.en->inter, L.en->inter_vdw, L.en->inter_q, L.en->reciprocal};
    std::memcpy(st.en, en_in, sizeof(st.en));
    std::memcpy(B.host.data() + L.o_state, &st, sizeof(st));
    std::memcpy(B.host.data() + L.o_mols, L.mols.data(), sizeof(int) * L.mols.size());
    NvtState *d = (NvtState *)(B.dev + L.o_state);
    const cass_nvt_record *rec = L.rec;
    NvtChainArgs &a = L.a;
    a.rng = d->rng;
    a.en = d->en;
    a.status = d->status;
    a.kind = rec && rec->kind ? (uint8_t *)(B.dev + L.o_kind) : nullptr;
    a.accepted = rec && rec->accepted ? (uint8_t *)(B.dev + L.o_acc) : nullptr;
    a.energy = rec && rec->energy ? (double *)(B.dev + L.o_energy) : nullptr;
    a.ln_pacc = rec && rec->ln_pacc ? (double *)(B.dev + L.o_lnp) : nullptr;
    a.rng_state = rec && rec->rng_state ? (int64_t *)(B.dev + L.o_rs) : nullptr;
    a.mols = (const int *)(B.dev + L.o_mols);
    a.ctrav = (double *)(B.dev + trav[k]);
    a.strav = a.ctrav + a.ew.nvecs;
  }
  return CASS_OK;
}

// Results of the batch back to the host: generator states, energies,
// records, the moved coordinates and centres.
int nvt_finish(cass_engine *e, std::vector<NvtLaunch> &Ls, int64_t nsteps, const NvtBuffers &B) {
  std::vector<int> ids;
  for (const NvtLaunch &L : Ls)
    if (!L.host_loop) ids.push_back(L.box);
  MirrorPull mirrors;
  if (int rc = mirrors.begin(e, ids, false, B.back)) return rc;
  if (B.back) HIP_TRY(e, hipMemcpyAsync(mirrors.host, B.dev, B.back, hipMemcpyDeviceToHost, e->stream));
  HIP_TRY(e, hipStreamSynchronize(e->stream));
  mirrors.end(e);
  ++e->gen;
  const size_t ns = (size_t)nsteps;
  bool bad = false;
  for (NvtLaunch &L : Ls) {
    if (L.host_loop) continue;
    cass_box_state &b = e->boxes[L.box];
    const char *h = mirrors.host;
    NvtState st;
    std::memcpy(&st, h + L.o_state, sizeof(st));
    const cass_nvt_record *rec = L.rec;
    if (L.a.kind) std::memcpy(rec->kind, h + L.o_kind, ns);
    if (L.a.accepted) std::memcpy(rec->accepted, h + L.o_acc, ns);
    if (L.a.energy) std::memcpy(rec->energy, h + L.o_energy, sizeof(double) * ns);
    if (L.a.ln_pacc) std::memcpy(rec->ln_pacc, h + L.o_lnp, sizeof(double) * ns);
    if (L.a.rng_state) std::memcpy(rec->rng_state, h + L.o_rs, sizeof(int64_t) * 5 * ns);
    std::memcpy(L.rng->s, st.rng, sizeof(st.rng));
    L.en->total = st.en[0];
    L.en->inter = st.en[1];
    L.en->inter_vdw = st.en[2];
    L.en->inter_q = st.en[3];
    L.en->reciprocal = st.en[4];
    if (L.charged) b.e_recip = st.en[4];
    b.staged_mol = -1;
    bad = bad || st.status[0];
  }
  if (bad) return cass_fail(e, CASS_ERR_STATE, "molecule energy too high before the move");
  return CASS_OK;
}

// chunks of moves per launch (a launch runs a few tens of milliseconds)
constexpr int64_t kNvtChunk = 4096;

}  // namespace

extern "C" int cass_nvt_run_device(cass_engine *e, int32_t box, cass_rng *rng, const cass_nvt_options *opt,
                                   int64_t nsteps, cass_energy *en, cass_nvt_record *rec) {
  std::vector<NvtLaunch> Ls(1);
  NvtLaunch &L = Ls[0];
  int rc = nvt_prepare(e, box, rng, opt, nsteps, en, rec, L);
  if (rc || nsteps == 0) return rc;
  if (L.host_loop) return cass_nvt_run(e, box, rng, opt, nsteps, en, rec);
  NvtBuffers B;
  if ((rc = nvt_buffers(e, Ls, nsteps, B))) return rc;
  HIP_TRY(e, hipMemcpyAsync(B.dev, B.host.data(), B.in, hipMemcpyHostToDevice, e->stream));
  nvt_kernel_t kern = nvt_kernel(L.pm, L.nse);
  HIP_TRY(e, hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)L.lds));
  for (int64_t s0 = 0; s0 < nsteps; s0 += kNvtChunk) {
    L.a.step0 = s0;
    L.a.nsteps = std::min(kNvtChunk, nsteps - s0);
    hipLaunchKernelGGL(kern, dim3(1), dim3(kNvtBlock), L.lds, e->stream, L.a);
    HIP_TRY(e, hipGetLastError());
  }
  return nvt_finish(e, Ls, nsteps, B);
}

extern "C" int cass_nvt_run_device_batch(cass_engine *e, int32_t nboxes, const int32_t *boxes, cass_rng *rngs,
                                         const cass_nvt_options *opts, int64_t nsteps, cass_energy *ens,
                                         cass_nvt_record *recs) {
  if (!e || nboxes < 0 || nsteps < 0 || (nboxes > 0 && (!boxes || !rngs || !opts || !ens))) return CASS_ERR_ARG;
  for (int i = 0; i < nboxes; ++i)
    for (int k = 0; k < i; ++k)
      if (boxes[k] == boxes[i]) return cass_fail(e, CASS_ERR_ARG, "a box appears twice in the batch");
  std::vector<NvtLaunch> Ls(nboxes);
  int rc = CASS_OK;
  for (int i = 0; i < nboxes; ++i)
    if ((rc = nvt_prepare(e, boxes[i], rngs + i, opts + i, nsteps, ens + i, recs ? recs + i : nullptr, Ls[i])))
      return rc;
  if (nsteps == 0 || nboxes == 0) return CASS_OK;
  NvtBuffers B;
  if ((rc = nvt_buffers(e, Ls, nsteps, B))) return rc;
  // the chains grouped by kernel (pair arithmetic, reciprocal site count);
  // every group is one launch per chunk of moves, one workgroup per box.  The
  // argument table holds the groups one after another.
  struct Group {
    nvt_multi_kernel_t kern;
    size_t lds, first, count;
  };
  std::vector<Group> groups;
  std::vector<NvtChainArgs> args;
  std::vector<int> done(nboxes, 0);
  for (int g = 0; g < nboxes; ++g) {
    if (done[g] || Ls[g].host_loop) continue;
    Group grp{nvt_multi_kernel(Ls[g].pm, Ls[g].nse), 0, args.size(), 0};
    for (int k = g; k < nboxes; ++k)
      if (!done[k] && !Ls[k].host_loop && Ls[k].pm == Ls[g].pm && Ls[k].nse == Ls[g].nse) {
        args.push_back(Ls[k].a);
        grp.lds = std::max(grp.lds, Ls[k].lds);
        ++grp.count;
        done[k] = 1;
      }
    groups.push_back(grp);
  }
  NvtChainArgs *d_args = (NvtChainArgs *)(B.dev + B.o_args);
  for (int64_t s0 = 0; s0 < nsteps; s0 += kNvtChunk) {
    for (NvtChainArgs &a : args) {
      a.step0 = s0;
      a.nsteps = std::min(kNvtChunk, nsteps - s0);
    }
    if (!args.empty()) std::memcpy(B.host.data() + B.o_args, args.data(), sizeof(NvtChainArgs) * args.size());
    if (s0 == 0) {
      HIP_TRY(e, hipMemcpyAsync(B.dev, B.host.data(), B.in, hipMemcpyHostToDevice, e->stream));
    } else {
      // the argument table is rewritten: wait for the launches that read it
      HIP_TRY(e, hipStreamSynchronize(e->stream));
      HIP_TRY(e, hipMemcpyAsync(d_args, B.host.data() + B.o_args, sizeof(NvtChainArgs) * args.size(),
                                hipMemcpyHostToDevice, e->stream));
    }
    for (const Group &g : groups) {
      HIP_TRY(e, hipFuncSetAttribute((const void *)g.kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)g.lds));
      hipLaunchKernelGGL(g.kern, dim3((unsigned)g.count), dim3(kNvtBlock), g.lds, e->stream,
                         (const NvtChainArgs *)(d_args + g.first));
      HIP_TRY(e, hipGetLastError());
    }
  }
  rc = nvt_finish(e, Ls, nsteps, B);
  for (int k = 0; !rc && k < nboxes; ++k)
    if (Ls[k].host_loop)
      rc = cass_nvt_run(e, boxes[k], rngs + k, opts + k, nsteps, ens + k, recs ? recs + k : nullptr);
  return rc;
}
