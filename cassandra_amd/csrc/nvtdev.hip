// nvtdev.hip -- the NVT move loop of cass_nvt_run resident on the device.
//
// nvtmc_driver.f90:94-152 choosing between Translate (move_translate.f90:23-360)
// and Rotate (move_rotate.f90:23-520), with the same random-number draws
// (random_generators.f90:51-122), energy bookkeeping and accept_or_reject
// (accept_or_reject.f90:22-65) as the host-driven loop in nvt.cpp.  One
// workgroup per box runs the moves in sequence on a copy of the box in LDS, or
// on the box itself where a copy does not fit (nvt_prepare):
// one wave prepares the next move while the others evaluate the current one,
// sharing the molecule-pair energies and the k vectors of the reciprocal
// update.  No host round trip per move: the host launches chunks of moves and
// reads the RNG state, energies and records back at the end.
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

// Waves per workgroup: the last wave prepares moves, the others share the
// molecules and the k segments.  12 waves are three per SIMD at up to 168
// VGPRs: a move of 512 waters takes 11.9 us on 12, 17.8 on 8 (the k segments
// no longer fit one per lane) and 13.7 on 16 (128 VGPRs, which spill).
constexpr int kNvtWaves = 12;
constexpr int kNvtSeg = kKSeg;   // k vectors per segment
constexpr int kNvtRing = 32;     // generator states kept around the current move
constexpr int kNvtAhead = 10;    // draws of one move (6 at most, its acceptance, the other start) and some
constexpr int kNvtStatic = 4096;  // LDS bytes left for the kernel's own
constexpr int kNvtList = 128;    // entries of a wave's molecule list and of its pair list

struct NvtChainArgs {
  BoxDev b;
  TopoDev tp;
  PairConst<double> cd;
  EwaldDev ew;
  const int4 *segs;   // k segments: (first k | length << 20, nx, ny, nz), nx rising by one per k
  int nsegs;
  int tx, ty, tz, nt_site;  // powers of the unit phases kept per axis; their sum
  int tabled;               // the phases' powers fit in LDS
  double *x, *y, *z;  // the box's site coordinates (the memory of b.x, b.y, b.z)
  double4 *comd;      // the box's (COM, max_dcom) (the memory of b.comd)
  int *meta;          // species and live flag per molecule where the box stays in device memory
  const int *mols;    // mobile molecules in locate order
  int nm, n, spa0, charged, linear;
  int nj_max;  // the largest site count of the box's molecules
  double prob_translate, max_disp, max_rot, beta;
  int64_t *rng;           // 5 words, in/out
  double *en;             // total, inter, inter_vdw, inter_q, reciprocal; in/out
  uint8_t *kind, *accepted;  // records per move or null
  double *energy, *ln_pacc;
  int64_t *rng_state;
  int *status;  // set to 1 when a molecule overlaps before its move
  // the box held in LDS for the whole chain, and the waves' buffers (offsets in bytes)
  int nsite, natoms_total, nspecies, ntypes;
  int o_x, o_y, o_z, o_comd, o_first, o_meta, o_atype, o_acharge, o_spn, o_spo, o_pt, o_pq, o_pm, o_prow, o_cand,
      o_eph, o_tab, o_ent, o_pr2, o_pcode;
};

// Orders this wave's LDS traffic for the compiler; a wave's LDS operations
// execute in order.
__device__ __forceinline__ void nvt_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The energies of one site pair of Compute_MoleculePair_Energy
// (energy_routines.f90:1589-1730) at squared distance r2d, full cutoffs, with
// the reference's FP64 operations (the arithmetic of molpair_energy<PrecFP64>).
// PM: 0 any style with the reference's FP64 operations (vdw_inter,
// qq_inter); 1 the common styles (LJ cut / cut_tail / cut_shift or none with
// Ewald, cut or no Coulomb), whose cutoff tests and pair terms are
// pair_cutoff, lj_cut, ewald_real and coul_cut directly (the branches
// vdw_inter and qq_inter take for them), FP64 operations; 2 the common
// styles in the mixed mode (hardware rcp/rsq seeds refined by Newton steps).
template <int PM>
__device__ __forceinline__ void nvt_cutoff(const PairConst<double> &cd, double r2d, bool &gv, bool &gq) {
  if (PM > 0) {
    gv = cd.vdw_style == CASS_VDW_LJ && r2d <= cd.rc_vdw2;
    gq = cd.q_style != CASS_Q_NONE && r2d <= cd.rc_coul2;
  } else {
    pair_cutoff(cd, false, r2d, gv, gq);
  }
}

template <int PM>
__device__ __forceinline__ void nvt_pair(const PairConst<double> &cd, double r2d, int ti, double qi,
                                         const double4 *prow_i, int tj, double qj, double &ev, double &eq) {
  bool gv, gq;
  nvt_cutoff<PM>(cd, r2d, gv, gq);
  using M = typename std::conditional<PM == 2, MathFast, MathRef>::type;
  gv = gv && ti >= 0 && tj >= 0;
  gq = gq && cd.q_style != CASS_Q_NONE && qi != 0.0 && qj != 0.0;
  if (PM > 0) {
    // both terms side by side and selected: their serial chains overlap
    const double4 p = prow_i[tj < 0 ? 0 : tj];
    double e_v = 0.0, e_q = 0.0;
    if (cd.vdw_style == CASS_VDW_LJ) e_v = lj_cut<double, M>(cd, r2d, p.x, p.y);
    if (cd.q_style == CASS_Q_EWALD)
      e_q = ewald_real<double, M>(cd, r2d, qi * qj);
    else if (cd.q_style != CASS_Q_NONE)
      e_q = coul_cut<double, M>(r2d, qi * qj);
    ev += gv ? e_v : 0.0;
    eq += gq ? e_q : 0.0;
  } else {
    if (gv) {
      const double4 p = prow_i[tj];
      ev += vdw_inter<double, MathRef>(cd, r2d, p.x, p.y, p.z, p.w);
    }
    if (gq) eq += qq_inter<double, MathRef>(cd, r2d, qi * qj);
  }
}

// min_image with the box kind known at compile time: the other kind's
// matrices would hold 36 scalar registers through the pair loop.
template <bool CUBIC>
__device__ __forceinline__ void nvt_image(const BoxDev &b, double &dx, double &dy, double &dz) {
  if (CUBIC) {
    if (dx > b.hL[0]) dx -= b.L[0]; else if (dx < -b.hL[0]) dx += b.L[0];
    if (dy > b.hL[1]) dy -= b.L[1]; else if (dy < -b.hL[1]) dy += b.L[1];
    if (dz > b.hL[2]) dz -= b.L[2]; else if (dz < -b.hL[2]) dz += b.L[2];
  } else {
    min_image(b, dx, dy, dz);
  }
}

// The centre prefilter of Check_MoleculePair_Cutoff (energy_routines.f90:
// 3027-3088) on squared distances.  The reference compares the square root;
// the two can differ only at the prefilter distance itself, where every site
// pair lies beyond the cutoff and beyond rcut_low, so the energies and the
// overlap test do not depend on the choice.
template <bool CUBIC>
__device__ __forceinline__ bool nvt_in_range(const BoxDev &b, double4 ci, double4 cj) {
  if (b.vdw_minimum) return true;
  double dx = ci.x - cj.x, dy = ci.y - cj.y, dz = ci.z - cj.z;
  nvt_image<CUBIC>(b, dx, dy, dz);
  const double rint = b.rcut_max + ci.w + cj.w;
  return dx * dx + dy * dy + dz * dz <= rint * rint;
}

__device__ __forceinline__ double nvt_readlane(double v, int l) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                          __builtin_amdgcn_readlane(__double2loint(v), l));
}

// Set bits of a ballot below this lane.
__device__ __forceinline__ int nvt_rank(uint64_t bal) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(bal >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bal, 0));
}

// Sums over the 16 lanes of each row, in the row's last lane.
__device__ __forceinline__ double nvt_row_sum(double v) {
  v = dpp_add<0x111, 0xf>(v);
  v = dpp_add<0x112, 0xf>(v);
  v = dpp_add<0x114, 0xf>(v);
  return dpp_add<0x118, 0xf>(v);
}

// A move ahead of its evaluation.  Two are prepared per step, since the move
// before it consumes one draw more when its acceptance is drawn.
struct NvtCand {
  double4 com_old, com_new;  // Get_COM of the old and of the trial sites
  double cx, cy, cz;         // the folded centre of a translation
  int m, rot, draws;         // molecule, rotation, draws before the acceptance
};

// The generator's states: ring[i % kNvtRing] after i draws, u[i % kNvtRing]
// the i-th draw of rranf (random_generators.f90:51-122): five-component LFSR,
// u in (0, 1).  The components step side by side on five lanes; `st` is the
// lane's component after `filled` draws.
struct NvtRng {
  int64_t st;
  int64_t filled;
};

__device__ __forceinline__ void nvt_fill(NvtRng &g, int64_t upto, int64_t (*ring)[5], double *u) {
  const int lane = threadIdx.x & 63;
  const int c = lane < 5 ? lane : 4;
  const int s1 = c == 0 ? 1 : c == 1 ? 24 : c == 3 ? 5 : 3;
  const int s2 = c == 0 ? 53 : c == 1 ? 50 : c == 2 ? 23 : c == 3 ? 24 : 33;
  const int s3 = c == 0 ? 10 : c == 1 ? 5 : c == 2 ? 29 : c == 3 ? 23 : 8;
  const uint64_t mask = c == 0 ? (uint64_t)-2 : c == 1 ? (uint64_t)-512 : c == 2 ? (uint64_t)-4096
                                                  : c == 3 ? (uint64_t)-131072 : (uint64_t)-8388608;
  const int64_t from = g.filled;
  while (g.filled < upto) {
    const uint64_t v = (uint64_t)g.st;
    const uint64_t b = ((v << s1) ^ v) >> s2;
    g.st = (int64_t)(((v & mask) << s3) ^ b);
    ++g.filled;
    if (lane < 5) ring[g.filled & (kNvtRing - 1)][lane] = g.st;
  }
  nvt_wave_sync();
  if (lane < (int)(g.filled - from)) {
    const int64_t *r = ring[(from + lane + 1) & (kNvtRing - 1)];
    u[(from + lane) & (kNvtRing - 1)] = (double)(r[0] ^ r[1] ^ r[2] ^ r[3] ^ r[4]) * 5.4210108624275221E-20 + 0.5;
  }
  nvt_wave_sync();
}

// One axis of Fold_Molecule for a cubic box: the shift of the centre c and of
// its sites by one box length when c leaves [-h, h].
__device__ __forceinline__ int nvt_fold(double c, double h) { return c > h ? -1 : c < -h ? 1 : 0; }
__device__ __forceinline__ double nvt_shift(double v, int f, double L) { return f < 0 ? v - L : f > 0 ? v + L : v; }

template <typename T>
using NvtGlobal = __attribute__((address_space(1))) T;

// The LDS of a chain; lx to lmeta stand in device memory where the box is not
// copied.
struct NvtLds {
  double *lx, *ly, *lz;
  double4 *lcomd;
  int *lfirst, *lmeta, *atype;
  double *acharge;
  int *spn, *spo, *pt;
  double *pq, *pm;
  double4 *prow;
  double *cand;  // [3][2][6 n]: old x, y, z, trial x, y, z
  cplx *eph;     // [2][3 n]
  cplx *tab;     // [2][2][n][nt_site]
};

// Both candidates of the move `step` by one wave, a half wave each: variant v
// starts at draw pos + v.  The draws and the operations are those of
// nvtmc_driver.f90:94-152 and Translate / Rotate.  A molecule whose accepted
// move the owning wave may still be writing (fm) is read from that move's
// candidate (fc, its sites at fq).
__device__ __forceinline__ void nvt_prepare_move(const NvtChainArgs &a, const NvtLds &S, const double *u,
                                                 int64_t pos, int step, NvtCand (*cand)[2], int fm,
                                                 const NvtCand *fc, const double *fq) {
  const int lane = threadIdx.x & 63, v = lane >> 5, l = lane & 31;
  const int n = a.n;
  auto draw = [&](int i) { return u[(pos + v + i) & (kNvtRing - 1)]; };
  const int rot = !(draw(0) <= a.prob_translate);
  // draw 1: the species pick (one mobile species)
  // rranf can round to 1.0 (random_generators.f90:118): the index is clamped
  const int m = a.mols[min((int)(draw(2) * a.nm), a.nm - 1)];
  const int f = S.lfirst[m];
  const bool fwd = m == fm;
  double4 co = S.lcomd[m];
  if (fwd) {
    co.x = fc->rot ? fc->com_new.x : fc->cx;
    co.y = fc->rot ? fc->com_new.y : fc->cy;
    co.z = fc->rot ? fc->com_new.z : fc->cz;
  }
  const int slot = step % 3;
  double *o = S.cand + (size_t)(slot * 2 + v) * 6 * n, *q = o + 3 * n;
  double cx = co.x, cy = co.y, cz = co.z;
  double r[9] = {};
  double dx = 0.0, dy = 0.0, dz = 0.0;
  int fx = 0, fy = 0, fz = 0, draws = 6;
  if (!rot) {
    dx = (2.0 * draw(3) - 1.0) * a.max_disp;
    dy = (2.0 * draw(4) - 1.0) * a.max_disp;
    dz = (2.0 * draw(5) - 1.0) * a.max_disp;
    cx = co.x + dx;
    cy = co.y + dy;
    cz = co.z + dz;
    // Fold_Molecule (minimum_image_separation.f90:162-240), cubic boxes
    if (a.b.cubic) {
      fx = nvt_fold(cx, a.b.hL[0]);
      fy = nvt_fold(cy, a.b.hL[1]);
      fz = nvt_fold(cz, a.b.hL[2]);
      cx = nvt_shift(cx, fx, a.b.L[0]);
      cy = nvt_shift(cy, fy, a.b.L[1]);
      cz = nvt_shift(cz, fz, a.b.L[2]);
    }
  } else if (a.linear) {
    // Rotate_Molecule_Eulerian (move_rotate.f90:468-520)
    const double th = acos(1.0 - 2.0 * draw(3));
    const double ph = (1.0 - 2.0 * draw(4)) * kPi;
    const double ps = (1.0 - 2.0 * draw(5)) * kPi;
    double sth, cth, sph, cph, sps, cps;
    sincos(th, &sth, &cth);
    sincos(ph, &sph, &cph);
    sincos(ps, &sps, &cps);
    r[0] = cps * cph - cth * sph * sps;
    r[1] = cps * sph + cth * cph * sps;
    r[2] = sps * sth;
    r[3] = -sps * cph - cth * sph * cps;
    r[4] = -sps * sph + cth * cph * cps;
    r[5] = cps * sth;
    r[6] = sth * sph;
    r[7] = -sth * cph;
    r[8] = cth;
  } else {
    // Rotate_Molecule_Axis (move_rotate.f90:362-463)
    const int axis = (int)(3.0 * draw(3)) + 1;
    const double ang = (2.0 * draw(4) - 1.0) * a.max_rot;
    draws = 5;
    // cos(0) = 1 and sin(0) = 0 exactly: only the drawn axis needs them
    double sa, ca;
    sincos(ang, &sa, &ca);
    const double c1 = axis == 1 ? ca : 1.0, c2 = axis == 2 ? ca : 1.0, c3 = axis == 3 ? ca : 1.0;
    const double s1 = axis == 1 ? sa : 0.0, s2 = axis == 2 ? sa : 0.0, s3 = axis == 3 ? sa : 0.0;
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
  for (int i = l; i < n; i += 32) {
    const double x = fwd ? fq[i] : S.lx[f + i], y = fwd ? fq[n + i] : S.ly[f + i], z = fwd ? fq[2 * n + i] : S.lz[f + i];
    o[i] = x;
    o[n + i] = y;
    o[2 * n + i] = z;
    if (!rot) {
      q[i] = nvt_shift(x + dx, fx, a.b.L[0]);
      q[n + i] = nvt_shift(y + dy, fy, a.b.L[1]);
      q[2 * n + i] = nvt_shift(z + dz, fz, a.b.L[2]);
    } else {
      const double px = x - co.x, py = y - co.y, pz = z - co.z;
      q[i] = (r[0] * px + r[1] * py + r[2] * pz) + co.x;
      q[n + i] = (r[3] * px + r[4] * py + r[5] * pz) + co.y;
      q[2 * n + i] = (r[6] * px + r[7] * py + r[8] * pz) + co.z;
    }
  }
  nvt_wave_sync();
  // the trial kernel's prefilter centres: Get_COM of each placement
  TopoDev tp = a.tp;
  tp.atom_mass = S.pm;
  const double *pp = (l & 1) ? q : o;
  const double4 com = molecule_com(tp, 0, n, pp, pp + n, pp + 2 * n);
  NvtCand &C = cand[slot][v];
  if (l == 0) {
    C.com_old = com;
    C.cx = cx;
    C.cy = cy;
    C.cz = cz;
    C.m = m;
    C.rot = rot;
    C.draws = draws;
  }
  if (l == 1) C.com_new = com;
  if (a.tabled) {
    // (2 pi as the reference truncates it) the unit phases exp(2 pi i s) of the trial sites' fractional
    // coordinates, then their powers
    cplx *eph = S.eph + v * 3 * n;
    for (int t = l; t < 3 * n; t += 32) {
      const int i = t / 3, d = t - 3 * i;
      const double sd = a.b.Li[d] * q[i] + a.b.Li[3 + d] * q[n + i] + a.b.Li[6 + d] * q[2 * n + i];
      double sv, cv;
      sincos(kTwoPi * sd, &sv, &cv);
      eph[t] = cplx{cv, sv};
    }
    nvt_wave_sync();
    cplx *tab = S.tab + (size_t)((step & 1) * 2 + v) * n * a.nt_site;
    for (int t = l; t < n * a.nt_site; t += 32) {
      const int i = t / a.nt_site;
      int p = t - i * a.nt_site, d = 0;
      if (p >= a.tx + a.ty) {
        p -= a.tx + a.ty;
        d = 2;
      } else if (p >= a.tx) {
        p -= a.tx;
        d = 1;
      }
      tab[t] = cpow_int(eph[3 * i + d], p);
    }
  }
  nvt_wave_sync();
}

// Molecule sums of one k segment from the powers of its sites' unit phases:
// exp(i k.r) at the segment's first vector is a product of three, then one
// factor exp(2 pi i s_x) per vector.
__device__ __forceinline__ void nvt_segment(const NvtChainArgs &a, const NvtLds &S, const cplx *tab, int4 sg,
                                            double (&c)[kNvtSeg], double (&s)[kNvtSeg]) {
  const int ny = sg.z < 0 ? -sg.z : sg.z, nz = sg.w < 0 ? -sg.w : sg.w;
#pragma unroll
  for (int t = 0; t < kNvtSeg; ++t) c[t] = s[t] = 0.0;
  for (int i = 0; i < a.n; ++i) {
    const cplx *ti = tab + i * a.nt_site;
    const cplx X = ti[sg.y], E = ti[1];
    cplx Y = ti[a.tx + ny], Z = ti[a.tx + a.ty + nz];
    Y.im = sg.z < 0 ? -Y.im : Y.im;
    Z.im = sg.w < 0 ? -Z.im : Z.im;
    cplx p = cmul(cmul(X, Z), Y);
    const double q = S.pq[i];
    p.re = q * p.re;
    p.im = q * p.im;
#pragma unroll
    for (int t = 0; t < kNvtSeg; ++t) {
      c[t] = c[t] + p.re;
      s[t] = s[t] + p.im;
      if (t + 1 < kNvtSeg) p = cmul(p, E);
    }
  }
}

// The same for one vector without tables: a sine and cosine per site.
__device__ __forceinline__ void nvt_vector(const NvtChainArgs &a, const NvtLds &S, const double *q, int k, double &c,
                                           double &s) {
  const double hx = a.ew.hx[k], hy = a.ew.hy[k], hz = a.ew.hz[k];
  c = s = 0.0;
  for (int i = 0; i < a.n; ++i) {
    double sn, cs;
    sincos(hx * q[i] + hy * q[a.n + i] + hz * q[2 * a.n + i], &sn, &cs);
    c = c + S.pq[i] * cs;
    s = s + S.pq[i] * sn;
  }
}

// The staged sums of one vector in device memory (Update_System_Ewald_
// Reciprocal_Energy) and its energy term.
__device__ __forceinline__ double nvt_stage(const EwaldDev &ew, size_t mk, int k, double c, double s) {
  const double cb = ew.cs[k] + (c - ew.cmol[mk + k]), sb = ew.sn[k] + (s - ew.smol[mk + k]);
  ew.cs_new[k] = cb;
  ew.sn_new[k] = sb;
  ew.cm_new[k] = c;
  ew.sm_new[k] = s;
  return ew.cn[k] * (cb * cb + sb * sb);
}

// The acceptance of a move from the waves' partial sums (accept_or_reject.f90:
// 22-65), taken by every wave for itself; en: the running energies.
struct NvtOutcome {
  int stop, acc, drawn;  // overlap before the move; accepted; acceptance drawn
  double lnp;
};

__device__ __forceinline__ NvtOutcome nvt_decide(const NvtChainArgs &a, const double (*red)[16], const int *redf,
                                                 int nc, int rot, double u, double (&en)[5]) {
  const int lane = threadIdx.x & 63, rw = lane & 15;
  const double part = nvt_row_sum(rw < nc ? red[lane >> 4][rw] : 0.0);
  const double pk = nvt_row_sum(rw < nc ? red[4][rw] : 0.0);
  const int f = rw < nc ? redf[rw] : 0;
  const double v0 = nvt_readlane(part, 15), v1 = nvt_readlane(part, 31), v2 = nvt_readlane(part, 47),
               v3 = nvt_readlane(part, 63);
  const double erm = nvt_readlane(pk, 15) * kChargeFactor;
  NvtOutcome r{__any(f & 1), 0, 0, std::numeric_limits<double>::quiet_NaN()};
  if (r.stop || __any(f & 2)) return r;
  double dE = 0.0;
  if (a.charged) dE = erm - en[4];
  if (!rot)
    dE = dE + (v2 - v0) + (v3 - v1);
  else
    dE = dE + v2 - v0 + v3 - v1;
  r.lnp = a.beta * dE;
  int acc = 0, drawn = 0;
  if (r.lnp <= 0.0) {
    acc = 1;
  } else if (r.lnp < kMaxKBT) {
    drawn = 1;
    if (u <= exp(-r.lnp)) acc = 1;
  }
  r.acc = __builtin_amdgcn_readfirstlane(acc);
  r.drawn = __builtin_amdgcn_readfirstlane(drawn);
  if (r.acc) {
    en[0] = en[0] + dE;
    en[1] = en[1] + dE;
    en[2] = en[2] + v2 - v0;
    en[3] = en[3] + v3 - v1;
    if (a.charged) en[4] = erm;
  }
  return r;
}

// The chain is one workgroup's serial work, so a move costs one compute unit's
// latency and, now, its issue rate: 28.6 us per move for 512 waters (2354 k
// vectors) when thread 0 drew and built the move, a workgroup-wide list was
// scanned together and the reciprocal sums went through global scratch, over
// a dozen barriers; 11.9 us here (6.2 to 8 the pairs, 1 the k vectors, 1.5 the
// sums and the decision), bound by the pair terms' instructions.  One barrier
// ends each move:
// - The last wave prepares the next move while the others evaluate this one:
//   both possible starts in the random stream (nvt_prepare_move).
// - Each other wave owns the molecules j = w, w + NC, ...: it alone reads and
//   commits their sites.  Its lanes list the molecules in range of either
//   placement, walk their site pairs for both r^2, and compact the pairs
//   within the cutoff, so that the pair terms run on full waves (4 in 10 pairs
//   of listed molecules lie outside the cutoff).
// - Each lane owns a k segment whose box sums stay in registers; the moving
//   molecule's old sums are loaded before the pairs and used after them.
// - Every wave adds up the partial sums and takes the decision itself.
// LOCAL: the box is copied to LDS; else it stays in device memory.
template <int PM, bool CUBIC, bool LOCAL>
__device__ __forceinline__ void nvt_chain_run(const NvtChainArgs &a, int64_t step0, int64_t nsteps) {
  __shared__ NvtCand cand[3][2];
  __shared__ int64_t ring[kNvtRing][5];
  __shared__ double uring[kNvtRing];
  __shared__ double red[2][5][16];
  __shared__ int redf[2][16];
  extern __shared__ char lds[];
  NvtLds S;
  if (LOCAL) {
    S.lx = (double *)(lds + a.o_x);
    S.ly = (double *)(lds + a.o_y);
    S.lz = (double *)(lds + a.o_z);
    S.lcomd = (double4 *)(lds + a.o_comd);
    S.lfirst = (int *)(lds + a.o_first);
    S.lmeta = (int *)(lds + a.o_meta);
  } else {
    // (through the global address space, for global loads and not flat ones)
    S.lx = (double *)(NvtGlobal<double> *)a.x;
    S.ly = (double *)(NvtGlobal<double> *)a.y;
    S.lz = (double *)(NvtGlobal<double> *)a.z;
    S.lcomd = (double4 *)(NvtGlobal<double4> *)a.comd;
    S.lfirst = (int *)(NvtGlobal<int> *)a.b.first;
    S.lmeta = (int *)(NvtGlobal<int> *)a.meta;
  }
  S.atype = (int *)(lds + a.o_atype);
  S.acharge = (double *)(lds + a.o_acharge);
  S.spn = (int *)(lds + a.o_spn);
  S.spo = (int *)(lds + a.o_spo);
  S.pt = (int *)(lds + a.o_pt);
  S.pq = (double *)(lds + a.o_pq);
  S.pm = (double *)(lds + a.o_pm);
  S.prow = (double4 *)(lds + a.o_prow);
  S.cand = (double *)(lds + a.o_cand);
  S.eph = (cplx *)(lds + a.o_eph);
  S.tab = (cplx *)(lds + a.o_tab);
  const int tid = threadIdx.x, nthr = blockDim.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), nc = (nthr >> 6) - 1;
  const bool ahead = w == nc;  // the preparing wave
  const int n = a.n, K = a.ew.nvecs, nmols = a.b.nmols;
  if (LOCAL)
    for (int i = tid; i < a.nsite; i += nthr) {
      S.lx[i] = a.x[i];
      S.ly[i] = a.y[i];
      S.lz[i] = a.z[i];
    }
  for (int i = tid; i < nmols; i += nthr) {
    if (LOCAL) {
      S.lcomd[i] = a.comd[i];
      S.lfirst[i] = a.b.first[i];
    }
    S.lmeta[i] = (a.b.species[i] << 1) | (a.b.live[i] ? 1 : 0);
  }
  for (int i = tid; i < a.natoms_total; i += nthr) {
    S.atype[i] = a.tp.atom_type[i];
    S.acharge[i] = a.tp.atom_charge[i];
  }
  for (int i = tid; i < a.nspecies; i += nthr) {
    S.spn[i] = a.tp.sp_natoms[i];
    S.spo[i] = a.tp.sp_atom_off[i];
  }
  for (int i = tid; i < n * a.ntypes; i += nthr) {
    const int ia = i / a.ntypes, tj = i - ia * a.ntypes;
    const int ti = a.tp.atom_type[a.spa0 + ia];
    const int k = (ti < 0 ? 0 : ti) * a.ntypes + tj;
    S.prow[i] = make_double4(a.tp.eps[k], a.tp.sig[k], a.tp.mn[k], a.tp.mm[k]);
  }
  if (tid < n) {
    S.pt[tid] = a.tp.atom_type[a.spa0 + tid];
    S.pq[tid] = a.tp.atom_charge[a.spa0 + tid];
    S.pm[tid] = a.tp.atom_mass[a.spa0 + tid];
  }
  double en[5];
#pragma unroll
  for (int k = 0; k < 5; ++k) en[k] = a.en[k];
  // this lane's first k segment and its box sums
  int4 sg = make_int4(0, 0, 0, 0);
  double rcs[kNvtSeg], rsn[kNvtSeg], kn[kNvtSeg];
  const int ct = w * 64 + lane, nct = nc * 64;  // evaluating lanes
  const bool has = a.charged && a.tabled && !ahead && ct < a.nsegs;
  const int more = a.tabled ? ct + nct : ct;  // the segments whose sums stay in device memory
#pragma unroll
  for (int t = 0; t < kNvtSeg; ++t) rcs[t] = rsn[t] = kn[t] = 0.0;
  if (has) {
    sg = a.segs[ct];
    const int k0 = sg.x & 0xfffff, len = sg.x >> 20;
#pragma unroll
    for (int t = 0; t < kNvtSeg; ++t) {
      const int k = k0 + (t < len ? t : len - 1);
      rcs[t] = a.ew.cs[k];
      rsn[t] = a.ew.sn[k];
      kn[t] = t < len ? a.ew.cn[k] : 0.0;
    }
  }
  const int sk0 = sg.x & 0xfffff, slen = sg.x >> 20;
  // this lane's place in a round of site pairs: E molecules of P pairs each
  const int P = n * a.nj_max, E = P <= 64 ? 64 / P : 1;
  const int pe = P <= 64 ? lane / P : 0, pp0 = P <= 64 ? lane - pe * P : lane;
  const int pia = pp0 / a.nj_max, pja = pp0 - pia * a.nj_max;
  int2 *ent = (int2 *)(lds + a.o_ent) + (ahead ? 0 : w) * kNvtList;
  double *pr2 = (double *)(lds + a.o_pr2) + (ahead ? 0 : w) * kNvtList;
  int *pcode = (int *)(lds + a.o_pcode) + (ahead ? 0 : w) * kNvtList;
  __syncthreads();
  int64_t pos = 0;  // draws consumed
  int var = 0;      // which candidate of the move holds
  int64_t st = 0;
  if (ahead) {
    NvtRng g;
    g.filled = 0;
    g.st = a.rng[lane < 5 ? lane : 4];
    if (lane < 5) ring[0][lane] = g.st;
    // the first move, then during move `st` the one after it; `to`: the move
    // to prepare, fm and pvar: the molecule moved last and its variant
    int fm = -1, pvar = 0;
    int64_t to = 0, next = 0;
    for (;;) {
      if (to < nsteps) {
        nvt_fill(g, next + kNvtAhead, ring, uring);
        const int ps = (int)((to + 1) % 3);  // the slot of the move before the current one
        nvt_prepare_move(a, S, uring, next, (int)(to % 6), cand, fm, &cand[ps][pvar],
                         S.cand + (size_t)(ps * 2 + pvar) * 6 * n + 3 * n);
      }
      __syncthreads();
      if (to > st) {
        // the current move has been evaluated
        const NvtCand &C = cand[st % 3][var];
        const int m = __builtin_amdgcn_readfirstlane(C.m), rot = __builtin_amdgcn_readfirstlane(C.rot);
        pos += __builtin_amdgcn_readfirstlane(C.draws);
        const NvtOutcome r = nvt_decide(a, red[st & 1], redf[st & 1], nc, rot, uring[pos & (kNvtRing - 1)], en);
        if (r.stop) {
          if (lane == 0) *a.status = 1;
          const int64_t from = step0 + st, to = step0 + nsteps;
          record_rest(a.kind, from, to);
          record_rest(a.accepted, from, to);
          record_rest(a.energy, from, to);
          record_rest(a.ln_pacc, from, to);
          record_rest(a.rng_state, 5 * from, 5 * to);
          break;
        }
        pos += r.drawn;
        const int64_t gi = step0 + st;
        if (lane == 0) {
          if (a.kind) a.kind[gi] = (uint8_t)rot;
          if (a.accepted) a.accepted[gi] = (uint8_t)r.acc;
          if (a.energy) a.energy[gi] = en[0];
          if (a.ln_pacc) a.ln_pacc[gi] = r.lnp;
        }
        if (a.rng_state && lane < 5) a.rng_state[5 * gi + lane] = ring[pos & (kNvtRing - 1)][lane];
        fm = r.acc ? m : -1;
        pvar = var;
        var = r.drawn;
        if (++st >= nsteps) break;
        if (r.acc && __builtin_amdgcn_readfirstlane(cand[st % 3][var].m) == m) {
          // the next move takes the molecule that has just moved: once more,
          // from the committed coordinates
          fm = -1;
          next = pos - var;
          to = st;
          __syncthreads();
          continue;
        }
      }
      // (the same start in the stream for both variants of the move after)
      next = pos + __builtin_amdgcn_readfirstlane(cand[st % 3][var].draws);
      to = st + 1;
    }
  }
  if (!ahead) __syncthreads();
  for (; !ahead && st < nsteps;) {
    const int slot = (int)(st % 3), buf = (int)(st & 1);
    const NvtCand &C = cand[slot][var];
    const int m = __builtin_amdgcn_readfirstlane(C.m), rot = __builtin_amdgcn_readfirstlane(C.rot);
    const double *o = S.cand + (size_t)(slot * 2 + var) * 6 * n, *q = o + 3 * n;
    const size_t mk = (size_t)m * K;
    double kc[kNvtSeg], ks[kNvtSeg], dc[kNvtSeg], ds[kNvtSeg];
    if (has) {
      // the old sums of the molecule, on their way during the pairs
#pragma unroll
      for (int t = 0; t < kNvtSeg; ++t) {
        const int k = sk0 + (t < slen ? t : slen - 1);
        dc[t] = a.ew.cmol[mk + k];
        ds[t] = a.ew.smol[mk + k];
      }
    }
    // --- inter energies of the old and the new placement (Compute_Molecule_Nonbond_Inter_Energy)
    double ev0 = 0.0, eq0 = 0.0, ev1 = 0.0, eq1 = 0.0;
    int ov = 0;
    // lists: molecules in range of either placement (ent, cnt from head on),
    // then site pairs within the cutoff (pr2, pcode, pcnt from phead on).  A
    // molecule beyond the prefilter of one placement has no site pair within
    // its cutoff there.
    int head = 0, cnt = 0, phead = 0, pcnt = 0;
    const double4 c0 = C.com_old, c1 = C.com_new;
    int jbase = w, pb = 0;
    for (;;) {
      if (cnt < E && jbase < nmols) {
        const int j = jbase + nc * lane;
        jbase += nct;
        bool take = false;
        int2 entry = make_int2(0, 0);
        if (j < nmols && j != m) {
          const int meta = S.lmeta[j], first = S.lfirst[j];
          const double4 cj = S.lcomd[j];
          const bool in0 = nvt_in_range<CUBIC>(a.b, c0, cj), in1 = nvt_in_range<CUBIC>(a.b, c1, cj);
          take = (meta & 1) && (in0 || in1);
          entry = make_int2(first, (S.spo[meta >> 1] << 8) | S.spn[meta >> 1]);
        }
        const uint64_t bal = __ballot(take);
        if (take) ent[(head + cnt + nvt_rank(bal)) & (kNvtList - 1)] = entry;
        cnt += __builtin_popcountll(bal);
        nvt_wave_sync();
        continue;
      }
      double r2o = 0.0, r2n = 0.0;
      bool co = false, cn = false;
      int code = 0;
      if (cnt > 0) {
        const int take = cnt < E ? cnt : E;
        int e = pe, ia = pia, ja = pja;
        bool in = pe < take;
        if (P > 64) {
          const int p = pb + lane;
          e = 0;
          ia = p / a.nj_max;
          ja = p - ia * a.nj_max;
          in = p < P;
        }
        if (in) {
          const int2 en2 = ent[(head + e) & (kNvtList - 1)];
          if (ja < (en2.y & 255)) {
            const double x = S.lx[en2.x + ja], y = S.ly[en2.x + ja], z = S.lz[en2.x + ja];
            double dx = o[ia] - x, dy = o[n + ia] - y, dz = o[2 * n + ia] - z;
            nvt_image<CUBIC>(a.b, dx, dy, dz);
            r2o = dx * dx + dy * dy + dz * dz;
            dx = q[ia] - x;
            dy = q[n + ia] - y;
            dz = q[2 * n + ia] - z;
            nvt_image<CUBIC>(a.b, dx, dy, dz);
            r2n = dx * dx + dy * dy + dz * dz;
            bool gv, gq;
            nvt_cutoff<PM>(a.cd, r2o, gv, gq);
            co = gv || gq;
            nvt_cutoff<PM>(a.cd, r2n, gv, gq);
            cn = gv || gq;
            code = (((en2.y >> 8) + ja) << 7) | (ia << 1);
            if (r2o < a.cd.rc_low2) {
              ov |= 1;
              co = false;
            }
            if (r2n < a.cd.rc_low2) {
              ov |= 2;
              cn = false;
            }
          }
        }
        pb += 64;
        if (pb >= P) {
          head += take;
          cnt -= take;
          pb = 0;
        }
      }
      // the old placement's pairs, the new one's, at the end the remainder
      const bool last = cnt == 0 && jbase >= nmols;
#pragma unroll 1
      for (int h = 0; h < (last ? 3 : 2); ++h) {
        const bool close = h == 0 ? co : h == 1 ? cn : false;
        const uint64_t bal = __ballot(close);
        if (close) {
          const int at = (phead + pcnt + nvt_rank(bal)) & (kNvtList - 1);
          pr2[at] = h ? r2n : r2o;
          pcode[at] = code | h;
        }
        pcnt += __builtin_popcountll(bal);
        nvt_wave_sync();
        if (pcnt >= 64 || (h == 2 && pcnt > 0)) {
          const int take = pcnt < 64 ? pcnt : 64;
          if (lane < take) {
            const int at = (phead + lane) & (kNvtList - 1), cd = pcode[at], ia = (cd >> 1) & 63, ja = cd >> 7;
            double ev = 0.0, eq = 0.0;
            nvt_pair<PM>(a.cd, pr2[at], S.pt[ia], S.pq[ia], S.prow + ia * a.ntypes, S.atype[ja], S.acharge[ja], ev,
                         eq);
            ev0 += (cd & 1) ? 0.0 : ev;
            eq0 += (cd & 1) ? 0.0 : eq;
            ev1 += (cd & 1) ? ev : 0.0;
            eq1 += (cd & 1) ? eq : 0.0;
          }
          phead += take;
          pcnt -= take;
          nvt_wave_sync();
        }
      }
      if (last) break;
    }
    // --- reciprocal space: Update_System_Ewald_Reciprocal_Energy (staged)
    double er = 0.0;
    if (a.charged) {
      const cplx *tab = S.tab + (size_t)(buf * 2 + var) * n * a.nt_site;
      if (has) {
        nvt_segment(a, S, tab, sg, kc, ks);
#pragma unroll
        for (int t = 0; t < kNvtSeg; ++t) {
          dc[t] = kc[t] - dc[t];
          ds[t] = ks[t] - ds[t];
          const double cb = rcs[t] + dc[t], sb = rsn[t] + ds[t];
          er += kn[t] * (cb * cb + sb * sb);
        }
      }
      // further segments, their staged sums in device memory
      for (int i = more; i < a.nsegs; i += nct) {
        const int4 s2 = a.segs[i];
        const int k0 = s2.x & 0xfffff, len = s2.x >> 20;
        double c[kNvtSeg], s[kNvtSeg];
        if (a.tabled) {
          nvt_segment(a, S, tab, s2, c, s);
#pragma unroll
          for (int t = 0; t < kNvtSeg; ++t)
            if (t < len) er += nvt_stage(a.ew, mk, k0 + t, c[t], s[t]);
        } else {
#pragma unroll 1
          for (int t = 0; t < len; ++t) {
            nvt_vector(a, S, q, k0 + t, c[0], s[0]);
            er += nvt_stage(a.ew, mk, k0 + t, c[0], s[0]);
          }
        }
      }
    }
    const double p0 = wave_total(ev0), p1 = wave_total(eq0), p2 = wave_total(ev1), p3 = wave_total(eq1);
    const double p4 = wave_total(er);
    const int f = (__any(ov & 1) ? 1 : 0) | (__any(ov & 2) ? 2 : 0);
    if (lane == 0) {
      red[buf][0][w] = p0;
      red[buf][1][w] = p1;
      red[buf][2][w] = p2;
      red[buf][3][w] = p3;
      red[buf][4][w] = p4;
      redf[buf][w] = f;
    }
    __syncthreads();
    pos += __builtin_amdgcn_readfirstlane(C.draws);
    const NvtOutcome r = nvt_decide(a, red[buf], redf[buf], nc, rot, uring[pos & (kNvtRing - 1)], en);
    if (r.stop) break;
    pos += r.drawn;
    var = r.drawn;
    ++st;
    if (r.acc) {
      if (w == m % nc) {
        // the owning wave commits the molecule; the stored centre is the
        // folded one after a translation, Get_COM after a rotation
        // (move_rotate.f90:287), max_dcom unchanged
        const int f0 = S.lfirst[m];
        for (int i = lane; i < n; i += 64) {
          S.lx[f0 + i] = q[i];
          S.ly[f0 + i] = q[n + i];
          S.lz[f0 + i] = q[2 * n + i];
        }
        if (lane == 0) {
          S.lcomd[m].x = rot ? C.com_new.x : C.cx;
          S.lcomd[m].y = rot ? C.com_new.y : C.cy;
          S.lcomd[m].z = rot ? C.com_new.z : C.cz;
        }
        nvt_wave_sync();
      }
      if (has) {
#pragma unroll
        for (int t = 0; t < kNvtSeg; ++t) {
          rcs[t] = rcs[t] + dc[t];
          rsn[t] = rsn[t] + ds[t];
          if (t < slen) {
            a.ew.cmol[mk + sk0 + t] = kc[t];
            a.ew.smol[mk + sk0 + t] = ks[t];
          }
        }
      }
      if (a.charged)
        for (int i = more; i < a.nsegs; i += nct) {
          const int4 s2 = a.segs[i];
          const int k0 = s2.x & 0xfffff, len = s2.x >> 20;
          for (int t = 0; t < len; ++t) {
            const int k = k0 + t;
            a.ew.cs[k] = a.ew.cs_new[k];
            a.ew.sn[k] = a.ew.sn_new[k];
            a.ew.cmol[mk + k] = a.ew.cm_new[k];
            a.ew.smol[mk + k] = a.ew.sm_new[k];
          }
        }
      if (st < nsteps && __builtin_amdgcn_readfirstlane(cand[st % 3][var].m) == m) {
        // the next move takes the same molecule: it is prepared anew
        __syncthreads();
        __syncthreads();
      }
    }
  }
  __syncthreads();
  if (LOCAL) {
    for (int i = tid; i < a.nsite; i += nthr) {
      a.x[i] = S.lx[i];
      a.y[i] = S.ly[i];
      a.z[i] = S.lz[i];
    }
    for (int i = tid; i < nmols; i += nthr) a.comd[i] = S.lcomd[i];
  }
  if (has) {
#pragma unroll
    for (int t = 0; t < kNvtSeg; ++t)
      if (t < slen) {
        a.ew.cs[sk0 + t] = rcs[t];
        a.ew.sn[sk0 + t] = rsn[t];
      }
  }
  if (tid < 5) a.rng[tid] = ring[pos & (kNvtRing - 1)][tid];
  if (tid == 0)
    for (int k = 0; k < 5; ++k) a.en[k] = en[k];
}

// Independent chains of several boxes, one workgroup per box: replicas of a
// system, or boxes of different state points, each on its own generator.  The
// table is constant while the kernel runs, which its address space tells the
// compiler: through a plain pointer every field would be loaded again after
// each store.
template <int PM, bool CUBIC, bool LOCAL>
__global__ void __launch_bounds__(64 * kNvtWaves)
    k_nvt_chain(const NvtChainArgs *__restrict__ args, int64_t step0, int64_t nsteps) {
  typedef const __attribute__((address_space(4))) NvtChainArgs *ConstArgs;
  nvt_chain_run<PM, CUBIC, LOCAL>(*(const NvtChainArgs *)((ConstArgs)args + blockIdx.x), step0, nsteps);
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
  int pm = 0;
  bool local = true;       // the box in LDS, else in device memory
  bool host_loop = false;  // the host-driven loop runs it
  int box = -1;
  cass_rng *rng = nullptr;
  const cass_nvt_options *opt = nullptr;
  cass_energy *en = nullptr;
  cass_nvt_record *rec = nullptr;
  bool charged = false;
  std::vector<int> mols;  // locate order of the mobile species
  size_t o_state = 0, o_kind = 0, o_acc = 0, o_energy = 0, o_lnp = 0, o_rs = 0, o_mols = 0, o_meta = 0;
};

typedef void (*nvt_kernel_t)(const NvtChainArgs *, int64_t, int64_t);

template <int PM>
nvt_kernel_t nvt_kernel(bool cubic, bool local) {
  return cubic ? (local ? k_nvt_chain<PM, true, true> : k_nvt_chain<PM, true, false>)
               : (local ? k_nvt_chain<PM, false, true> : k_nvt_chain<PM, false, false>);
}

nvt_kernel_t nvt_kernel(const NvtLaunch &L) {
  const bool cubic = L.a.b.cubic;
  return L.pm == 0 ? nvt_kernel<0>(cubic, L.local) : L.pm == 1 ? nvt_kernel<1>(cubic, L.local)
                                                               : nvt_kernel<2>(cubic, L.local);
}

// Checks, the LDS layout of the box copy, the kernel choice and the arguments
// of one chain but for its buffers (nvt_buffers).  With nsteps == 0 or
// host_loop there is nothing to launch.
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
  // LDS layout of the box copy and the waves' buffers, with the phase powers
  // where they fit
  const int nsite = (int)(b.xyz_h.size() / 3), nt = std::max(e->ntypes, 1);
  int lds_max = 0;
  HIP_TRY(e, hipDeviceGetAttribute(&lds_max, hipDeviceAttributeMaxSharedMemoryPerBlock, e->device));
  NvtChainArgs &a = L.a;
  std::memset(&a, 0, sizeof(a));
  a.nj_max = 1;
  for (int m = 0; m < b.nmols; ++m) a.nj_max = std::max(a.nj_max, e->sp_natoms[b.mol_species[m]]);
  a.tx = std::max(2, b.kmax[0] + 1);
  a.ty = b.kmax[1] + 1;
  a.tz = b.kmax[2] + 1;
  a.nt_site = a.tx + a.ty + a.tz;
  auto layout = [&](bool tabled, bool local) {
    size_t lds = 0;
    auto take = [&](size_t bytes) {
      const size_t o = lds;
      lds = (lds + bytes + 15) & ~(size_t)15;
      return (int)o;
    };
    if (local) {
      a.o_x = take(sizeof(double) * nsite);
      a.o_y = take(sizeof(double) * nsite);
      a.o_z = take(sizeof(double) * nsite);
      a.o_comd = take(sizeof(double4) * b.nmols);
      a.o_first = take(sizeof(int) * b.nmols);
      a.o_meta = take(sizeof(int) * b.nmols);
    }
    a.o_atype = take(sizeof(int) * e->natoms_total);
    a.o_acharge = take(sizeof(double) * e->natoms_total);
    a.o_spn = take(sizeof(int) * e->nspecies);
    a.o_spo = take(sizeof(int) * e->nspecies);
    a.o_pt = take(sizeof(int) * n);
    a.o_pq = take(sizeof(double) * n);
    a.o_pm = take(sizeof(double) * n);
    a.o_prow = take(sizeof(double4) * n * nt);
    a.o_cand = take(sizeof(double) * 36 * n);
    a.o_eph = take(tabled ? sizeof(cplx) * 6 * n : 0);
    a.o_tab = take(tabled ? sizeof(cplx) * 4 * n * a.nt_site : 0);
    a.o_ent = take(sizeof(int2) * kNvtList * (kNvtWaves - 1));
    a.o_pr2 = take(sizeof(double) * kNvtList * (kNvtWaves - 1));
    a.o_pcode = take(sizeof(int) * kNvtList * (kNvtWaves - 1));
    L.lds = lds;
    L.local = local;
    a.tabled = tabled ? 1 : 0;
    return lds + kNvtStatic <= (size_t)lds_max;
  };
  // A copy with the phase powers, the box in device memory with them, then
  // both without.  In device memory a move of 512 waters takes 12.4 us for
  // 12.0, one of 1080 (the largest copy) 24.3 for 23.2; fewer waves beside a
  // copy are the slower choice (1130 waters: 29.0 on eight, 24.9 here; 1300
  // without Coulomb sums: 16.9 on six, 14.9 here), so is a sine and cosine per
  // site and vector on twelve (1.3 ms for molecules of 64 sites and 16700
  // vectors, of which the vectors take 0.8).
  if (!layout(charged, true) && !layout(charged, false) && !layout(false, true) && !layout(false, false)) {
    L.host_loop = true;
    return CASS_OK;
  }
  // One workgroup passes over all molecules and k vectors for every move; from
  // some size on the host loop's launches over the whole chip are faster.  Both
  // sides in us a move, from runs of 2500 to 160000 one-site molecules (9 to
  // 245 here; 47 to 123 there), 1360 to 20000 waters without Coulomb sums (13
  // to 38; 38 to 45) and with 6000 to 55000 vectors (27 to 256; 80 to 92), and
  // molecules of 20 and 64 sites (104 and 690; 391 and 2500).
  if (!L.local) {
    const double pairs = (double)n * a.nj_max, K = charged ? b.nvecs : 0.0;
    const double here = 8.0 + 1.35e-3 * b.nmols + 0.17 * pairs + (a.tabled ? 3.5e-3 * K : 0.75e-3 * K * n);
    const double there = 40.0 + 0.6 * pairs + (charged ? 40.0 + 0.5e-3 * K : 0.0);
    if (here > there) {
      L.host_loop = true;
      return CASS_OK;
    }
  }
  const bool common = (b.p.vdw_style == CASS_VDW_NONE ||
                       (b.p.vdw_style == CASS_VDW_LJ &&
                        (b.p.vdw_sum_style == CASS_SUM_CUT || b.p.vdw_sum_style == CASS_SUM_CUT_TAIL ||
                         b.p.vdw_sum_style == CASS_SUM_CUT_SHIFT))) &&
                      (b.p.charge_style == CASS_Q_NONE || b.p.charge_style == CASS_Q_EWALD ||
                       b.p.charge_style == CASS_Q_CUT);
  // the mixed and FP32 modes take the mixed pair arithmetic for the common
  // styles (FP64 accumulation, reciprocal space and acceptance in every mode)
  L.pm = common ? (e->prec == CASS_PREC_FP64 ? 1 : 2) : 0;
  a.b = cass_box_view(e, b);
  a.tp = cass_topo_view(e);
  a.cd = make_pair_const<double>(b.p, e->ntypes);
  a.ew = cass_ewald_view(b);
  a.segs = b.segs();
  a.nsegs = charged ? b.nsegs : 0;
  if (!charged) a.ew.nvecs = 0;
  a.x = b.x;
  a.y = b.y;
  a.z = b.z;
  a.comd = b.comd;
  a.nm = nm;
  a.n = n;
  a.spa0 = e->sp_atom_off[sp];
  a.charged = charged ? 1 : 0;
  a.linear = opt->linear;
  a.prob_translate = opt->prob_translate;
  a.max_disp = opt->max_disp;
  a.max_rot = opt->max_rot;
  a.beta = b.p.beta;
  a.nsite = nsite;
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

// The buffers of a batch, laid out over all its chains: first the mobile lists
// and argument tables, then the states, then the records.  One copy in, of all
// but the records, and one out, of the states and records: with a set of copies
// per chain the calls themselves outlasted the chains.
struct NvtBuffers {
  char *dev = nullptr;
  size_t o_back = 0, in = 0;  // where the states begin; where they end
  size_t o_args = 0;
  std::vector<char> host;   // the first `in` bytes
  ChainRecords rec;
};

int nvt_buffers(cass_engine *e, std::vector<NvtLaunch> &Ls, int64_t nsteps, NvtBuffers &B) {
  size_t off = 0;
  auto take = [&](size_t bytes) {
    const size_t o = off;
    off = (off + bytes + 255) & ~(size_t)255;
    return o;
  };
  for (NvtLaunch &L : Ls)
    if (!L.host_loop) {
      L.o_mols = take(sizeof(int) * L.mols.size());
      if (!L.local) L.o_meta = take(sizeof(int) * e->boxes[L.box].nmols);
    }
  B.o_args = take(sizeof(NvtChainArgs) * std::max<size_t>(1, Ls.size()));
  B.o_back = off;
  const size_t ns = (size_t)nsteps;
  for (NvtLaunch &L : Ls) {
    if (L.host_loop) continue;
    const cass_nvt_record *rec = L.rec;
    L.o_state = take(sizeof(NvtState));
    if (rec && rec->kind) L.o_kind = B.rec.add(rec->kind, ns);
    if (rec && rec->accepted) L.o_acc = B.rec.add(rec->accepted, ns);
    if (rec && rec->energy) L.o_energy = B.rec.add(rec->energy, sizeof(double) * ns);
    if (rec && rec->ln_pacc) L.o_lnp = B.rec.add(rec->ln_pacc, sizeof(double) * ns);
    if (rec && rec->rng_state) L.o_rs = B.rec.add(rec->rng_state, sizeof(int64_t) * 5 * ns);
  }
  B.in = off;
  B.dev = (char *)cass_scratch(e, off + B.rec.staged() + 256);
  if (!B.dev) return cass_fail(e, CASS_ERR_NOMEM, "scratch");
  if (int rc = B.rec.place(e, B.dev + off)) return rc;
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
    a.kind = rec && rec->kind ? B.rec.at<uint8_t>(L.o_kind) : nullptr;
    a.accepted = rec && rec->accepted ? B.rec.at<uint8_t>(L.o_acc) : nullptr;
    a.energy = rec && rec->energy ? B.rec.at<double>(L.o_energy) : nullptr;
    a.ln_pacc = rec && rec->ln_pacc ? B.rec.at<double>(L.o_lnp) : nullptr;
    a.rng_state = rec && rec->rng_state ? B.rec.at<int64_t>(L.o_rs) : nullptr;
    a.mols = (const int *)(B.dev + L.o_mols);
    a.meta = L.local ? nullptr : (int *)(B.dev + L.o_meta);
  }
  return CASS_OK;
}

// Results of the batch back to the host: generator states, energies,
// records, the moved coordinates and centres.
int nvt_finish(cass_engine *e, std::vector<NvtLaunch> &Ls, NvtBuffers &B, MirrorPull &mirrors) {
  if (int rc = mirrors.queue(e)) return rc;
  const size_t back = B.in - B.o_back + B.rec.staged();
  if (back) HIP_TRY(e, hipMemcpyAsync(mirrors.host, B.dev + B.o_back, back, hipMemcpyDeviceToHost, e->stream));
  if (int rc = B.rec.queue(e)) return rc;
  HIP_TRY(e, hipStreamSynchronize(e->stream));
  mirrors.end(e);
  B.rec.end(mirrors.host + (B.in - B.o_back));
  ++e->gen;
  bool bad = false;
  for (NvtLaunch &L : Ls) {
    if (L.host_loop) continue;
    cass_box_state &b = e->boxes[L.box];
    const char *h = mirrors.host;
    NvtState st;
    std::memcpy(&st, h + (L.o_state - B.o_back), sizeof(st));
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
  std::vector<int> ids;
  for (const NvtLaunch &L : Ls)
    if (!L.host_loop) ids.push_back(L.box);
  MirrorPull mirrors;
  if ((rc = mirrors.reserve(e, ids, false, B.in - B.o_back + B.rec.staged()))) return rc;
  // the chains grouped by kernel; every group is one launch per chunk of
  // moves, one workgroup per box.  The argument table holds the groups one
  // after another.
  struct Group {
    nvt_kernel_t kern;
    size_t lds, first, count;
  };
  std::vector<Group> groups;
  std::vector<NvtChainArgs> args;
  std::vector<int> done(nboxes, 0);
  for (int g = 0; g < nboxes; ++g) {
    if (done[g] || Ls[g].host_loop) continue;
    Group grp{nvt_kernel(Ls[g]), 0, args.size(), 0};
    for (int k = g; k < nboxes; ++k)
      if (!done[k] && !Ls[k].host_loop && nvt_kernel(Ls[k]) == grp.kern) {
        args.push_back(Ls[k].a);
        grp.lds = std::max(grp.lds, Ls[k].lds);
        ++grp.count;
        done[k] = 1;
      }
    groups.push_back(grp);
  }
  if (!args.empty()) std::memcpy(B.host.data() + B.o_args, args.data(), sizeof(NvtChainArgs) * args.size());
  const NvtChainArgs *d_args = (const NvtChainArgs *)(B.dev + B.o_args);
  HIP_TRY(e, hipMemcpyAsync(B.dev, B.host.data(), B.in, hipMemcpyHostToDevice, e->stream));
  int lds_max = 0;
  HIP_TRY(e, hipDeviceGetAttribute(&lds_max, hipDeviceAttributeMaxSharedMemoryPerBlock, e->device));
  for (const Group &g : groups) {
    // the attribute belongs to the process: always the largest, so that engines
    // on other threads never find a smaller one than they launch with
    HIP_TRY(e, hipFuncSetAttribute((const void *)g.kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                   lds_max - kNvtStatic));
    for (int64_t s0 = 0; s0 < nsteps; s0 += kNvtChunk) {
      hipLaunchKernelGGL(g.kern, dim3((unsigned)g.count), dim3(64 * kNvtWaves), g.lds, e->stream, d_args + g.first, s0,
                         std::min(kNvtChunk, nsteps - s0));
      HIP_TRY(e, hipGetLastError());
    }
  }
  rc = nvt_finish(e, Ls, B, mirrors);
  for (int k = 0; !rc && k < nboxes; ++k)
    if (Ls[k].host_loop)
      rc = cass_nvt_run(e, boxes[k], rngs + k, opts + k, nsteps, ens + k, recs ? recs + k : nullptr);
  return rc;
}

extern "C" int cass_nvt_run_device(cass_engine *e, int32_t box, cass_rng *rng, const cass_nvt_options *opt,
                                   int64_t nsteps, cass_energy *en, cass_nvt_record *rec) {
  if (!rng || !opt || !en) return CASS_ERR_ARG;
  return cass_nvt_run_device_batch(e, 1, &box, rng, opt, nsteps, en, rec);
}
