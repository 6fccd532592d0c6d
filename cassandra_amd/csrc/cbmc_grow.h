// cbmc_grow.h -- configurational-bias growth of flexible molecules on the device.
//
// One workgroup grows one molecule fragment by fragment as Build_Molecule
// does (fragment_growth.f90:72-707, Fragment_Order :1317-1446,
// Fragment_Placement :1449-2132).  Wave 0 keeps the growth's books, a lane per
// atom, dihedral or trial: the reference's random draws (rranf,
// random_generators.f90:51-122) in its order, the rigid-body geometry and the
// selection.  The whole workgroup scores the trials of a stage -- kappa_ins
// placements of the first fragment, kappa_dih rotations of each further
// fragment -- a wave per trial, against the molecules of the box in reach.
// Its drivers:
//   k_gcmc_chain: one workgroup per box runs that box's whole sequence of
//     GCMC insertions and deletions (gcmc_driver.f90:90-200,
//     move_insert.f90:22-424, move_delete.f90:22-416) in one launch, so every
//     box of a multi-box run advances in the same persistent kernel;
//   k_gemc_chain: one workgroup per pair of boxes runs its particle transfers
//     (gemc_driver.f90:91-195, move_mol_swap.f90:22-769);
//   k_regrow_chain: one workgroup per box runs its Cut_N_Grow moves
//     (move_regrow.f90:22-510);
//   k_widom_cbmc: one workgroup per Widom insertion of a grown species
//     (widom_insert.f90:22-594), or one workgroup walking all insertions on
//     the reference's single stream.
#pragma once

#include <hip/hip_runtime.h>

#include "kernels.h"

namespace cass {

constexpr int kCbA = 16;    // atoms of a grown species
constexpr int kCbF = 8;     // fragments
constexpr int kCbK = 32;    // trials per stage
constexpr int kCbAng = 32;  // angles
constexpr int kCbDih = 32;  // dihedrals
constexpr int kCbPair = kCbA * (kCbA - 1) / 2;

// Growth description of one species (cass_cbmc_species plus what the
// reference derives from it), in device memory.
struct CbmcSpeciesDev {
  int species, natoms, nfrag, spa0, coul_cbmc;
  int frag_natoms[kCbF], frag_atoms[kCbF][kCbA];
  int frag_nconnect[kCbF], frag_connect[kCbF][kCbF];
  int frag_anchor[kCbF];
  double prob_ins[kCbF], cum_prob_ins[kCbF];
  int nconfig[kCbF];
  long long lib_off[kCbF];
  int nangles, angle[kCbAng][3];
  double angle_k[kCbAng], angle_t0[kCbAng];
  int ndihed, dihed[kCbDih][4];
  double rb[kCbDih][6];
  int kappa_ins, kappa_rot, kappa_dih;
  // fragment bonds (Fragment_Connectivity order) and the probability of
  // cutting off fragment1's side of each (prob_del1)
  int nfbond, fbond[kCbF][2];
  double prob_del1[kCbF];
  // bit masks: a fragment's atoms, a dihedral's atoms, the atoms an atom has
  // a nonzero intramolecular scaling with; the atom pairs (i < j) in order
  unsigned frag_mask[kCbF], dihed_mask[kCbDih], intra_mask[kCbA];
  uint8_t pair_i[kCbPair], pair_j[kCbPair];
  // per atom and atom pair of the species (nonbond_list, intra scaling)
  int type[kCbA];
  double q[kCbA], mass[kCbA];
  double vs[kCbA * kCbA], qs[kCbA * kCbA];
  int bonded[kCbA * kCbA];
  const double *lib;  // conformation libraries, lib_off[f] doubles in
};

// The topology's type and site tables in LDS, for the stage sums of the
// growth kernels (ok = 0 when the topology is larger than these arrays: the
// sums then read the device tables).
constexpr int kCtSp = 8, kCtAt = 128, kCtT = 16;
struct ChainTopo {
  int ok, ntypes, njmax;
  int sp_natoms[kCtSp], sp_atom_off[kCtSp];
  int atom_type[kCtAt];
  double atom_charge[kCtAt];
  double eps[kCtT * kCtT], sig[kCtT * kCtT], mn[kCtT * kCtT], mm[kCtT * kCtT];
};

// One live molecule of a box as the stage sums walk them: slot, and first
// site << 4 | species (species only where the LDS tables are used, <= 8).
// Its centre stands beside it for the distance prefilter.
struct LiveMol {
  int slot, fs;
};
// The live molecules of one box, in LDS or in device memory.
struct LiveList {
  LiveMol *mol;
  double *com;  // x[cap], y[cap], z[cap], max_dcom[cap]: lanes on neighbouring entries read without bank conflicts
  int cap;
  __device__ __forceinline__ double4 centre(int i) const {
    return make_double4(com[i], com[cap + i], com[2 * cap + i], com[3 * cap + i]);
  }
  __device__ __forceinline__ void put(int i, double4 c) const {
    com[i] = c.x;
    com[cap + i] = c.y;
    com[2 * cap + i] = c.z;
    com[3 * cap + i] = c.w;
  }
};

constexpr int kRing = 128;   // random draws held ready
constexpr int kTs = kCbA + 1;  // doubles per trial row (odd: spreads LDS banks)

// LDS state of one growing molecule (these_atoms / this_molecule) and of
// the current stage's trials.  Wave 0 keeps the growth's own bookkeeping in
// registers (GrowReg); what the other waves read stands here.
template <int NT>
struct GrowLds {
  double x[kCbA], y[kCbA], z[kCbA];
  double4 com;  // (xcom, ycom, zcom, max_dcom)
  // trial coordinates of the stage's atoms (first fragment: all its atoms;
  // later fragments: the atoms it adds), per trial
  double tx[kCbK][kTs], ty[kCbK][kTs], tz[kCbK][kTs];
  double4 tcom[kCbK];
  int tatom[kCbA], ntatom;  // the stage's atoms
  int tpos[kCbA];           // position of an atom in tatom, -1 if absent
  double sv[kCbK], sq[kCbK];
  int sov[kCbK];
  double sem;  // Eij_max of the full-cutoff pass
  double *rsq; // closest r^2 per (species site, stage atom) of the
               // full-cutoff pass, global memory; null: not kept
  // partials of the full-cutoff pass, per wave
  double pv[NT / 64], pq[NT / 64], pem[NT / 64];
  int pov[NT / 64];
  int flag, ntotal;
  double cx[kCbA], cy[kCbA], cz[kCbA];  // wave 0: the fragment being added
  // random draws: ru[i] the i-th uniform, rw[.][i] the generator's words
  // before it (indices modulo kRing); rgen draws are ready, wave 0 has
  // consumed rpos when the current phase began
  int64_t rw[5][kRing];
  double ru[kRing];
  unsigned rgen, rpos;
  double lprob[kCbF];  // log(prob_ins)
  double lk[3];        // log(kappa_ins), log(kappa_rot), (nfrag - 1) log(kappa_dih)
  double thstep;       // 2 pi / kappa_dih
  // the growth description and the topology tables, copied from device
  // memory at kernel start
  CbmcSpeciesDev sp;
  ChainTopo ct;
  // candidates of the trial a wave scores (list entries)
  int cl[NT / 64][128];
};

// Wave 0's registers of the growth (uniform over the wave): the atoms that
// exist, the fragments placed, the growth order (4 bits a fragment), draws
// consumed, and the growth's log-probabilities.
struct GrowReg {
  unsigned ex, placed, order, rpos;
  int ntotal;
  double ln_pbias, ln_pseq;
};

__device__ __forceinline__ int ufi(int v) { return __builtin_amdgcn_readfirstlane(v); }

// Orders this wave's LDS traffic for the compiler; a wave's LDS operations
// execute in order.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Copies the growth description into S.sp and the topology tables into
// S.ct, and sets up the draw ring from the generator words (every thread; a
// barrier must follow before any is read).
template <int NT>
__device__ __forceinline__ void load_tables(GrowLds<NT> &S, const CbmcSpeciesDev *src, const TopoDev &tp) {
  static_assert(sizeof(CbmcSpeciesDev) % 8 == 0, "8-byte words");
  const uint64_t *s = (const uint64_t *)src;
  uint64_t *d = (uint64_t *)&S.sp;
  const int lane = threadIdx.x;
  for (int i = lane; i < (int)(sizeof(CbmcSpeciesDev) / 8); i += NT) d[i] = s[i];
  const bool ok = tp.nspecies <= kCtSp && tp.natoms_total <= kCtAt && tp.ntypes <= kCtT;
  if (lane == 0) {
    S.ct.ok = ok;
    S.ct.ntypes = tp.ntypes;
    int m = 0;
    if (ok)
      for (int i = 0; i < tp.nspecies; ++i) m = max(m, tp.sp_natoms[i]);
    S.ct.njmax = m;
    S.rsq = nullptr;
    S.flag = 0;
  }
  // the constant logarithms and the dihedral step
  if (lane < kCbF) S.lprob[lane] = lane < src->nfrag ? log(src->prob_ins[lane]) : 0.0;
  if (lane < 3) {
    const int k = lane == 0 ? src->kappa_ins : (lane == 1 ? src->kappa_rot : src->kappa_dih);
    const double l = k != 0 ? log((double)k) : 0.0;
    S.lk[lane] = lane == 2 ? __dmul_rn((double)(src->nfrag - 1), l) : l;
    if (lane == 2) S.thstep = k != 0 ? __ddiv_rn(kTwoPi, (double)k) : 0.0;
  }
  if (!ok) return;
  for (int i = lane; i < tp.nspecies; i += NT) {
    S.ct.sp_natoms[i] = tp.sp_natoms[i];
    S.ct.sp_atom_off[i] = tp.sp_atom_off[i];
  }
  for (int i = lane; i < tp.natoms_total; i += NT) {
    S.ct.atom_type[i] = tp.atom_type[i];
    S.ct.atom_charge[i] = tp.atom_charge[i];
  }
  for (int i = lane; i < tp.ntypes * tp.ntypes; i += NT) {
    S.ct.eps[i] = tp.eps[i];
    S.ct.sig[i] = tp.sig[i];
    S.ct.mn[i] = tp.mn ? tp.mn[i] : 0.0;
    S.ct.mm[i] = tp.mm ? tp.mm[i] : 0.0;
  }
}

// reads of device memory this kernel also writes go through vector loads
template <typename T>
__device__ __forceinline__ T vld(const T *p) {
  return *(const volatile T *)p;
}

// ------------------------------------------------------------------- draws
// rranf (random_generators.f90:97-120) is five independent shift registers
// whose words are combined by XOR.  One wave advances them ahead of use, a
// register a lane, into a ring in LDS; the draws themselves are then LDS
// reads.  A draw by one lane took about 0.25 us on the growth's serial
// path, and a first fragment takes 3 kappa_ins + 6 of them.
template <int NT>
__device__ __forceinline__ void ring_start(GrowLds<NT> &S, const int64_t *words) {
  if (threadIdx.x < 5) S.rw[threadIdx.x][0] = words[threadIdx.x];
  if (threadIdx.x == 0) S.rgen = S.rpos = 0;
}

// Fills the ring to kRing - 4 draws past S.rpos (the whole wave calls it).
// Nothing else writes rgen, and the wave that consumes the draws reads only
// those that were ready when its phase began.
template <int NT>
__device__ __forceinline__ void ring_fill(GrowLds<NT> &S) {
  const int wl = threadIdx.x & 63;
  const unsigned g0 = S.rgen;
  const int n = ufi((int)(S.rpos + (kRing - 4) - g0));
  if (n <= 0) return;
  if (wl < 5) {
    const int s1 = wl == 0 ? 1 : (wl == 1 ? 24 : (wl == 3 ? 5 : 3));
    const int s2 = wl == 0 ? 53 : (wl == 1 ? 50 : (wl == 2 ? 23 : (wl == 3 ? 24 : 33)));
    const int s3 = wl == 0 ? 10 : (wl == 1 ? 5 : (wl == 2 ? 29 : (wl == 3 ? 23 : 8)));
    const uint64_t mk =
        (uint64_t)(int64_t)(wl == 0 ? -2 : (wl == 1 ? -512 : (wl == 2 ? -4096 : (wl == 3 ? -131072 : -8388608))));
    uint64_t s = (uint64_t)S.rw[wl][g0 & (kRing - 1)];
    for (int i = 1; i <= n; ++i) {
      const uint64_t b = ((s << s1) ^ s) >> s2;
      s = ((s & mk) << s3) ^ b;
      S.rw[wl][(g0 + i) & (kRing - 1)] = (int64_t)s;
    }
  }
  wave_sync();
  for (int i = wl; i < n; i += 64) {
    const unsigned k = (g0 + i + 1) & (kRing - 1);
    const int64_t w = S.rw[0][k] ^ S.rw[1][k] ^ S.rw[2][k] ^ S.rw[3][k] ^ S.rw[4][k];
    S.ru[(g0 + i) & (kRing - 1)] = (double)w * 5.4210108624275221E-20 + 0.5;
  }
  if (wl == 0) S.rgen = g0 + n;
}

// The wave that keeps the ring filled while wave 0 works.
template <int NT>
__device__ __forceinline__ bool fill_wave() {
  return (threadIdx.x >> 6) == (NT > 64 ? 1 : 0);
}

// rranf; wave 0.
template <int NT>
__device__ __forceinline__ double draw(const GrowLds<NT> &S, GrowReg &G) {
  const double u = S.ru[G.rpos & (kRing - 1)];
  G.rpos++;
  return u;
}

__device__ __forceinline__ double readlane_f64(double v, int l) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), l);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), l);
  return __hiloint2double(hi, lo);
}

__device__ __forceinline__ double readfirstlane_f64(double v) {
  const int lo = __builtin_amdgcn_readfirstlane(__double2loint(v));
  const int hi = __builtin_amdgcn_readfirstlane(__double2hiint(v));
  return __hiloint2double(hi, lo);
}

// The selection among ntrial weighted trials (fragment_growth.f90:529-620,
// 2044-2099), by the whole of wave 0: lane t < ntrial holds its trial's
// weight w and kind wk (0 a weight; 1 none: an overlap or beta E >= max_kBT;
// 2 an intramolecular overlap, whose cumulative weight repeats the previous
// one).  The cumulative weights are summed in trial order as the reference
// sums them, and the pick u W selects the first trial whose cumulative
// weight exceeds it (without del_flag; with it trial 1 is kept).  Returns,
// uniform over the wave, the trial, or -1 (cbmc_overlap) when no trial has a
// weight or the pick passes the last; wsum = W.
template <int NT>
__device__ __forceinline__ int select_trial(const GrowLds<NT> &S, GrowReg &G, int ntrial, double w, int wk, bool del_flag,
                                   double &wsum) {
  const int lane = threadIdx.x;
  const uint64_t carry = __builtin_amdgcn_ballot_w64(lane < ntrial && wk == 2);
  const uint64_t have = __builtin_amdgcn_ballot_w64(lane < ntrial && wk == 0);
  double run = 0.0, mycum = 0.0;
  for (int ii = 0; ii < ntrial; ++ii) {
    const double wi = readlane_f64(w, ii);
    if (!((carry >> ii) & 1ull)) run = ii > 0 ? __dadd_rn(run, wi) : wi;
    if (lane == ii) mycum = run;
  }
  wsum = run;
  if (!have) return -1;
  if (del_flag) return 0;
  const double pick = __dmul_rn(draw(S, G), run);
  const uint64_t b = __builtin_amdgcn_ballot_w64(lane < ntrial && pick < mycum);
  return b ? __builtin_ctzll(b) : -1;
}

// Arguments common to the drivers.
struct GrowArgs {
  BoxDev b;
  TopoDev tp;
  PairConst<double> cd;
  PairConst<float> cf;
  const CbmcSpeciesDev *sp;
  double beta;
};

// ------------------------------------------------------- the live molecules
// Lists the box's live molecules in slot order (wave 0) and returns their
// number.
template <int NT>
__device__ __forceinline__ int build_live_list(const GrowArgs &a, const LiveList &l) {
  const int wl = threadIdx.x & 63;
  int n = 0;
  for (int s0 = 0; s0 < a.b.nmols; s0 += 64) {
    const int j = s0 + wl;
    const bool on = j < a.b.nmols && vld(a.b.live + min(j, a.b.nmols - 1)) != 0;
    const uint64_t m = __builtin_amdgcn_ballot_w64(on);
    if (on) {
      const int p = n + __popcll(m & ((1ull << wl) - 1ull));
      const double *c = (const double *)(a.b.comd + j);
      l.mol[p] = LiveMol{j, (a.b.first[j] << 4) | (a.b.species[j] & 15)};
      l.put(p, make_double4(vld(c), vld(c + 1), vld(c + 2), vld(c + 3)));
    }
    n += __popcll(m);
  }
  return n;
}

// The position of slot m in the list (whole wave; -1 if absent).
__device__ __forceinline__ int live_find(const LiveList &l, int n, int m) {
  const int wl = threadIdx.x & 63;
  for (int i0 = 0; i0 < n; i0 += 64) {
    const uint64_t b = __builtin_amdgcn_ballot_w64(i0 + wl < n && l.mol[min(i0 + wl, n - 1)].slot == m);
    if (b) return i0 + __builtin_ctzll(b);
  }
  return -1;
}

// Check_MoleculePair_Cutoff (energy_routines.f90:3027-3088) for the walk of a
// stage, in double precision: reach is the cutoff and the trial's max_dcom.
// Squared distances where molpair_in_range takes the root as the reference
// does, and in cubic boxes the nearest image where the reference shifts by one
// box length: the two differ at the prefilter distance itself and for centres
// more than 1.5 lengths apart, where every site pair that the walk then meets
// (with the one shift) lies beyond the cutoff.
struct Reach {
  double x, y, z, r;
};

__device__ __forceinline__ Reach make_reach(const BoxDev &b, bool cbmc, double4 ci) {
  return Reach{ci.x, ci.y, ci.z, (cbmc ? b.rcut_cbmc : b.rcut_max) + ci.w};
}

__device__ __forceinline__ bool in_reach(const BoxDev &b, const Reach &r, double4 c) {
  if (b.vdw_minimum) return true;
  double dx = r.x - c.x, dy = r.y - c.y, dz = r.z - c.z;
  if (b.cubic) {
    dx = fma(-rint(dx * b.Li[0]), b.L[0], dx);
    dy = fma(-rint(dy * b.Li[4]), b.L[1], dy);
    dz = fma(-rint(dz * b.Li[8]), b.L[2], dz);
  } else {
    min_image(b, dx, dy, dz);
  }
  const double q = r.r + c.w;
  return dx * dx + dy * dy + dz * dz <= q * q;
}

// Atomic minimum in device memory.
__device__ __forceinline__ void global_min(double *p, double v) {
  __hip_atomic_fetch_min((__attribute__((address_space(1))) double *)p, v, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
}

// ---------------------------------------------------------------- one pair
// Atom `at` of the grown molecule at (px, py, pz) against one site (xj, yj,
// zj) of type tj and charge qj: the pair terms of Compute_MoleculePair_Energy
// (energy_routines.f90:1589-1730) with the tables in LDS, added to ev / eq;
// returns overlap (the caller discards the energies then).  LJ: the box's
// pair style is LJ cut / cut_tail / cut_shift and the grown species is
// uncharged or the box has no Coulomb style (its q-q terms are 0), so that
// branch of Check_AtomPair_Cutoff and of the pair energy is all there is.
// EM: em is raised to each in-cutoff pair's Eij_inter_vdw plus its bare q-q
// energy (the Eij_max of energy_routines.f90:1702-1705; bare q-q per style as
// Compute_AtomPair_Energy returns it, Ewald :2119, DSF :2074-2081, cut and
// minimum image :2036-2046), in FP64 from the pair's vdW term; and with
// S.rsq set, S.rsq[site_j * natoms + atom] is lowered to the pair's r^2
// (swi_atompair_rsqmin, energy_routines.f90:1636-1643, 1700).
template <typename P, int NT, bool LJ, bool EM>
__device__ __forceinline__ bool pair_term(const GrowArgs &a, const GrowLds<NT> &S, bool cbmc, int at, double px, double py,
                                 double pz, double xj, double yj, double zj, int tj, double qj, int site_j, double &ev,
                                 double &eq, double &em) {
  using TV = typename P::V;
  using TQ = typename P::Q;
  const BoxDev &b = a.b;
  const ChainTopo &ct = S.ct;
  const PairConst<double> &cd = a.cd;
  const PairConst<TV> &cv = pconst<TV>(a.cd, a.cf);
  double dx = px - xj, dy = py - yj, dz = pz - zj;
  min_image(b, dx, dy, dz);
  const double r2d = dx * dx + dy * dy + dz * dz;
  if (r2d < cd.rc_low2) return true;
  const int ti = S.sp.type[at];
  if constexpr (LJ) {
    const bool gv = r2d <= (cbmc ? cd.rc_cbmc2 : cd.rc_vdw2);
    if (!(gv || EM)) return false;
    double e_v = 0.0;
    if (gv && ti >= 0 && tj >= 0) {
      const int k = ti * ct.ntypes + tj;
      e_v = (double)lj_cut<TV, typename P::M>(cv, (TV)r2d, (TV)ct.eps[k], (TV)ct.sig[k]);
      ev += e_v;
    }
    if constexpr (EM) {
      bool g0, gq;
      pair_cutoff(cd, cbmc, r2d, g0, gq);
      if (!(gv || gq)) return false;
      if (e_v > em) em = e_v;
      if (S.rsq) {
        double *m = S.rsq + site_j * S.sp.natoms + at;
        if (r2d < *m) global_min(m, r2d);
      }
    }
    return false;
  }
  bool gv, gq;
  pair_cutoff(cd, cbmc, r2d, gv, gq);
  if (cbmc && S.sp.coul_cbmc == 0) gq = false;
  if (!(gv || gq)) return false;
  TV e_v = (TV)0;
  TQ e_q = (TQ)0;
  if (ti >= 0 && tj >= 0 && gv) {
    const int k = ti * ct.ntypes + tj;
    e_v = vdw_inter<TV, typename P::M>(cv, (TV)r2d, (TV)ct.eps[k], (TV)ct.sig[k], (TV)ct.mn[k], (TV)ct.mm[k]);
  }
  const double qi = S.sp.q[at];
  const bool any_q = cd.q_style != CASS_Q_NONE && qi != 0.0 && qj != 0.0;
  if (any_q && gq) e_q = qq_inter<TQ, typename P::M>(pconst<TQ>(a.cd, a.cf), (TQ)r2d, (TQ)(qi * qj));
  if (gv) ev += (double)e_v;
  if (gq) eq += (double)e_q;
  if (EM) {
    double bare = 0.0;
    if (any_q && gq) {
      const double rij = sqrt(r2d);
      if (cd.q_style == CASS_Q_EWALD)
        bare = qi * qj / rij * kChargeFactor;
      else if (cd.q_style == CASS_Q_DSF)
        bare = qi * qj * kChargeFactor / rij;
      else
        bare = kChargeFactor * (qi * qj) / rij;
    }
    const double eij = (gv ? (double)e_v : 0.0) + bare;
    if (eij > em) em = eij;
    if (S.rsq) {
      double *m = S.rsq + site_j * S.sp.natoms + at;
      if (r2d < *m) global_min(m, r2d);
    }
  }
  return false;
}

// The trials (tasks) of a stage this wave takes, round by round; -1: none in
// this round; a value past the last ends the stage.  late: wave 0 joins two
// rounds later, where it has each trial's intramolecular terms to do first.
// (A shared counter would balance them, but a lane's atomic under a branch
// inside such a loop was compiled so that the other lanes went round without
// it for ever.)
template <int NT>
__device__ __forceinline__ int wave_task(int round, bool late) {
  constexpr int W = NT / 64;
  const int w = ufi(threadIdx.x >> 6), skip = W > 1 && late ? 2 : 0;
  const int base = round < skip ? round * (W - 1) : skip * (W - 1) + (round - skip) * W;
  if (w == 0) return round < skip ? -1 : base + W - 1;
  return base + w - 1;
}

// idx / n with rn = 1 / n where every idx is below 2^21 (the float quotient
// is then off by less than 1 / (2 n)); big: integer division.
__device__ __forceinline__ int fast_div(int idx, int n, float rn, bool big) {
  return big ? idx / n : (int)(((float)idx + 0.5f) * rn);
}

// ------------------------------------------------------------ stage scoring
// One trial against `cnt` candidates (list entries in cl): a lane takes
// (candidate, site) items in turn, each against the stage's atoms.  With the device tables (a
// topology beyond the LDS arrays) or the CBMC energy table a lane takes
// whole molecules.
template <typename P, int NT, bool LJ>
__device__ __forceinline__ void score_candidates(const GrowArgs &a, const GrowLds<NT> &S, const LiveList &l,
                                        const int *cl, int cnt, int t, double &ev, double &eq, bool &ov) {
  const int wl = threadIdx.x & 63;
  const BoxDev &b = a.b;
  if (!LJ && (!S.ct.ok || b.apt_res > 0)) {
    int spa[kCbA];
    const int na = ufi(S.ntatom);
    for (int j = 0; j < na; ++j) spa[j] = S.sp.spa0 + S.tatom[j];
    for (int i = wl; i < cnt; i += 64) {
      const int j = l.mol[cl[i]].slot;
      ov = molpair_energy<P>(b, a.tp, a.cd, a.cf, true, S.sp.coul_cbmc != 0, na, S.tx[t], S.ty[t], S.tz[t], spa, j,
                             ev, eq, nullptr) || ov;
    }
    return;
  }
  const int na = ufi(S.ntatom), nj = ufi(S.ct.njmax);
  const float rnj = 1.0f / (float)nj;
  const int items = cnt * nj;  // cnt <= 64, nj <= 128
  double em = 0.0;
  for (int it = wl; it < items; it += 64) {
    const int c = fast_div(it, nj, rnj, false), ja = it - c * nj;
    const LiveMol m = l.mol[cl[c]];
    const int sj = m.fs & 15;
    if (ja >= S.ct.sp_natoms[sj]) continue;
    const int f = (m.fs >> 4) + ja, o = S.ct.sp_atom_off[sj] + ja;
    const double xj = b.x[f], yj = b.y[f], zj = b.z[f], qj = LJ ? 0.0 : S.ct.atom_charge[o];
    const int tj = S.ct.atom_type[o];
    for (int ia = 0; ia < na; ++ia)
      ov = pair_term<P, NT, LJ, false>(a, S, true, S.tatom[ia], S.tx[t][ia], S.ty[t][ia], S.tz[t][ia], xj, yj, zj, tj,
                                       qj, o, ev, eq, em) ||
           ov;
  }
}

// Compute_Molecule_Nonbond_Inter_Energy (energy_routines.f90:1088-1206) at
// the CBMC cutoff of the stage's atoms (tatom) at each of ntrial placements
// against every live molecule but slot `self`.  A wave takes one trial at a
// time (wave_task): it lists the molecules in reach by ballots
// over the live list, then its 64 lanes share the listed ones' sites, so no barrier stands inside a stage and a trial
// in a crowded place holds up only its own wave.  A trial's sum is the same
// whichever wave takes it.  What bounds a stage is latency, some 7 rounds of
// dependent loads per trial; results in sv / sq / sov after the caller's
// barrier.
template <typename P, int NT, bool LJ>
__device__ __forceinline__ void stage_trials(const GrowArgs &a, GrowLds<NT> &S, const LiveList &l,
                                                            int nl, int ntrial, int self, bool late) {
  const int wl = threadIdx.x & 63;
  int *cl = S.cl[ufi(threadIdx.x >> 6)];
  for (int round = 0;; ++round) {
    const int t = wave_task<NT>(round, late);
    if (t >= ntrial) break;
    if (t < 0) continue;
    const Reach r = make_reach(a.b, true, S.tcom[t]);
    double ev = 0.0, eq = 0.0;
    bool ov = false;
    int cnt = 0;
    for (int s0 = 0; s0 < nl; s0 += 64) {
      const int i = s0 + wl;
      bool in = false;
      if (i < nl) in = in_reach(a.b, r, l.centre(i)) && l.mol[i].slot != self;
      const uint64_t m = __builtin_amdgcn_ballot_w64(in);
      if (in) cl[cnt + __popcll(m & ((1ull << wl) - 1ull))] = i;
      cnt += __popcll(m);
      if (cnt >= 64) {
        wave_sync();
        score_candidates<P, NT, LJ>(a, S, l, cl, 64, t, ev, eq, ov);
        cnt -= 64;
        const int v = cl[64 + wl];
        wave_sync();
        cl[wl] = v;
      }
    }
    wave_sync();
    score_candidates<P, NT, LJ>(a, S, l, cl, cnt, t, ev, eq, ov);
    wave_sync();
    ev = wave_total(ev);
    if (!LJ) eq = wave_total(eq);
    const bool any = __builtin_amdgcn_ballot_w64(ov) != 0ull;
    if (wl == 0) {
      S.sv[t] = ev;
      S.sq[t] = eq;
      S.sov[t] = any ? 1 : 0;
    }
  }
}

// The same of the whole molecule (S.x / y / z, centre S.com) at the full
// cutoff: the (molecule, site) items go round the lanes of all waves (wave 0,
// which has the molecule's own terms to do first, comes last), a lane takes
// its item against every atom; full_sums adds the waves in order.  EM (the
// LDS tables): also the largest pair term Eij_max.
template <typename P, int NT, bool LJ, bool EM = false>
__device__ __forceinline__ void stage_full(const GrowArgs &a, GrowLds<NT> &S, const LiveList &l,
                                                          int nl, int self) {
  constexpr int W = NT / 64;
  const int wl = threadIdx.x & 63, w = ufi((threadIdx.x >> 6) + W - 1) % W;
  const BoxDev &b = a.b;
  const int na = ufi(S.sp.natoms), nj = ufi(S.ct.njmax);
  const Reach r = make_reach(b, false, S.com);
  double ev = 0.0, eq = 0.0, em = 0.0;
  bool ov = false;
  if (!LJ && !S.ct.ok) {
    // a lane takes whole molecules
    for (int i = w * 64 + wl; i < nl; i += NT) {
      const int j = l.mol[i].slot;
      if (j == self || !in_reach(b, r, l.centre(i))) continue;
      int spa[kCbA];
      for (int q = 0; q < na; ++q) spa[q] = S.sp.spa0 + q;
      ov = molpair_energy<P>(b, a.tp, a.cd, a.cf, false, S.sp.coul_cbmc != 0, na, S.x, S.y, S.z, spa, j, ev, eq,
                             nullptr) || ov;
    }
  } else {
    const int items = nl * nj;
    const bool big = items >= (1 << 21);
    const float rnj = 1.0f / (float)nj;
    for (int it = w * 64 + wl; it < items; it += NT) {
      const int c = fast_div(it, nj, rnj, big), ja = it - c * nj;
      const LiveMol m = l.mol[c];
      const int sj = m.fs & 15;
      if (m.slot == self || ja >= S.ct.sp_natoms[sj] || !in_reach(b, r, l.centre(c))) continue;
      const int f = (m.fs >> 4) + ja, o = S.ct.sp_atom_off[sj] + ja;
      const double xj = b.x[f], yj = b.y[f], zj = b.z[f], qj = LJ ? 0.0 : S.ct.atom_charge[o];
      const int tj = S.ct.atom_type[o];
      for (int ia = 0; ia < na; ++ia)
        ov = pair_term<P, NT, LJ, EM>(a, S, false, ia, S.x[ia], S.y[ia], S.z[ia], xj, yj, zj, tj, qj, o, ev, eq, em) ||
             ov;
    }
  }
  ev = wave_total(ev);
  if (!LJ) eq = wave_total(eq);
  if (EM)
    for (int off = 32; off > 0; off >>= 1) em = fmax(em, __shfl_xor(em, off));
  const bool any = __builtin_amdgcn_ballot_w64(ov) != 0ull;
  if (wl == 0) {
    S.pv[w] = ev;
    S.pq[w] = eq;
    S.pem[w] = em;
    S.pov[w] = any ? 1 : 0;
  }
}

// The waves of stage_full added in order (wave 0, after the barrier);
// returns the overlap.
template <int NT, bool EM = false>
__device__ __forceinline__ bool full_sums(GrowLds<NT> &S, double &ev, double &eq) {
  constexpr int W = NT / 64;
  ev = eq = 0.0;
  double em = 0.0;
  bool ov = false;
#pragma unroll
  for (int k = 0; k < W; ++k) {
    ev += S.pv[k];
    eq += S.pq[k];
    em = fmax(em, S.pem[k]);
    ov = ov || S.pov[k] != 0;
  }
  if (EM && threadIdx.x == 0) S.sem = em;
  return ufi(ov ? 1 : 0) != 0;
}

// ------------------------------------------------------- per-trial helpers
// Coordinates of atom k for trial t: the stage's atoms from the trial, the
// others from the grown molecule.
template <int NT>
__device__ __forceinline__ void atom_xyz(const GrowLds<NT> &S, int t, int k, double &x, double &y, double &z) {
  const int p = t >= 0 ? S.tpos[k] : -1;
  if (p >= 0) {
    x = S.tx[t][p];
    y = S.ty[t][p];
    z = S.tz[t][p];
  } else {
    x = S.x[k];
    y = S.y[k];
    z = S.z[k];
  }
}

// Dihedral d of Compute_Molecule_Dihedral_Energy (energy_routines.f90:350-447),
// RB form, with trial t's coordinates; Get_Dihedral_Angle_COS
// (internal_coordinate_routines.f90:305-410).
template <int NT>
__device__ __forceinline__ double dihedral_term(const CbmcSpeciesDev &c, const GrowLds<NT> &S, int t, int d) {
  const int *q = c.dihed[d];
  double x1, y1, z1, x2, y2, z2, x3, y3, z3, x4, y4, z4;
  atom_xyz(S, t, q[0], x1, y1, z1);
  atom_xyz(S, t, q[1], x2, y2, z2);
  atom_xyz(S, t, q[2], x3, y3, z3);
  atom_xyz(S, t, q[3], x4, y4, z4);
  const double rx12 = __dsub_rn(x1, x2), ry12 = __dsub_rn(y1, y2), rz12 = __dsub_rn(z1, z2);
  const double rx32 = __dsub_rn(x3, x2), ry32 = __dsub_rn(y3, y2), rz32 = __dsub_rn(z3, z2);
  const double rx34 = __dsub_rn(x3, x4), ry34 = __dsub_rn(y3, y4), rz34 = __dsub_rn(z3, z4);
  const double mx = __dsub_rn(__dmul_rn(ry12, rz32), __dmul_rn(ry32, rz12));
  const double my = __dadd_rn(-__dmul_rn(rx12, rz32), __dmul_rn(rz12, rx32));
  const double mz = __dsub_rn(__dmul_rn(rx12, ry32), __dmul_rn(ry12, rx32));
  const double nx = __dsub_rn(__dmul_rn(ry32, rz34), __dmul_rn(rz32, ry34));
  const double ny = __dadd_rn(-__dmul_rn(rx32, rz34), __dmul_rn(rz32, rx34));
  const double nz = __dsub_rn(__dmul_rn(rx32, ry34), __dmul_rn(ry32, rx34));
  const double msq = __dadd_rn(__dadd_rn(__dmul_rn(mx, mx), __dmul_rn(my, my)), __dmul_rn(mz, mz));
  const double nsq = __dadd_rn(__dadd_rn(__dmul_rn(nx, nx), __dmul_rn(ny, ny)), __dmul_rn(nz, nz));
  const double mdn = __dadd_rn(__dadd_rn(__dmul_rn(mx, nx), __dmul_rn(my, ny)), __dmul_rn(mz, nz));
  const double c1 = __ddiv_rn(mdn, __dsqrt_rn(__dmul_rn(msq, nsq)));
  const double c2 = __dmul_rn(c1, c1), c3 = __dmul_rn(c1, c2), c4 = __dmul_rn(c2, c2), c5 = __dmul_rn(c2, c3);
  const double *rb = c.rb[d];
  double dot = __dmul_rn(1.0, rb[0]);
  dot = __dadd_rn(dot, __dmul_rn(c1, rb[1]));
  dot = __dadd_rn(dot, __dmul_rn(c2, rb[2]));
  dot = __dadd_rn(dot, __dmul_rn(c3, rb[3]));
  dot = __dadd_rn(dot, __dmul_rn(c4, rb[4]));
  dot = __dadd_rn(dot, __dmul_rn(c5, rb[5]));
  return dot;
}

// Compute_Molecule_Dihedral_Energy of trial t: the dihedrals whose four atoms
// are in ex, summed in order.
template <int NT>
__device__ __forceinline__ double dihedral_energy(const CbmcSpeciesDev &c, const GrowLds<NT> &S, int t, unsigned ex) {
  double e = 0.0;
  const int nd = ufi(c.ndihed);
  for (int d = 0; d < nd; ++d) {
    if (ufi((int)(c.dihed_mask[d] & ~ex)) != 0) continue;
    e = __dadd_rn(e, dihedral_term(c, S, t, d));
  }
  return e;
}

// The same of the molecule itself, a lane per dihedral, by the whole of
// wave 0.
template <int NT>
__device__ __forceinline__ double dihedral_wave(const CbmcSpeciesDev &c, const GrowLds<NT> &S, unsigned ex) {
  const int lane = threadIdx.x, nd = ufi(c.ndihed);
  const bool on = lane < nd && (c.dihed_mask[min(lane, kCbDih - 1)] & ~ex) == 0;
  uint64_t m = __builtin_amdgcn_ballot_w64(on);
  if (m == 0) return 0.0;
  const double v = on ? dihedral_term(c, S, -1, lane) : 0.0;
  double e = 0.0;
  for (; m; m &= m - 1) e = __dadd_rn(e, readlane_f64(v, __builtin_ctzll(m)));
  return e;
}

// Angle k of Compute_Molecule_Angle_Energy (energy_routines.f90:283-347) of
// the grown molecule, harmonic (0 for a fixed angle); Get_Bond_Angle
// (internal_coordinate_routines.f90:188-272).
template <int NT>
__device__ __forceinline__ double angle_term(const CbmcSpeciesDev &c, const GrowLds<NT> &S, int k) {
  if (c.angle_k[k] == 0.0) return 0.0;
  const int *q = c.angle[k];
  const double rx21 = __dsub_rn(S.x[q[1]], S.x[q[0]]), ry21 = __dsub_rn(S.y[q[1]], S.y[q[0]]),
               rz21 = __dsub_rn(S.z[q[1]], S.z[q[0]]);
  const double rx32 = __dsub_rn(S.x[q[2]], S.x[q[1]]), ry32 = __dsub_rn(S.y[q[2]], S.y[q[1]]),
               rz32 = __dsub_rn(S.z[q[2]], S.z[q[1]]);
  const double c23 = __dadd_rn(__dadd_rn(__dmul_rn(rx21, rx32), __dmul_rn(ry21, ry32)), __dmul_rn(rz21, rz32));
  const double c22 = __dadd_rn(__dadd_rn(__dmul_rn(rx21, rx21), __dmul_rn(ry21, ry21)), __dmul_rn(rz21, rz21));
  const double c33 = __dadd_rn(__dadd_rn(__dmul_rn(rx32, rx32), __dmul_rn(ry32, ry32)), __dmul_rn(rz32, rz32));
  const double inv = __ddiv_rn(1.0, __dsqrt_rn(__dmul_rn(c33, c22)));
  double ct = __dmul_rn(c23, inv);
  ct = fmin(ct, 0.999999);
  ct = fmax(ct, -0.999999);
  const double th = __dsub_rn(kPi, acos(ct));
  const double d = __dsub_rn(th, c.angle_t0[k]);
  return __dmul_rn(c.angle_k[k], __dmul_rn(d, d));
}

// One intramolecular site pair of Compute_AtomPair_Energy's intra branch
// (energy_routines.f90:1831-2053, Ewald :2115-2135, DSF :2056-2082) with
// the scaling of the pair; adds E_intra_vdw, E_intra_qq and the periodic
// E_inter_qq.  LJ as in pair_term.
template <int NT, bool LJ>
__device__ __forceinline__ void intra_pair(const GrowArgs &a, const CbmcSpeciesDev &c, const GrowLds<NT> &S, int i, int j,
                                  double r2, bool gv, bool gq, double &ev, double &eq, double &eqi) {
  const int n = c.natoms;
  const double vs = c.vs[i * n + j], qs = c.qs[i * n + j];
  const int ti = c.type[i], tj = c.type[j];
  if (gv && ti >= 0 && tj >= 0) {
    const int k = ti * a.tp.ntypes + tj;
    if (LJ) {
      ev = __dadd_rn(ev, lj_cut<double>(a.cd, r2, __dmul_rn(S.ct.eps[k], vs), S.ct.sig[k]));
    } else {
      const double eps = __dmul_rn(a.tp.eps[k], vs);
      ev = __dadd_rn(ev, vdw_inter<double>(a.cd, r2, eps, a.tp.sig[k], a.tp.mn[k], a.tp.mm[k]));
    }
  }
  if (!LJ && gq) {
    const double qi = c.q[i], qj = c.q[j];
    if (a.cd.q_style == CASS_Q_EWALD) {
      const double rij = __dsqrt_rn(r2);
      const double erf_val = __dsub_rn(1.0, erfc_as<double>(__dmul_rn((double)a.cd.alpha, rij)));
      const double eij = __dmul_rn(__ddiv_rn(__dmul_rn(qi, qj), rij), kChargeFactor);
      eq = __dadd_rn(eq, __dmul_rn(qs, eij));
      eqi = __dadd_rn(eqi, __dsub_rn(0.0, __dmul_rn(erf_val, eij)));
    } else if (a.cd.q_style == CASS_Q_DSF) {
      const double rij = __dsqrt_rn(r2);
      const double cfqq = __dmul_rn(__dmul_rn(qi, qj), kChargeFactor);
      double eij = __dadd_rn(__dsub_rn(__dmul_rn((double)a.cd.dsf2, __dsub_rn(rij, (double)a.cd.rc_coul)),
                                       (double)a.cd.dsf1),
                             __ddiv_rn(erfc(__dmul_rn((double)a.cd.alpha_dsf, rij)), rij));
      eij = __dmul_rn(eij, cfqq);
      eq = __dadd_rn(eq, __dsub_rn(eij, __dmul_rn(__dsub_rn(1.0, qs), __ddiv_rn(cfqq, rij))));
    } else if (a.cd.q_style == CASS_Q_CUT || a.cd.q_style == CASS_Q_MINIMUM) {
      eq = __dadd_rn(eq, __dmul_rn(qs, __ddiv_rn(__dmul_rn(kChargeFactor, __dmul_rn(qi, qj)), __dsqrt_rn(r2))));
    }
  }
}

// Compute_Atom_Nonbond_Intra_Energy (energy_routines.f90:691-737) of atom ia
// against the atoms in the bit mask exist (bit k: atom k exists), trial t's
// coordinates; returns overlap.  Atoms whose scalings with ia are both 0 are
// skipped through intra_mask.
template <int NT, bool LJ>
__device__ __forceinline__ bool atom_intra(const GrowArgs &a, const CbmcSpeciesDev &c, const GrowLds<NT> &S, int t, int ia,
                                  unsigned exist, double &ev, double &eq, double &eqi) {
  ev = eq = eqi = 0.0;
  double xi, yi, zi;
  atom_xyz(S, t, ia, xi, yi, zi);
  const int n = c.natoms;
  unsigned m = (unsigned)ufi((int)(exist & c.intra_mask[ia] & ~(1u << ia)));
  bool over = false;
  for (; m; m &= m - 1) {
    const int ja = __builtin_ctz(m);
    const bool nzv = c.vs[ia * n + ja] > 0.0, nzq = c.qs[ia * n + ja] > 0.0;
    double xj, yj, zj;
    atom_xyz(S, t, ja, xj, yj, zj);
    const double rx = __dsub_rn(xj, xi), ry = __dsub_rn(yj, yi), rz = __dsub_rn(zj, zi);
    const double r2 = __dadd_rn(__dadd_rn(__dmul_rn(rx, rx), __dmul_rn(ry, ry)), __dmul_rn(rz, rz));
    if (r2 < (double)a.cd.rc_low2 && nzv) over = true;
    bool gv, gq;
    pair_cutoff(a.cd, true, r2, gv, gq);
    gv = gv && nzv;
    gq = gq && nzq;
    if (!over && (gv || gq)) intra_pair<NT, LJ>(a, c, S, ja, ia, r2, gv, gq, ev, eq, eqi);
  }
  return over;
}

// The grown molecule's intramolecular terms (every atom existing) by wave 0:
// every lane below 64 calls it and gets the results.  The nonbonded part of
// Compute_Molecule_Nonbond_Intra_Energy (energy_routines.f90:980-1085) takes
// one lane per atom pair and adds the pair terms in the reference's (ia, ja)
// order up to the first pair that overlaps, where the reference returns; the
// angles and dihedrals (:283-447) take one lane per term, added in order.
// Returns the intramolecular overlap.
template <int NT, bool LJ>
__device__ __forceinline__ bool mol_terms_wave(const GrowArgs &a, const CbmcSpeciesDev &c, const GrowLds<NT> &S, double &ev,
                               double &eq, double &eqi, double &ea, double &ed) {
  const int lane = threadIdx.x;
  const int n = ufi(c.natoms), np = n * (n - 1) / 2;
  ev = eq = eqi = 0.0;
  bool ov = false;
  for (int p0 = 0; p0 < np && !ov; p0 += 64) {
    const int p = p0 + lane;
    double pv = 0.0, pq = 0.0, pqi = 0.0;
    bool po = false, some = false;
    if (p < np) {
      const int ia = c.pair_i[p], ja = c.pair_j[p];
      const double rx = __dsub_rn(S.x[ia], S.x[ja]), ry = __dsub_rn(S.y[ia], S.y[ja]),
                   rz = __dsub_rn(S.z[ia], S.z[ja]);
      const double r2 = __dadd_rn(__dadd_rn(__dmul_rn(rx, rx), __dmul_rn(ry, ry)), __dmul_rn(rz, rz));
      if (r2 <= (double)a.cd.rc_low2 && !c.bonded[ia * n + ja]) {
        po = true;
      } else {
        bool gv, gq;
        pair_cutoff(a.cd, false, r2, gv, gq);
        some = gv || gq;
        if (some) intra_pair<NT, LJ>(a, c, S, ia, ja, r2, gv, gq, pv, pq, pqi);
      }
    }
    const uint64_t bo = __builtin_amdgcn_ballot_w64(po);
    // pairs outside every cutoff or wholly scaled away add 0
    uint64_t m = __builtin_amdgcn_ballot_w64(some && (pv != 0.0 || pq != 0.0 || pqi != 0.0));
    if (bo) m &= (bo & (0ull - bo)) - 1ull;
    for (; m; m &= m - 1) {
      const int k = __builtin_ctzll(m);
      ev = __dadd_rn(ev, readlane_f64(pv, k));
      eq = __dadd_rn(eq, readlane_f64(pq, k));
      eqi = __dadd_rn(eqi, readlane_f64(pqi, k));
    }
    ov = bo != 0;
  }
  ea = 0.0;
  const int nan = ufi(c.nangles);
  const double va = lane < nan ? angle_term(c, S, lane) : 0.0;
  for (int k = 0; k < nan; ++k) ea = __dadd_rn(ea, readlane_f64(va, k));
  ed = dihedral_wave(c, S, (1u << n) - 1u);
  return ov;
}

// Get_COM / Compute_Max_Com_Distance (get_com.f90:45-121, 220-295) over the
// atoms in the bit mask ex with trial t's coordinates.
template <int NT>
__device__ __forceinline__ double4 com_of(const CbmcSpeciesDev &c, const GrowLds<NT> &S, int t, unsigned ex) {
  double tm = 0.0, cx = 0.0, cy = 0.0, cz = 0.0;
  for (unsigned m = ex; m; m &= m - 1) {
    const int k = __builtin_ctz(m);
    double x, y, z;
    atom_xyz(S, t, k, x, y, z);
    tm = __dadd_rn(tm, c.mass[k]);
    cx = __dadd_rn(cx, __dmul_rn(c.mass[k], x));
    cy = __dadd_rn(cy, __dmul_rn(c.mass[k], y));
    cz = __dadd_rn(cz, __dmul_rn(c.mass[k], z));
  }
  cx = __ddiv_rn(cx, tm);
  cy = __ddiv_rn(cy, tm);
  cz = __ddiv_rn(cz, tm);
  double dmax = 0.0;
  for (unsigned m = ex; m; m &= m - 1) {
    const int k = __builtin_ctz(m);
    double x, y, z;
    atom_xyz(S, t, k, x, y, z);
    const double dx = __dsub_rn(x, cx), dy = __dsub_rn(y, cy), dz = __dsub_rn(z, cz);
    const double r2 = __dadd_rn(__dadd_rn(__dmul_rn(dx, dx), __dmul_rn(dy, dy)), __dmul_rn(dz, dz));
    dmax = r2 > dmax ? r2 : dmax;
  }
  return make_double4(cx, cy, cz, __dsqrt_rn(dmax));
}

// com_of of the molecule itself by wave 0, lane k holding atom k at
// (x, y, z): the sums in atom order, the distances side by side.
__device__ __forceinline__ double4 com_wave(const CbmcSpeciesDev &c, unsigned ex, double x, double y, double z) {
  const int lane = threadIdx.x;
  const double ms = c.mass[min(lane, kCbA - 1)];
  const double mx = __dmul_rn(ms, x), my = __dmul_rn(ms, y), mz = __dmul_rn(ms, z);
  double tm = 0.0, cx = 0.0, cy = 0.0, cz = 0.0;
  for (unsigned m = ex; m; m &= m - 1) {
    const int k = __builtin_ctz(m);
    tm = __dadd_rn(tm, readlane_f64(ms, k));
    cx = __dadd_rn(cx, readlane_f64(mx, k));
    cy = __dadd_rn(cy, readlane_f64(my, k));
    cz = __dadd_rn(cz, readlane_f64(mz, k));
  }
  cx = __ddiv_rn(cx, tm);
  cy = __ddiv_rn(cy, tm);
  cz = __ddiv_rn(cz, tm);
  const double dx = __dsub_rn(x, cx), dy = __dsub_rn(y, cy), dz = __dsub_rn(z, cz);
  const double r2 = __dadd_rn(__dadd_rn(__dmul_rn(dx, dx), __dmul_rn(dy, dy)), __dmul_rn(dz, dz));
  double dmax = 0.0;
  for (unsigned m = ex; m; m &= m - 1) {
    const double v = readlane_f64(r2, __builtin_ctz(m));
    dmax = v > dmax ? v : dmax;
  }
  return make_double4(cx, cy, cz, __dsqrt_rn(dmax));
}

// Get_Aligner_Hanger (fragment_growth.f90:2135-2185)
__device__ __forceinline__ void aligner_hanger(double v1[3], double v2[3], double al[3][3], double ha[3][3]) {
  const double n1 = __dsqrt_rn(__dadd_rn(__dadd_rn(__dmul_rn(v1[0], v1[0]), __dmul_rn(v1[1], v1[1])),
                                         __dmul_rn(v1[2], v1[2])));
  for (int i = 0; i < 3; ++i) v1[i] = __ddiv_rn(v1[i], n1);
  const double n2 = __dsqrt_rn(__dadd_rn(__dadd_rn(__dmul_rn(v2[0], v2[0]), __dmul_rn(v2[1], v2[1])),
                                         __dmul_rn(v2[2], v2[2])));
  for (int i = 0; i < 3; ++i) v2[i] = __ddiv_rn(v2[i], n2);
  double p1[3], p2[3];
  p1[0] = __dsub_rn(__dmul_rn(v1[1], v2[2]), __dmul_rn(v1[2], v2[1]));
  p1[1] = __dadd_rn(-__dmul_rn(v1[0], v2[2]), __dmul_rn(v1[2], v2[0]));
  p1[2] = __dsub_rn(__dmul_rn(v1[0], v2[1]), __dmul_rn(v1[1], v2[0]));
  const double np1 = __dsqrt_rn(__dadd_rn(__dadd_rn(__dmul_rn(p1[0], p1[0]), __dmul_rn(p1[1], p1[1])),
                                          __dmul_rn(p1[2], p1[2])));
  for (int i = 0; i < 3; ++i) p1[i] = __ddiv_rn(p1[i], np1);
  p2[0] = __dsub_rn(__dmul_rn(v1[1], p1[2]), __dmul_rn(v1[2], p1[1]));
  p2[1] = __dadd_rn(-__dmul_rn(v1[0], p1[2]), __dmul_rn(v1[2], p1[0]));
  p2[2] = __dsub_rn(__dmul_rn(v1[0], p1[1]), __dmul_rn(v1[1], p1[0]));
  const double np2 = __dsqrt_rn(__dadd_rn(__dadd_rn(__dmul_rn(p2[0], p2[0]), __dmul_rn(p2[1], p2[1])),
                                          __dmul_rn(p2[2], p2[2])));
  for (int i = 0; i < 3; ++i) p2[i] = __ddiv_rn(p2[i], np2);
  for (int i = 0; i < 3; ++i) {
    al[0][i] = v1[i];
    al[1][i] = p2[i];
    al[2][i] = p1[i];
    ha[i][0] = v1[i];
    ha[i][1] = p2[i];
    ha[i][2] = p1[i];
  }
}

// 3x3 matrix times vector in the reference's order (x m1 + y m2 + z m3)
__device__ __forceinline__ double mrow(const double m[3], double x, double y, double z) {
  return __dadd_rn(__dadd_rn(__dmul_rn(x, m[0]), __dmul_rn(y, m[1])), __dmul_rn(z, m[2]));
}

// ------------------------------------------------------------ Build_Molecule
// Fragment_Order (fragment_growth.f90:1317-1446) from fragment start; wave 0.
// live: bit mask of the live fragments; the hanging fragments stand 4 bits
// each in one word.
template <int NT>
__device__ __forceinline__ void fragment_order(const CbmcSpeciesDev &c, const GrowLds<NT> &S, GrowReg &G, int start,
                                      unsigned live) {
  unsigned hang = 0;
  int nc = 0;
  auto hang_from = [&](int f) {
    const int n = ufi(c.frag_nconnect[f]);
    for (int i = 0; i < n; ++i) {
      const int id = ufi(c.frag_connect[f][i]);
      if (!((live >> id) & 1u)) hang |= (unsigned)id << (4 * nc++);
    }
  };
  hang_from(start);
  while (nc > 0) {
    double tot = 0.0;
    for (int i = 0; i < nc; ++i) {
      const double p = (double)(ufi(c.frag_natoms[(hang >> (4 * i)) & 15u]) - 2);
      tot = i == 0 ? p : __dadd_rn(tot, p);
    }
    const double u = draw(S, G);
    double cum = 0.0, p = 0.0;
    int i = 0;
    for (;; ++i) {
      p = (double)(ufi(c.frag_natoms[(hang >> (4 * i)) & 15u]) - 2);
      cum = i == 0 ? p : __dadd_rn(cum, p);
      if (i >= nc - 1 || u < __ddiv_rn(cum, tot)) break;
    }
    const int id = (int)((hang >> (4 * i)) & 15u);
    // one hanging fragment: log(p / p) = 0
    if (nc > 1) G.ln_pseq = __dadd_rn(G.ln_pseq, log(__ddiv_rn(p, tot)));
    G.order |= (unsigned)id << (4 * G.ntotal++);
    live |= 1u << id;
    const unsigned below = (1u << (4 * i)) - 1u;
    hang = (hang & below) | ((i < 7 ? hang >> (4 * (i + 1)) : 0u) << (4 * i));
    nc--;
    hang_from(id);
  }
}

// The first fragment of Build_Molecule with get_fragorder
// (fragment_growth.f90:72-450); the whole of wave 0.  Step 1: the fragment
// and the growth order; Step 2: its conformation; Step 3: orientation; then
// the kappa_ins placements, a lane each.  del_flag: S.x / y / z hold the
// molecule, trial 1 is its own placement.  keep_order: get_fragorder off (the
// GEMC deletion half, :245-253): G.order and G.ln_pseq stay.
template <int NT>
__device__ __forceinline__ void first_fragment(const GrowArgs &a, GrowLds<NT> &S, GrowReg &G, bool del_flag, bool keep_order) {
  const CbmcSpeciesDev &c = S.sp;
  const int lane = threadIdx.x;
  const int ki = ufi(c.kappa_ins), nfrag = ufi(c.nfrag);
  G.ln_pbias = 0.0;
  G.placed = 0;
  int fs;
  if (keep_order) {
    fs = (int)(G.order & 15u);
    G.ntotal = nfrag;
  } else {
    const double u = draw(S, G);
    const uint64_t b =
        __builtin_amdgcn_ballot_w64(lane < nfrag - 1 && u < c.cum_prob_ins[min(lane, kCbF - 1)]);
    fs = b ? (int)__builtin_ctzll(b) : nfrag - 1;
    G.ln_pseq = S.lprob[fs];
    G.order = (unsigned)fs;
    G.ntotal = 1;
    if (nfrag > 1) fragment_order(c, S, G, fs, 1u << fs);
  }
  const int nfa = ufi(c.frag_natoms[fs]);
  const int at = c.frag_atoms[fs][min(lane, kCbA - 1)];
  G.ex = (unsigned)ufi((int)c.frag_mask[fs]);
  double r11 = 1.0, r12 = 0.0, r13 = 0.0, r21 = 0.0, r22 = 1.0, r23 = 0.0, r31 = 0.0, r32 = 0.0, r33 = 1.0;
  if (!del_flag) {
    // rranf can round to 1.0 (random_generators.f90:118): the index is clamped
    const int nconf = ufi(c.nconfig[fs]);
    const int conf = ufi(min((int)(draw(S, G) * nconf), nconf - 1));
    const double *lib = c.lib + c.lib_off[fs] + (size_t)conf * nfa * 3;
    double lx = 0.0, ly = 0.0, lz = 0.0;
    if (lane < nfa) {
      lx = lib[3 * lane];
      ly = lib[3 * lane + 1];
      lz = lib[3 * lane + 2];
    }
    // Rotate_Molecule_Eulerian (rotation_routines.f90:41-137): the three
    // angles' sines and cosines on three lanes
    const double u1 = draw(S, G), u2 = draw(S, G), u3 = draw(S, G);
    const double ang = lane == 0 ? acos(__dsub_rn(1.0, __dmul_rn(2.0, u1)))
                                 : __dmul_rn(__dsub_rn(1.0, __dmul_rn(2.0, lane == 1 ? u2 : u3)), kPi);
    double sn, cs;
    sincos(ang, &sn, &cs);
    const double cth = readlane_f64(cs, 0), sth = readlane_f64(sn, 0), cph = readlane_f64(cs, 1),
                 sph = readlane_f64(sn, 1), cps = readlane_f64(cs, 2), sps = readlane_f64(sn, 2);
    r11 = __dsub_rn(__dmul_rn(cps, cph), __dmul_rn(__dmul_rn(cth, sph), sps));
    r12 = __dadd_rn(__dmul_rn(cps, sph), __dmul_rn(__dmul_rn(cth, cph), sps));
    r13 = __dmul_rn(sps, sth);
    r21 = __dsub_rn(__dmul_rn(-sps, cph), __dmul_rn(__dmul_rn(cth, sph), cps));
    r22 = __dadd_rn(__dmul_rn(-sps, sph), __dmul_rn(__dmul_rn(cth, cph), cps));
    r23 = __dmul_rn(cps, sth);
    r31 = __dmul_rn(sth, sph);
    r32 = __dmul_rn(-sth, cph);
    r33 = cth;
    if (lane < nfa) {
      S.x[at] = lx;
      S.y[at] = ly;
      S.z[at] = lz;
    }
    wave_sync();
  }
  // lane k: atom k
  const int k0 = min(lane, kCbA - 1);
  double x = S.x[k0], y = S.y[k0], z = S.z[k0];
  const double4 com = com_wave(c, G.ex, x, y, z);
  if (!del_flag) {
    const double dx = __dsub_rn(x, com.x), dy = __dsub_rn(y, com.y), dz = __dsub_rn(z, com.z);
    x = __dadd_rn(__dadd_rn(__dadd_rn(__dmul_rn(r11, dx), __dmul_rn(r12, dy)), __dmul_rn(r13, dz)), com.x);
    y = __dadd_rn(__dadd_rn(__dadd_rn(__dmul_rn(r21, dx), __dmul_rn(r22, dy)), __dmul_rn(r23, dz)), com.y);
    z = __dadd_rn(__dadd_rn(__dadd_rn(__dmul_rn(r31, dx), __dmul_rn(r32, dy)), __dmul_rn(r33, dz)), com.z);
    if (lane < kCbA && ((G.ex >> lane) & 1u)) {
      S.x[lane] = x;
      S.y[lane] = y;
      S.z[lane] = z;
    }
  }
  // the stage's atoms: the first fragment's, in Fragment_Info order
  if (lane < kCbA) S.tpos[lane] = -1;
  wave_sync();
  double fx = 0.0, fy = 0.0, fz = 0.0;  // lane j: the fragment's atom j from the centre
  if (lane < nfa) {
    S.tatom[lane] = at;
    S.tpos[at] = lane;
    fx = __dsub_rn(S.x[at], com.x);
    fy = __dsub_rn(S.y[at], com.y);
    fz = __dsub_rn(S.z[at], com.z);
    S.cx[lane] = fx;
    S.cy[lane] = fy;
    S.cz[lane] = fz;
  }
  wave_sync();
  // the placements' centres: three draws each, none for trial 1 of a deletion
  double xa = com.x, ya = com.y, za = com.z;
  const int skip = del_flag ? 1 : 0;
  if (lane < ki && lane >= skip) {
    const unsigned r = G.rpos + 3u * (unsigned)(lane - skip);
    xa = __dmul_rn(__dsub_rn(0.5, S.ru[r & (kRing - 1)]), a.b.L[0]);
    ya = __dmul_rn(__dsub_rn(0.5, S.ru[(r + 1) & (kRing - 1)]), a.b.L[1]);
    za = __dmul_rn(__dsub_rn(0.5, S.ru[(r + 2) & (kRing - 1)]), a.b.L[2]);
  }
  G.rpos += 3u * (unsigned)(ki - skip);
  // Compute_Max_COM_Distance once, at the first trial's placement
  const double xa0 = readlane_f64(xa, 0), ya0 = readlane_f64(ya, 0), za0 = readlane_f64(za, 0);
  const double ex = __dsub_rn(__dadd_rn(fx, xa0), xa0), ey = __dsub_rn(__dadd_rn(fy, ya0), ya0),
               ez = __dsub_rn(__dadd_rn(fz, za0), za0);
  const double r2 = __dadd_rn(__dadd_rn(__dmul_rn(ex, ex), __dmul_rn(ey, ey)), __dmul_rn(ez, ez));
  double dmax = 0.0;
  for (int j = 0; j < nfa; ++j) {
    const double v = readlane_f64(r2, j);
    dmax = v > dmax ? v : dmax;
  }
  const double md = __dsqrt_rn(dmax);
  if (lane < ki) {
    for (int j = 0; j < nfa; ++j) {
      S.tx[lane][j] = __dadd_rn(S.cx[j], xa);
      S.ty[lane][j] = __dadd_rn(S.cy[j], ya);
      S.tz[lane][j] = __dadd_rn(S.cz[j], za);
    }
    S.tcom[lane] = make_double4(xa, ya, za, md);
  }
  if (lane == 0) {
    S.ntatom = nfa;
    S.ntotal = G.ntotal;
    S.flag = 0;
    S.rpos = G.rpos;
  }
}

template <typename P, int NT, bool LJ>
__device__ __forceinline__ void fragment_placement(const GrowArgs &a, GrowLds<NT> &S, GrowReg &G,
                                                                  const LiveList &l, int nl, int self, bool del_flag,
                                                                  int i0, double e_prev);

// Build_Molecule from its first fragment's placements on (first_fragment,
// wave 0, before a barrier): scores them, selects one (fragment_growth.f90:
// 529-620) and grows the rest.  Every thread calls it; S.flag = cbmc_overlap
// after the caller's next barrier, G the growth's log-probabilities (wave 0),
// S.x / y / z the grown molecule, S.com its centre.
template <typename P, int NT, bool LJ>
__device__ __forceinline__ void build_molecule(const GrowArgs &a, GrowLds<NT> &S, GrowReg &G,
                                                              const LiveList &l, int nl, int self, bool del_flag) {
  const CbmcSpeciesDev &c = S.sp;
  const int lane = threadIdx.x;
  const int ki = ufi(c.kappa_ins);
  stage_trials<P, NT, LJ>(a, S, l, nl, ki, self, false);
  __syncthreads();
  double e_prev = 0.0;
  if (lane < 64) {
    // weights, one lane per trial
    double w = 0.0, e_t = 0.0;
    int wk = 1;
    if (lane < ki && !S.sov[lane]) {
      e_t = __dadd_rn(S.sv[lane], S.sq[lane]);
      const double bk = __dmul_rn(a.beta, e_t);
      if (!(bk >= kMaxKBT)) {
        w = exp(-bk);
        wk = 0;
      }
    }
    double wsum;
    const int trial = select_trial(S, G, ki, w, wk, del_flag, wsum);
    if (trial < 0) {
      if (lane == 0) S.flag = 1;
    } else {
      G.ln_pbias = __dsub_rn(__dsub_rn(G.ln_pbias, __dmul_rn(a.beta, readlane_f64(e_t, trial))), log(wsum));
      if (lane < S.ntatom) {
        const int at = S.tatom[lane];
        S.x[at] = S.tx[trial][lane];
        S.y[at] = S.ty[trial][lane];
        S.z[at] = S.tz[trial][lane];
      }
      if (lane == 0) S.com = S.tcom[trial];
      wave_sync();
      G.placed |= 1u << (G.order & 15u);
      e_prev = dihedral_wave(c, S, G.ex);  // e_total of Fragment_Placement
    }
    wave_sync();
  }
  // Step 5: Fragment_Placement of the remaining fragments
  fragment_placement<P, NT, LJ>(a, S, G, l, nl, self, del_flag, 1, e_prev);
}

// One fragment's trials (fragment_growth.f90:1449-1925); the whole of wave 0:
// the conformation, its frame turned onto the grown part, and the kappa_dih
// rotations about the connecting bond, a lane each.  grown: the atoms before
// the fragment.  The stage's atoms are those the fragment adds (neither
// anchor).
template <int NT>
__device__ __forceinline__ void fragment_trials(const GrowArgs &a, GrowLds<NT> &S, GrowReg &G, int i, bool del_flag,
                                       unsigned &newx, unsigned &grown) {
  const CbmcSpeciesDev &c = S.sp;
  const int lane = threadIdx.x;
  const int kd = ufi(c.kappa_dih);
  const int ifrag = (int)((G.order >> (4 * i)) & 15u);
  const int nfa = ufi(c.frag_natoms[ifrag]);
  const int at = c.frag_atoms[ifrag][min(lane, kCbA - 1)];
  const unsigned fmask = (unsigned)ufi((int)c.frag_mask[ifrag]);
  double lx = 0.0, ly = 0.0, lz = 0.0;
  if (del_flag) {
    if (lane < nfa) {
      lx = S.x[at];
      ly = S.y[at];
      lz = S.z[at];
    }
  } else {
    (void)draw(S, G);  // drawn twice, as written (:1578, :1584)
    const int nconf = ufi(c.nconfig[ifrag]);
    const int conf = ufi(min((int)(draw(S, G) * nconf), nconf - 1));
    const double *lib = c.lib + c.lib_off[ifrag] + (size_t)conf * nfa * 3;
    if (lane < nfa) {
      lx = lib[3 * lane];
      ly = lib[3 * lane + 1];
      lz = lib[3 * lane + 2];
    }
  }
  grown = G.ex;
  newx = (G.ex | fmask) & ~grown;
  G.ex |= fmask;
  // the first placed neighbour and the two anchors
  const int conn = c.frag_connect[ifrag][min(lane, kCbF - 1)];
  const uint64_t pl = __builtin_amdgcn_ballot_w64(lane < c.frag_nconnect[ifrag] && ((G.placed >> (conn & 31)) & 1u));
  const int fconn = __builtin_amdgcn_readlane(conn, pl ? (int)__builtin_ctzll(pl) : 0);
  const int anc_i = ufi(c.frag_anchor[ifrag]), anc_c = ufi(c.frag_anchor[fconn]);
  const int nfc = ufi(c.frag_natoms[fconn]);
  const int atc = c.frag_atoms[fconn][min(lane, kCbA - 1)];
  const bool isnew = lane < nfa && at != anc_i && at != anc_c;
  const uint64_t bn = __builtin_amdgcn_ballot_w64(isnew);
  const uint64_t bc = __builtin_amdgcn_ballot_w64(lane < nfc && atc != anc_i && atc != anc_c);
  const int ntat = __popcll(bn), pos = __popcll(bn & ((1ull << lane) - 1ull));
  const int atom_if = __builtin_amdgcn_readlane(at, bn ? (int)__builtin_ctzll(bn) : nfa - 1);
  const int atom_fc = __builtin_amdgcn_readlane(atc, bc ? (int)__builtin_ctzll(bc) : nfc - 1);
  if (lane < kCbA) {
    S.tpos[lane] = -1;
    S.cx[lane] = S.cy[lane] = S.cz[lane] = 0.0;
  }
  wave_sync();
  if (isnew) {
    S.tpos[at] = pos;
    S.tatom[pos] = at;
  }
  if (lane < nfa) {
    S.cx[at] = lx;
    S.cy[at] = ly;
    S.cz[at] = lz;
  }
  wave_sync();
  // Get_Aligner_Hanger of the library frame on lane 0, of the grown part's
  // on lane 1 (of the fragment's own frame in a deletion)
  const bool own = lane == 1 && !del_flag;
  const double *px = own ? S.x : S.cx, *py = own ? S.y : S.cy, *pz = own ? S.z : S.cz;
  const int a3 = own ? atom_fc : atom_if;
  const double x0 = px[anc_c], y0 = py[anc_c], z0 = pz[anc_c];
  double v1[3] = {__dsub_rn(px[anc_i], x0), __dsub_rn(py[anc_i], y0), __dsub_rn(pz[anc_i], z0)};
  double v2[3] = {__dsub_rn(px[a3], x0), __dsub_rn(py[a3], y0), __dsub_rn(pz[a3], z0)};
  double al[3][3], ha[3][3];
  aligner_hanger(v1, v2, al, ha);
  const double tx0 = readlane_f64(x0, 0), ty0 = readlane_f64(y0, 0), tz0 = readlane_f64(z0, 0);
#pragma unroll
  for (int r = 0; r < 3; ++r)
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      al[r][q] = readlane_f64(al[r][q], 0);
      ha[r][q] = readlane_f64(ha[r][q], 1);
    }
  const double bx = S.x[anc_c], by = S.y[anc_c], bz = S.z[anc_c];
  const double rx = __dsub_rn(lx, tx0), ry = __dsub_rn(ly, ty0), rz = __dsub_rn(lz, tz0);
  wave_sync();
  if (isnew) {
    S.cx[pos] = mrow(al[0], rx, ry, rz);
    S.cy[pos] = mrow(al[1], rx, ry, rz);
    S.cz[pos] = mrow(al[2], rx, ry, rz);
  }
  wave_sync();
  double th = del_flag ? 0.0 : __dmul_rn(kTwoPi, draw(S, G)), my = th;
  const double step = S.thstep;
  for (int t = 1; t < kd; ++t) {
    th = __dadd_rn(th, step);
    if (lane == t) my = th;
  }
  if (lane < kd) {
    double st, ct;
    sincos(my, &st, &ct);
    for (int p = 0; p < ntat; ++p) {
      const double x = S.cx[p], cy = S.cy[p], cz = S.cz[p];
      const double y = __dadd_rn(__dmul_rn(ct, cy), __dmul_rn(st, cz));
      const double z = __dadd_rn(__dmul_rn(-st, cy), __dmul_rn(ct, cz));
      S.tx[lane][p] = __dadd_rn(mrow(ha[0], x, y, z), bx);
      S.ty[lane][p] = __dadd_rn(mrow(ha[1], x, y, z), by);
      S.tz[lane][p] = __dadd_rn(mrow(ha[2], x, y, z), bz);
    }
    // COM of the added atoms
    S.tcom[lane] = com_of(c, S, lane, newx);
  }
  if (lane == 0) {
    S.ntatom = ntat;
    S.rpos = G.rpos;
  }
}

// Fragment_Placement (fragment_growth.f90:1449-2132) of the fragments
// i0 .. ntotal of the growth order: each is attached to its first placed
// neighbour at kappa_dih rotations about the connecting bond, scored
// (intramolecular, dihedral and CBMC-cutoff intermolecular terms against
// e_prev, the dihedral energy before the fragment) and one rotation drawn by
// its Boltzmann weight; with del_flag trial 1 is the fragment's own
// placement.  Every thread calls it; S.flag = cbmc_overlap after the caller's
// next barrier (or set before: nothing is placed), G.ln_pbias accumulates.
template <typename P, int NT, bool LJ>
__device__ __forceinline__ void fragment_placement(const GrowArgs &a, GrowLds<NT> &S, GrowReg &G,
                                                                  const LiveList &l, int nl, int self, bool del_flag,
                                                                  int i0, double e_prev) {
  const CbmcSpeciesDev &c = S.sp;
  const int lane = threadIdx.x;
  const int kd = ufi(c.kappa_dih);
  // uniform over the workgroup: written by wave 0 before the last barrier
  const int ntotal = ufi(S.ntotal);
  for (int i = i0; i < ntotal; ++i) {
    unsigned newx = 0, oldx = 0;
    if (lane < 64 && !ufi(S.flag)) fragment_trials(a, S, G, i, del_flag, newx, oldx);
    if (fill_wave<NT>()) ring_fill(S);
    __syncthreads();
    if (ufi(S.flag)) return;
    // wave 0: each trial's intramolecular energy (the added atoms one by one
    // with the atoms placed so far) and dihedrals, while the others score
    double iv = 0.0, iq = 0.0, iqi = 0.0, ed = 0.0;
    int intra_ov = 0;
    if (lane < 64) {
      const int t = min(lane, kd - 1);
      unsigned ex = oldx;
      const int ntat = ufi(S.ntatom);
      for (int p = 0; p < ntat; ++p) {
        const int at = ufi(S.tatom[p]);
        ex |= 1u << at;
        double ev, eq, eqi;
        const bool o = atom_intra<NT, LJ>(a, c, S, t, at, ex, ev, eq, eqi);
        if (o) intra_ov = 1;
        if (!intra_ov) {
          iv = __dadd_rn(iv, ev);
          iq = __dadd_rn(iq, eq);
          iqi = __dadd_rn(iqi, eqi);
        }
      }
      ed = dihedral_energy(c, S, t, G.ex);
    }
    stage_trials<P, NT, LJ>(a, S, l, nl, kd, self, true);
    __syncthreads();
    // the trial's energy and weight (fragment_growth.f90:2014-2056), one lane
    // per trial; selection (:2074-2099)
    if (lane < 64) {
      double w = 0.0, e = 0.0;
      int wk = 1;
      if (lane < kd) {
        const int ov = intra_ov ? 2 : S.sov[lane];
        // an overlapping trial's dihedrals are not taken (:2030-2044): the next
        // fragment starts from 0 where a deletion keeps one
        if (ov) ed = 0.0;
        if (!ov) {
          const double qsum = __dadd_rn(iqi, S.sq[lane]);
          e = __dsub_rn(__dadd_rn(__dadd_rn(__dadd_rn(__dadd_rn(ed, iv), iq), S.sv[lane]), qsum), e_prev);
          const double bk = __dmul_rn(a.beta, e);
          if (!(bk >= kMaxKBT)) {
            w = exp(-bk);
            wk = 0;
          }
        } else if (ov == 2) {
          wk = 2;  // intramolecular overlap: the cumulative weight carries over
        }
      }
      double wsum;
      const int trial = select_trial(S, G, kd, w, wk, del_flag, wsum);
      if (trial < 0) {
        if (lane == 0) S.flag = 1;
      } else {
        G.ln_pbias = __dsub_rn(__dsub_rn(G.ln_pbias, __dmul_rn(a.beta, readlane_f64(e, trial))), log(wsum));
        if (lane < S.ntatom) {
          const int at = S.tatom[lane];
          S.x[at] = S.tx[trial][lane];
          S.y[at] = S.ty[trial][lane];
          S.z[at] = S.tz[trial][lane];
        }
        G.placed |= 1u << ((G.order >> (4 * i)) & 15u);
        e_prev = readlane_f64(ed, trial);
      }
      wave_sync();
    }
  }
}

// ln_pbias of the caller after Build_Molecule (widom_insert.f90:361-370,
// move_insert.f90:166-180, move_delete.f90:196-210); wave 0.
template <int NT>
__device__ __forceinline__ double ln_pbias_total(const GrowLds<NT> &S, const GrowReg &G) {
  double v = __dadd_rn(G.ln_pbias, G.ln_pseq);
  v = __dadd_rn(v, S.lk[0]);
  if (S.sp.kappa_rot != 0) v = __dadd_rn(v, S.lk[1]);
  if (S.sp.kappa_dih != 0) v = __dadd_rn(v, S.lk[2]);
  return v;
}

// After the growth (wave 0): every atom exists; the grown molecule's centre,
// Fold_Molecule (minimum_image_separation.f90:162-260, cubic boxes) with
// `fold`, and the set-up of the full-cutoff stage.  again: the centre taken
// once more after the fold, where the caller does so.
template <int NT>
__device__ __forceinline__ void whole_molecule(const GrowArgs &a, GrowLds<NT> &S, GrowReg &G, bool grown_com, bool fold,
                                      bool again) {
  const CbmcSpeciesDev &c = S.sp;
  const int lane = threadIdx.x, n = ufi(c.natoms);
  G.ex = (1u << n) - 1u;
  const int k = min(lane, kCbA - 1);
  double x = S.x[k], y = S.y[k], z = S.z[k];
  double4 com = S.com;
  if (grown_com) com = com_wave(c, G.ex, x, y, z);
  if (fold && a.b.cubic) {
    auto axis = [&](double &cc, double &q, int d) {
      if (cc > a.b.hL[d]) {
        cc = __dsub_rn(cc, a.b.L[d]);
        q = __dsub_rn(q, a.b.L[d]);
      } else if (cc < -a.b.hL[d]) {
        cc = __dadd_rn(cc, a.b.L[d]);
        q = __dadd_rn(q, a.b.L[d]);
      }
    };
    axis(com.x, x, 0);
    axis(com.y, y, 1);
    axis(com.z, z, 2);
    if (lane < n) {
      S.x[lane] = x;
      S.y[lane] = y;
      S.z[lane] = z;
    }
  }
  if (again) com = com_wave(c, G.ex, x, y, z);
  wave_sync();
  if (lane == 0) {
    S.com = com;
    S.rpos = G.rpos;
  }
}

// ---------------------------------------------------------------- Widom
struct WidomCbmcArgs {
  GrowArgs g;
  int64_t n_ins;
  uint64_t seed;
  int sequential;       // one workgroup, the reference's stream in rng
  int64_t *rng;         // 5 words (sequential mode), in/out
  double e_const;       // lrc_diff + E_self - E_recip_in
  double *wvar;         // [n_ins]
  uint8_t *over;        // [n_ins]
  double *eij_max;      // [n_ins] or null: est_emax's Eij_max (0 where over)
  double *rsq_min;      // [n_ins][rsq_rows][natoms] or null: closest r^2 per
  int rsq_rows;         // (species site, inserted atom), 10000 if none in range
  LiveList live;        // the frame's live molecules (k_widom_live)
  int *nlive;
};

// The per-insertion LFSR of the parallel mode: five components from
// (seed, insertion), each with the bits its shift masks keep non-zero.
__device__ __forceinline__ int64_t seed_word(uint64_t seed, uint64_t i, int k) {
  const int64_t lo = k == 0 ? 2 : (k == 1 ? 512 : (k == 2 ? 4096 : (k == 3 ? 131072 : 8388608)));
  const uint64_t h = mix64(mix64(seed ^ (i * 0xD1B54A32D192ED03ull)) + 0x9E37ull * (uint64_t)(k + 1));
  return (int64_t)(h | (uint64_t)lo << 1);
}

template <typename P, int NT, bool LJ>
__global__ void __launch_bounds__(NT) k_widom_cbmc(WidomCbmcArgs w) {
  __shared__ GrowLds<NT> S;
  const CbmcSpeciesDev &c = S.sp;
  const int lane = threadIdx.x;
  const int64_t i0 = w.sequential ? 0 : (int64_t)blockIdx.x;
  const int64_t i1 = w.sequential ? w.n_ins : i0 + 1;
  const int nl = *w.nlive;
  load_tables(S, w.g.sp, w.g.tp);
  if (lane < 5) S.rw[lane][0] = w.sequential ? vld(w.rng + lane) : seed_word(w.seed, (uint64_t)i0, lane);
  if (lane == 0) S.rgen = S.rpos = 0;
  __syncthreads();
  if (fill_wave<NT>()) ring_fill(S);
  __syncthreads();
  GrowReg G{};
  for (int64_t i = i0; i < i1; ++i) {
    if (lane < 64) first_fragment(w.g, S, G, false, false);
    __syncthreads();
    build_molecule<P, NT, LJ>(w.g, S, G, w.live, nl, -1, false);
    // the full-cutoff energy of the grown molecule (widom_insert.f90:378-399)
    if (lane < 64 && !ufi(S.flag)) whole_molecule(w.g, S, G, G.ntotal > 1, c.nfrag > 1, false);
    if (lane == 0) S.rpos = G.rpos;
    if (fill_wave<NT>()) ring_fill(S);
    if (w.rsq_min) {
      // swi_atompair_rsqmin = 10000 for every insertion (widom_insert.f90:325)
      double *rm = w.rsq_min + i * (int64_t)w.rsq_rows * c.natoms;
      for (int k = lane; k < w.rsq_rows * c.natoms; k += NT) rm[k] = 10000.0;
      if (lane == 0) S.rsq = rm;
    }
    __syncthreads();
    const int cov = ufi(S.flag);
    double iv = 0.0, iq = 0.0, ip = 0.0, e_ang = 0.0, e_dih = 0.0;
    bool intra_ov = false;
    if (!cov) {
      if (lane < 64) intra_ov = mol_terms_wave<NT, LJ>(w.g, c, S, iv, iq, ip, e_ang, e_dih);
      if (w.eij_max)
        stage_full<P, NT, LJ, true>(w.g, S, w.live, nl, -1);
      else
        stage_full<P, NT, LJ>(w.g, S, w.live, nl, -1);
    }
    __syncthreads();
    if (lane < 64) {
      double wv = 0.0;
      int ov = 1;
      if (!cov) {
        double ev, eq;
        const bool sov = full_sums<NT, true>(S, ev, eq);
        if (!sov && !intra_ov) {
          const double e_inter = __dadd_rn(__dadd_rn(ev, eq), ip);
          const double ln_pbias = ln_pbias_total(S, G);
          const double de_inter = __dadd_rn(e_inter, w.e_const);
          double de_intra = __dadd_rn(iv, iq);
          de_intra = __dadd_rn(__dadd_rn(__dadd_rn(__dadd_rn(de_intra, 0.0), e_ang), e_dih), 0.0);
          const double de = __dadd_rn(de_intra, de_inter);
          const double de_frag = __dadd_rn(e_ang, 0.0);
          wv = exp(__dsub_rn(-__dmul_rn(w.g.beta, __dsub_rn(de, de_frag)), ln_pbias));
          ov = 0;
        }
      }
      wave_sync();
      if (lane == 0) {
        w.wvar[i] = wv;
        w.over[i] = (uint8_t)ov;
        if (w.eij_max) w.eij_max[i] = ov ? 0.0 : S.sem;
      }
    }
  }
  if (w.sequential && lane < 5) w.rng[lane] = S.rw[lane][G.rpos & (kRing - 1)];
}

// ----------------------------------------------------------------- GCMC
// Per box of the chain kernel.
struct GcmcBoxArgs {
  GrowArgs g;
  double *x, *y, *z;  // the box's coordinates (the memory of g.b.x/y/z)
  double4 *comd;      // (COM, max_dcom) per slot
  int *live;          // per slot
  int first_slot, max_mols;
  double prob_insert, mu, lambda, log_volume;
  // state, in/out
  int64_t *rng;       // 5
  double *energy;     // cass_energy as 14 doubles
  int *nmols, *nres, *locate, *reservoir;
  double *nbeads;     // per type
  double volume, rcut3, rcut9, rcut_vdw;
  int vdw_style, tail;
  int commit;  // 0: a timing run that leaves the box untouched
  LiveList list;  // device memory for the live list, where LDS is too small
  // records [nsteps] per box, or null
  uint8_t *kind, *accepted;
  int *rec_nmols;
  double *rec_energy;
  int64_t *rec_rng;
};

enum { kE_total = 0, kE_intra, kE_inter, kE_bond, kE_angle, kE_dihedral, kE_improper, kE_intra_vdw, kE_intra_q,
       kE_inter_vdw, kE_lrc, kE_inter_q, kE_reciprocal, kE_self };

// The bracket of Compute_LR_Correction for a type pair.
__device__ __forceinline__ double lrc_bracket(double sig, double rcut3, double rcut9) {
  const double s2 = __dmul_rn(sig, sig), s6 = __dmul_rn(__dmul_rn(s2, s2), s2), s12 = __dmul_rn(s6, s6);
  return __dsub_rn(__ddiv_rn(s12, __dmul_rn(9.0, rcut9)), __ddiv_rn(s6, __dmul_rn(3.0, rcut3)));
}

// Compute_LR_Correction (energy_routines.f90:2956-3023) by wave 0, lane t
// holding the bead count nb of type t: a lane per type's row, the rows added
// in order.  br: the brackets of the type pairs (LDS) where the topology fits
// the LDS tables.
template <int NT>
__device__ __forceinline__ double lrc_wave(const GcmcBoxArgs &a, const GrowLds<NT> &S, const double *br, double nb) {
  if (a.vdw_style != CASS_VDW_LJ) return 0.0;
  const TopoDev &tp = a.g.tp;
  const int lane = threadIdx.x, nt = ufi(tp.ntypes);
  const bool ok = S.ct.ok != 0;
  const int i = min(lane, nt - 1);
  double eij = 0.0;
  for (int j = 0; j < nt; ++j) {
    const int k = i * nt + j;
    const double eps = ok ? S.ct.eps[k] : tp.eps[k];
    const double b = ok ? br[k] : lrc_bracket(tp.sig[k], a.rcut3, a.rcut9);
    eij = __dadd_rn(eij, __dmul_rn(__dmul_rn(__dmul_rn(readlane_f64(nb, j), 4.0), eps), b));
  }
  const double row = __dmul_rn(nb, eij);
  double el = 0.0;
  for (int t = 0; t < nt; ++t) el = __dadd_rn(el, readlane_f64(row, t));
  return __ddiv_rn(__dmul_rn(__dmul_rn(2.0, kPi), el), a.volume);
}

template <int NT>
__device__ __forceinline__ void lrc_tables(const GcmcBoxArgs &a, const TopoDev &tp, double *br) {
  if (tp.nspecies > kCtSp || tp.natoms_total > kCtAt || tp.ntypes > kCtT) return;
  for (int k = threadIdx.x; k < tp.ntypes * tp.ntypes; k += NT) br[k] = lrc_bracket(tp.sig[k], a.rcut3, a.rcut9);
}

// The beads of type `lane` in the grown species.
__device__ __forceinline__ double type_beads(const CbmcSpeciesDev &c) {
  const int n = ufi(c.natoms);
  double v = 0.0;
  for (int k = 0; k < n; ++k)
    if (c.type[k] == (int)threadIdx.x) v += 1.0;
  return v;
}

// accept_or_reject (accept_or_reject.f90:22-65); wave 0.
template <int NT>
__device__ __forceinline__ int accept_or_reject(const GrowLds<NT> &S, GrowReg &G, double lp) {
  if (lp <= 0.0) return 1;
  return lp < kMaxKBT && draw(S, G) <= exp(-lp) ? 1 : 0;
}

// Where a chain kernel keeps its lists: cap > 0: in the dynamic LDS, per box
// the centres, the entries, then (gcmc) locate and reservoir.
constexpr size_t kCentre = 4 * sizeof(double);
constexpr size_t kListBytes = kCentre + sizeof(LiveMol) + 2 * sizeof(int);
__device__ __forceinline__ LiveList chain_list(char *dyn, int cap, int box, const LiveList &g) {
  if (cap == 0) return g;
  char *p = dyn + (size_t)box * cap * kListBytes;
  return LiveList{(LiveMol *)(p + kCentre * cap), (double *)p, cap};
}
__device__ __forceinline__ int *chain_slots(char *dyn, int cap, int box, int which) {
  return (int *)(dyn + (size_t)box * cap * kListBytes + (kCentre + sizeof(LiveMol)) * cap) + which * cap;
}

// Removes entry im of locate[0 .. n): the later ones move down (whole wave).
__device__ __forceinline__ void locate_remove(int *locate, int im, int n) {
  const int wl = threadIdx.x & 63;
  for (int k0 = im + 1; k0 < n; k0 += 64) {
    const int k = k0 + wl;
    const int v = k < n ? *(volatile int *)(locate + k) : 0;
    wave_sync();
    if (k < n) *(volatile int *)(locate + k - 1) = v;
    wave_sync();
  }
}

// A molecule joins or leaves the live list (wave 0).
__device__ __forceinline__ void list_add(const LiveList &l, int &n, const BoxDev &b, int m, double4 com) {
  if (threadIdx.x == 0) {
    l.mol[n] = LiveMol{m, (b.first[m] << 4) | (b.species[m] & 15)};
    l.put(n, com);
  }
  ++n;
}
__device__ __forceinline__ void list_drop(const LiveList &l, int &n, int m) {
  const int p = live_find(l, n, m);
  if (p < 0) return;
  --n;
  if (threadIdx.x == 0) {
    l.mol[p] = l.mol[n];
    l.put(p, l.centre(n));
  }
}
__device__ __forceinline__ void list_move(const LiveList &l, int n, int m, double4 com) {
  const int p = live_find(l, n, m);
  if (p >= 0 && threadIdx.x == 0) l.put(p, com);
}

// Copies a slot list between device memory and LDS (wave 0).
__device__ __forceinline__ void copy_slots(int *dst, const int *src, int n) {
  for (int k = threadIdx.x; k < n; k += 64) *(volatile int *)(dst + k) = *(const volatile int *)(src + k);
}

// One workgroup per box.  Wave 0 makes the draws, the growth's geometry and
// the acceptance, with the box's bookkeeping in its registers and lists in
// LDS; every wave takes trials in the stages, wave 1 keeps the draws ready.
// A move is a chain of dependent stages on one CU, bound by latency.  Serial
// work of one lane was two thirds of it, and scratch traffic of the general
// pair styles much of the rest: now what can be spread over the lanes of wave
// 0 is, barriers stand only between stages, and plain LJ species have kernels
// of their own without scratch.  40 moves in 48 pentane boxes (kappa 12 / 24,
// up to 233 molecules): 7.5 ms before, 2.4 ms now, or 188 and 60 us a move of
// the slowest box; in boxes that have settled 5.7 and 1.4 ms, 143 and 35 us a
// move.  The vector units of the CUs in use are busy 17 % of the time.
template <typename P, int NT, bool LJ>
__global__ void __launch_bounds__(NT) k_gcmc_chain(const GcmcBoxArgs *__restrict__ boxes, int64_t nsteps,
                                                   int list_cap) {
  __shared__ GrowLds<NT> S;
  __shared__ double E[14];
  __shared__ double br[kCtT * kCtT];
  __shared__ int q_lm, q_kind, q_skip, q_nl;
  extern __shared__ __align__(16) char dyn[];
  const GcmcBoxArgs &a = boxes[blockIdx.x];
  const CbmcSpeciesDev &c = S.sp;
  const int lane = threadIdx.x;
  const int nt = a.g.tp.ntypes;
  const LiveList l = chain_list(dyn, list_cap, 0, a.list);
  int *locate = list_cap ? chain_slots(dyn, list_cap, 0, 0) : a.locate;
  int *reservoir = list_cap ? chain_slots(dyn, list_cap, 0, 1) : a.reservoir;
  load_tables(S, a.g.sp, a.g.tp);
  lrc_tables<NT>(a, a.g.tp, br);
  ring_start(S, a.rng);
  if (lane < 14) E[lane] = vld(a.energy + lane);
  // wave 0's registers
  GrowReg G{};
  int nmols = 0, nres = 0, nl = 0, stop = 0;
  int64_t done = 0;  // moves recorded
  double nb = 0.0, beads = 0.0;
  if (lane < 64) {
    nmols = ufi(vld(a.nmols));
    nres = ufi(vld(a.nres));
    nl = build_live_list<NT>(a.g, l);
    if (list_cap) {
      copy_slots(locate, a.locate, nmols);
      copy_slots(reservoir, a.reservoir, nres);
    }
    if (lane < nt) nb = vld(a.nbeads + lane);
    if (lane == 0) q_nl = nl;
  }
  __syncthreads();
  if (lane < 64) beads = type_beads(c);
  if (fill_wave<NT>()) ring_fill(S);
  __syncthreads();
  const double beta = a.g.beta;
  const int natoms = ufi(c.natoms);
  const double lam3 = __dmul_rn(3.0, log(a.lambda));
  for (int64_t st = 0; st < nsteps; ++st) {
    // the move draw, the species draw, the molecule slot and the first
    // fragment's trials
    int im = 0;
    if (lane < 64) {
      int skip = stop ? 2 : 0, kind = 0, lm = 0;
      if (!stop) {
        const double u = draw(S, G);
        kind = ufi(u <= a.prob_insert ? 0 : 1);
        (void)draw(S, G);  // is_rand: one sorbate species (move_insert.f90:108, move_delete.f90:99)
        if (kind == 0) {
          if (nres == 0) {
            skip = 2;  // max_molecules reached: the reference aborts
            stop = 1;
          } else {
            lm = ufi(*(volatile int *)(reservoir + nres - 1));
            nres--;
            if (lane == 0) *(volatile int *)(locate + nmols) = lm;
            nmols++;
          }
        } else if (nmols == 0) {
          skip = 1;
        } else {
          im = ufi(min((int)(draw(S, G) * nmols), nmols - 1));
          lm = ufi(*(volatile int *)(locate + im));
          const int f = a.g.b.first[a.first_slot + lm];
          if (lane < natoms) {
            S.x[lane] = vld(a.x + f + lane);
            S.y[lane] = vld(a.y + f + lane);
            S.z[lane] = vld(a.z + f + lane);
          }
          wave_sync();
        }
      }
      if (lane == 0) {
        q_skip = skip;
        q_kind = kind;
        q_lm = lm;
      }
      if (!skip) first_fragment(a.g, S, G, kind == 1, false);
    }
    __syncthreads();
    const int skip = ufi(q_skip);
    if (skip == 2) break;
    const bool del = ufi(q_kind) == 1;
    const int lm = ufi(q_lm), m = a.first_slot + lm;
    int acc = 0;
    if (skip) {
      if (lane == 0) S.rpos = G.rpos;
      __syncthreads();  // q_skip is read before the next move writes it
      if (fill_wave<NT>()) ring_fill(S);
      __syncthreads();
    } else {
      const int nlv = ufi(q_nl);
      build_molecule<P, NT, LJ>(a.g, S, G, l, nlv, m, del);
      if (lane < 64 && !ufi(S.flag)) whole_molecule(a.g, S, G, G.ntotal > 1, !del, true);
      if (lane == 0) S.rpos = G.rpos;
      if (fill_wave<NT>()) ring_fill(S);
      __syncthreads();
      const int cov = ufi(S.flag);
      // the whole molecule's intramolecular, angle and dihedral terms
      double iv = 0.0, iq = 0.0, ip = 0.0, e_ang = 0.0, e_dih = 0.0;
      bool intra_ov = false;
      if (!cov) {
        if (lane < 64) intra_ov = mol_terms_wave<NT, LJ>(a.g, c, S, iv, iq, ip, e_ang, e_dih);
        stage_full<P, NT, LJ>(a.g, S, l, nlv, m);
      }
      __syncthreads();
      if (lane < 64) {
        double ev = 0.0, eq = 0.0;
        bool sov = false;
        if (!cov) sov = full_sums<NT>(S, ev, eq);
        if (del && cov) {
          stop = 1;  // the molecule to delete cannot be regrown: the reference aborts
        } else if (!del && (cov || sov || intra_ov)) {
          nmols--;
          if (lane == 0) *(volatile int *)(reservoir + nres) = lm;
          nres++;
        } else {
          const double sgn = del ? -1.0 : 1.0;
          double de_inter, de_intra, e_lrc = 0.0, nb2 = nb;
          if (!del) {
            // Insertion (move_insert.f90:186-351)
            eq = __dadd_rn(eq, ip);
            de_inter = __dadd_rn(ev, eq);
            de_intra = __dadd_rn(iv, iq);
            de_intra = __dadd_rn(__dadd_rn(__dadd_rn(__dadd_rn(de_intra, 0.0), e_ang), e_dih), 0.0);
          } else {
            // Deletion (move_delete.f90:196-330)
            de_inter = __dsub_rn(-ev, eq);
            de_intra = __dsub_rn(__dsub_rn(__dsub_rn(-0.0, e_ang), e_dih), 0.0);
            eq = __dadd_rn(eq, ip);
            de_intra = __dsub_rn(__dsub_rn(de_intra, iv), iq);
            de_inter = __dsub_rn(de_inter, ip);
          }
          if (a.tail) {
            nb2 = __dadd_rn(nb, __dmul_rn(sgn, beads));
            e_lrc = lrc_wave<NT>(a, S, br, nb2);
            if (!del)
              de_inter = __dsub_rn(__dadd_rn(de_inter, e_lrc), E[kE_lrc]);
            else
              de_inter = __dadd_rn(de_inter, __dsub_rn(e_lrc, E[kE_lrc]));
          }
          const double de = __dadd_rn(de_intra, de_inter);
          const double de_frag = del ? __dsub_rn(-e_ang, 0.0) : __dadd_rn(e_ang, 0.0);
          const double ln_pbias = ln_pbias_total(S, G);
          double lp = __dmul_rn(beta, __dsub_rn(de, de_frag));
          if (!del) {
            lp = __dsub_rn(lp, __dmul_rn(a.mu, beta));
            lp = __dadd_rn(lp, ln_pbias);
            lp = __dadd_rn(__dadd_rn(lp, log((double)nmols)), lam3);
            lp = __dsub_rn(lp, a.log_volume);
          } else {
            lp = __dadd_rn(lp, __dmul_rn(beta, a.mu));
            lp = __dsub_rn(lp, ln_pbias);
            lp = __dsub_rn(__dsub_rn(lp, log((double)nmols)), lam3);
            lp = __dadd_rn(lp, a.log_volume);
          }
          acc = ufi(accept_or_reject(S, G, lp));
          // an accepted insertion is stored; a deletion's grown coordinates
          // (trial 1 of every stage) replace the stored ones as in the
          // reference
          if (a.commit && (del || acc)) {
            const int f = a.g.b.first[m];
            if (lane < natoms) {
              a.x[f + lane] = S.x[lane];
              a.y[f + lane] = S.y[lane];
              a.z[f + lane] = S.z[lane];
            }
            if (lane == 0) a.comd[m] = S.com;
          }
          if (acc) {
            if (lane == 0) {
              E[kE_total] = __dadd_rn(E[kE_total], de);
              E[kE_intra] = __dadd_rn(E[kE_intra], de_intra);
              E[kE_inter] = __dadd_rn(E[kE_inter], de_inter);
              E[kE_angle] = __dadd_rn(E[kE_angle], sgn * e_ang);
              E[kE_dihedral] = __dadd_rn(E[kE_dihedral], sgn * e_dih);
              E[kE_intra_vdw] = __dadd_rn(E[kE_intra_vdw], sgn * iv);
              E[kE_intra_q] = __dadd_rn(E[kE_intra_q], sgn * iq);
              E[kE_inter_vdw] = __dadd_rn(E[kE_inter_vdw], sgn * ev);
              E[kE_inter_q] = __dadd_rn(E[kE_inter_q], sgn * eq);
              if (a.tail) E[kE_lrc] = e_lrc;
              if (a.commit) a.live[m] = del ? 0 : 1;
            }
            nb = nb2;
            if (del) {
              locate_remove(locate, im, nmols);
              nmols--;
              if (lane == 0) *(volatile int *)(reservoir + nres) = lm;
              nres++;
              if (a.commit) list_drop(l, nl, m);
            } else if (a.commit) {
              list_add(l, nl, a.g.b, m, S.com);
            }
            if (lane == 0) q_nl = nl;
          } else if (!del) {
            nmols--;
            if (lane == 0) *(volatile int *)(reservoir + nres) = lm;
            nres++;
          }
        }
      }
    }
    if (lane < 64 && !stop) {
      done = st + 1;
      wave_sync();
      if (lane == 0) {
        if (a.kind) a.kind[st] = (uint8_t)(del ? 1 : 0);
        if (a.accepted) a.accepted[st] = (uint8_t)acc;
        if (a.rec_nmols) a.rec_nmols[st] = nmols;
        if (a.rec_energy) a.rec_energy[st] = E[kE_total];
      }
      if (a.rec_rng && lane < 5) a.rec_rng[5 * st + lane] = S.rw[lane][G.rpos & (kRing - 1)];
    }
  }
  if (lane < 64) {
    wave_sync();
    if (lane < 5) a.rng[lane] = S.rw[lane][G.rpos & (kRing - 1)];
    if (lane < 14) a.energy[lane] = E[lane];
    if (list_cap) {
      copy_slots(a.locate, locate, nmols);
      copy_slots(a.reservoir, reservoir, nres);
    }
    if (lane < nt) a.nbeads[lane] = nb;
    record_rest(a.kind, done, nsteps);
    record_rest(a.accepted, done, nsteps);
    record_rest(a.rec_nmols, done, nsteps);
    record_rest(a.rec_energy, done, nsteps);
    record_rest(a.rec_rng, 5 * done, 5 * nsteps);
    if (lane == 0) {
      *a.nmols = nmols;
      *a.nres = stop ? -1 : nres;
    }
  }
}

// ----------------------------------------------------------------- GEMC
// GEMC_Particle_Transfer (move_mol_swap.f90:22-769) between the two boxes of
// a pair, one workgroup per pair running the pair's whole sequence of moves
// (gemc_driver.f90:91-195 with transfers only: one move draw each).  Per
// move: box_out by molecule fraction, box_in the other box, the species draw
// (one sorbate), the molecule; Build_Molecule into box_in drawing the
// fragment order, its energies there (a core overlap of the grown molecule
// rejects); then the reverse Build_Molecule in box_out with the same order,
// its energies, and the acceptance with ln_pfor - ln_prev and
// log(P_forward / P_reverse).  The box_out molecule keeps its re-placed
// coordinates when rejected, as in the reference.  The pair's boxes are
// boxes[2 * blockIdx.x] and the next; the generator is the first box's.
// Waves as in k_gcmc_chain.  30 transfers in 96 pairs of pentane boxes (kappa
// 12 / 16): 8.1 ms before, 2.4 ms now.
template <typename P, int NT, bool LJ>
__global__ void __launch_bounds__(NT) k_gemc_chain(const GcmcBoxArgs *__restrict__ boxes, int64_t nsteps,
                                                   int list_cap) {
  __shared__ GrowLds<NT> S;
  __shared__ double E[2][14];
  __shared__ double br[2][kCtT * kCtT];
  __shared__ int q_bo, q_lm_out, q_lm_in, q_skip, q_go, q_nl[2];
  extern __shared__ __align__(16) char dyn[];
  const GcmcBoxArgs *A = boxes + 2 * blockIdx.x;
  const CbmcSpeciesDev &c = S.sp;
  const int lane = threadIdx.x;
  const int nt = A[0].g.tp.ntypes;
  const LiveList l0 = chain_list(dyn, list_cap, 0, A[0].list), l1 = chain_list(dyn, list_cap, 1, A[1].list);
  int *loc0 = list_cap ? chain_slots(dyn, list_cap, 0, 0) : A[0].locate;
  int *loc1 = list_cap ? chain_slots(dyn, list_cap, 1, 0) : A[1].locate;
  int *res0 = list_cap ? chain_slots(dyn, list_cap, 0, 1) : A[0].reservoir;
  int *res1 = list_cap ? chain_slots(dyn, list_cap, 1, 1) : A[1].reservoir;
  load_tables(S, A[0].g.sp, A[0].g.tp);
  lrc_tables<NT>(A[0], A[0].g.tp, br[0]);
  lrc_tables<NT>(A[1], A[1].g.tp, br[1]);
  ring_start(S, A[0].rng);
  if (lane < 28) E[lane / 14][lane % 14] = vld(A[lane / 14].energy + lane % 14);
  // wave 0's registers
  GrowReg G{};
  int nm0 = 0, nm1 = 0, nr0 = 0, nr1 = 0, stop = 0;
  int64_t done = 0;  // moves recorded
  double nb0 = 0.0, nb1 = 0.0, beads = 0.0;
  if (lane < 64) {
    nm0 = ufi(vld(A[0].nmols));
    nm1 = ufi(vld(A[1].nmols));
    nr0 = ufi(vld(A[0].nres));
    nr1 = ufi(vld(A[1].nres));
    const int n0 = build_live_list<NT>(A[0].g, l0), n1 = build_live_list<NT>(A[1].g, l1);
    if (list_cap) {
      copy_slots(loc0, A[0].locate, nm0);
      copy_slots(loc1, A[1].locate, nm1);
      copy_slots(res0, A[0].reservoir, nr0);
      copy_slots(res1, A[1].reservoir, nr1);
    }
    if (lane < nt) {
      nb0 = vld(A[0].nbeads + lane);
      nb1 = vld(A[1].nbeads + lane);
    }
    if (lane == 0) {
      q_nl[0] = n0;
      q_nl[1] = n1;
    }
  }
  __syncthreads();
  if (lane < 64) beads = type_beads(c);
  if (fill_wave<NT>()) ring_fill(S);
  __syncthreads();
  const int natoms = ufi(c.natoms);
  for (int64_t st = 0; st < nsteps; ++st) {
    // Steps 1-3: the draws, box_in's free slot, the molecule's coordinates,
    // and the first fragment's trials in box_in
    double xo = 0.0, yo = 0.0, zo = 0.0;  // lane k: atom k of the molecule in box_out
    double pf = 0.0, pr = 0.0, ln_pfor = 0.0;
    double xn = 0.0, yn = 0.0, zn = 0.0;  // lane k: atom k as grown into box_in
    double4 com_new = make_double4(0.0, 0.0, 0.0, 0.0);
    int im = 0;
    if (lane < 64) {
      int skip = 0, bo0 = 0, lm_out = 0, lm_in = 0;
      if (stop) {
        skip = 2;
      } else {
        (void)draw(S, G);  // the move draw: transfers only
        const int tot = nm0 + nm1;
        if (tot == 0) {
          skip = 2;  // no swappable molecules: the reference aborts
        } else {
          const double x0 = __ddiv_rn((double)nm0, (double)tot);
          bo0 = ufi(draw(S, G) <= x0 ? 0 : 1);  // x_box(2) = 1
          (void)draw(S, G);                     // box_in: the other box of two (:202-204)
          const int nmo = bo0 ? nm1 : nm0, nmi = bo0 ? nm0 : nm1, nri = bo0 ? nr0 : nr1;
          const double no = (double)nmo, ni1 = (double)(nmi + 1);
          pf = __ddiv_rn(__dmul_rn(1.0, no), (double)tot);
          pr = __ddiv_rn(__dmul_rn(1.0, ni1), (double)tot);
          (void)draw(S, G);  // the species: x_is(1) = 1
          pf = __ddiv_rn(__dmul_rn(pf, no), no);
          pr = __ddiv_rn(__dmul_rn(pr, ni1), ni1);
          im = ufi(min((int)(draw(S, G) * nmo), nmo - 1));
          const GcmcBoxArgs &Ao = A[bo0];
          lm_out = ufi(*(volatile int *)((bo0 ? loc1 : loc0) + im));
          const int f = Ao.g.b.first[Ao.first_slot + lm_out];
          if (lane < natoms) {
            xo = vld(Ao.x + f + lane);
            yo = vld(Ao.y + f + lane);
            zo = vld(Ao.z + f + lane);
          }
          if (nri == 0) {
            skip = 2;  // box_in has no free slot
          } else {
            lm_in = ufi(*(volatile int *)((bo0 ? res0 : res1) + nri - 1));
            if (lane == 0) *(volatile int *)((bo0 ? loc0 : loc1) + nmi) = lm_in;
            if (bo0) {
              nr0--;
              nm0++;
            } else {
              nr1--;
              nm1++;
            }
          }
        }
        if (skip) stop = 1;
      }
      if (lane == 0) {
        q_skip = skip;
        q_bo = bo0;
        q_lm_out = lm_out;
        q_lm_in = lm_in;
      }
      if (!skip) first_fragment(A[1 - bo0].g, S, G, false, false);
    }
    __syncthreads();
    if (ufi(q_skip) == 2) break;
    const int bo = ufi(q_bo), bi = 1 - bo;
    const GcmcBoxArgs &Ai = A[bi], &Ao = A[bo];
    const LiveList li = bi ? l1 : l0, lo = bo ? l1 : l0;
    const int nli = ufi(q_nl[bi]), nlo = ufi(q_nl[bo]);
    const int lm_in = ufi(q_lm_in), lm_out = ufi(q_lm_out);
    const int m_in = Ai.first_slot + lm_in, m_out = Ao.first_slot + lm_out;
    int acc = 0;
    // Step 4: the molecule grown into box_in
    build_molecule<P, NT, LJ>(Ai.g, S, G, li, nli, m_in, false);
    if (lane < 64 && !ufi(S.flag)) whole_molecule(Ai.g, S, G, true, true, false);
    if (lane == 0) S.rpos = G.rpos;
    if (fill_wave<NT>()) ring_fill(S);
    __syncthreads();
    const int cov = ufi(S.flag);
    double iv = 0.0, iq = 0.0, ip = 0.0, e_ang = 0.0, e_dih = 0.0;
    if (!cov) {
      if (lane < 64) (void)mol_terms_wave<NT, LJ>(Ai.g, c, S, iv, iq, ip, e_ang, e_dih);
      stage_full<P, NT, LJ>(Ai.g, S, li, nli, m_in);
    }
    __syncthreads();
    // Step 5: box_in's change (intra_overlap is not acted on, :375-393)
    double ti_intra = 0.0, ti_inter = 0.0, ti_ev = 0.0, ti_eq = 0.0, lrc_in = 0.0;
    if (lane < 64) {
      double ev = 0.0, eq = 0.0;
      bool sov = false;
      if (!cov) sov = full_sums<NT>(S, ev, eq);
      int go = 0;
      if (cov || sov) {
        if (lane == 0) *(volatile int *)((bi ? res1 : res0) + (bi ? nr1 : nr0)) = lm_in;
        if (bi) {
          nm1--;
          nr1++;
        } else {
          nm0--;
          nr0++;
        }
      } else {
        go = 1;
        ti_inter = __dadd_rn(ev, eq);
        ti_intra = __dadd_rn(__dadd_rn(__dadd_rn(0.0, e_ang), e_dih), 0.0);
        eq = __dadd_rn(eq, ip);
        ti_intra = __dadd_rn(__dadd_rn(ti_intra, iv), iq);
        ti_inter = __dadd_rn(ti_inter, ip);
        if (Ai.tail) {
          lrc_in = lrc_wave<NT>(Ai, S, br[bi], __dadd_rn(bi ? nb1 : nb0, beads));
          ti_inter = __dsub_rn(__dadd_rn(ti_inter, lrc_in), E[bi][kE_lrc]);
        }
        ti_ev = ev;
        ti_eq = eq;
        ln_pfor = G.ln_pbias;
        const int k = min(lane, kCbA - 1);
        xn = S.x[k];
        yn = S.y[k];
        zn = S.z[k];
        com_new = S.com;
        wave_sync();
        if (lane < natoms) {
          S.x[lane] = xo;
          S.y[lane] = yo;
          S.z[lane] = zo;
        }
        wave_sync();
        // Step 6: the reverse growth in box_out with the forward order
        first_fragment(Ao.g, S, G, true, true);
      }
      if (lane == 0) {
        q_go = go;
        S.rpos = G.rpos;
      }
    }
    __syncthreads();
    const int go = ufi(q_go);
    if (go) {
      build_molecule<P, NT, LJ>(Ao.g, S, G, lo, nlo, m_out, true);
      if (lane < 64 && !ufi(S.flag)) whole_molecule(Ao.g, S, G, true, false, false);
      if (lane == 0) S.rpos = G.rpos;
      if (fill_wave<NT>()) ring_fill(S);
      __syncthreads();
      const int cov_out = ufi(S.flag);
      double ivo = 0.0, iqo = 0.0, ipo = 0.0, ango = 0.0, diho = 0.0;
      if (!cov_out) {
        if (lane < 64) (void)mol_terms_wave<NT, LJ>(Ao.g, c, S, ivo, iqo, ipo, ango, diho);
        stage_full<P, NT, LJ>(Ao.g, S, lo, nlo, m_out);
      }
      __syncthreads();
      if (lane < 64) {
        if (cov_out) {
          stop = 1;  // the molecule cannot be regrown in box_out: the reference aborts
        } else {
          double evo, eqo;
          (void)full_sums<NT>(S, evo, eqo);
          double de_intra_o = __dsub_rn(__dsub_rn(__dsub_rn(-0.0, ango), diho), 0.0);
          eqo = __dadd_rn(eqo, ipo);
          de_intra_o = __dsub_rn(__dsub_rn(de_intra_o, ivo), iqo);
          double de_inter_o = __dsub_rn(-evo, eqo);
          double lrc_out = 0.0;
          if (Ao.tail) {
            lrc_out = lrc_wave<NT>(Ao, S, br[bo], __dsub_rn(bo ? nb1 : nb0, beads));
            de_inter_o = __dadd_rn(de_inter_o, __dsub_rn(lrc_out, E[bo][kE_lrc]));
          }
          // Step 7 (:586-614)
          const double de_in = __dadd_rn(ti_intra, ti_inter);
          const double de_out = __dadd_rn(de_intra_o, de_inter_o);
          const double frag_in = __dadd_rn(e_ang, 0.0), frag_out = __dsub_rn(-ango, 0.0);
          double lp = __dadd_rn(__dmul_rn(Ai.g.beta, __dsub_rn(de_in, frag_in)),
                                __dmul_rn(Ao.g.beta, __dsub_rn(de_out, frag_out)));
          lp = __dadd_rn(__dsub_rn(lp, log((double)(bo ? nm1 : nm0))), log((double)(bi ? nm1 : nm0)));
          lp = __dsub_rn(lp, Ai.log_volume);
          lp = __dadd_rn(lp, Ao.log_volume);
          lp = __dadd_rn(__dsub_rn(__dadd_rn(lp, ln_pfor), G.ln_pbias), log(__ddiv_rn(pf, pr)));
          acc = ufi(accept_or_reject(S, G, lp));
          if (acc) {
            locate_remove(bo ? loc1 : loc0, im, bo ? nm1 : nm0);
            if (lane == 0) *(volatile int *)((bo ? res1 : res0) + (bo ? nr1 : nr0)) = lm_out;
            if (bo) {
              nm1--;
              nr1++;
              nb1 = __dsub_rn(nb1, beads);
              nb0 = __dadd_rn(nb0, beads);
            } else {
              nm0--;
              nr0++;
              nb0 = __dsub_rn(nb0, beads);
              nb1 = __dadd_rn(nb1, beads);
            }
            if (lane == 0) {
              E[bi][kE_total] = __dadd_rn(E[bi][kE_total], de_in);
              E[bi][kE_intra] = __dadd_rn(E[bi][kE_intra], ti_intra);
              E[bi][kE_inter] = __dadd_rn(E[bi][kE_inter], ti_inter);
              E[bi][kE_angle] = __dadd_rn(E[bi][kE_angle], e_ang);
              E[bi][kE_dihedral] = __dadd_rn(E[bi][kE_dihedral], e_dih);
              E[bi][kE_intra_vdw] = __dadd_rn(E[bi][kE_intra_vdw], iv);
              E[bi][kE_intra_q] = __dadd_rn(E[bi][kE_intra_q], iq);
              E[bi][kE_inter_vdw] = __dadd_rn(E[bi][kE_inter_vdw], ti_ev);
              E[bi][kE_inter_q] = __dadd_rn(E[bi][kE_inter_q], ti_eq);
              E[bo][kE_total] = __dadd_rn(E[bo][kE_total], de_out);
              E[bo][kE_intra] = __dadd_rn(E[bo][kE_intra], de_intra_o);
              E[bo][kE_inter] = __dadd_rn(E[bo][kE_inter], de_inter_o);
              E[bo][kE_angle] = __dsub_rn(E[bo][kE_angle], ango);
              E[bo][kE_dihedral] = __dsub_rn(E[bo][kE_dihedral], diho);
              E[bo][kE_intra_vdw] = __dsub_rn(E[bo][kE_intra_vdw], ivo);
              E[bo][kE_intra_q] = __dsub_rn(E[bo][kE_intra_q], iqo);
              E[bo][kE_inter_vdw] = __dsub_rn(E[bo][kE_inter_vdw], evo);
              E[bo][kE_inter_q] = __dsub_rn(E[bo][kE_inter_q], eqo);
              if (Ai.tail) E[bi][kE_lrc] = lrc_in;
              if (Ao.tail) E[bo][kE_lrc] = lrc_out;
            }
            if (Ai.commit) {
              const int fi = Ai.g.b.first[m_in];
              if (lane < natoms) {
                Ai.x[fi + lane] = xn;
                Ai.y[fi + lane] = yn;
                Ai.z[fi + lane] = zn;
              }
              if (lane == 0) {
                Ai.comd[m_in] = com_new;
                Ai.live[m_in] = 1;
                Ao.live[m_out] = 0;
              }
              int ni = nli, no = nlo;
              list_add(li, ni, Ai.g.b, m_in, com_new);
              list_drop(lo, no, m_out);
              if (lane == 0) {
                q_nl[bi] = ni;
                q_nl[bo] = no;
              }
            }
          } else {
            if (lane == 0) *(volatile int *)((bi ? res1 : res0) + (bi ? nr1 : nr0)) = lm_in;
            if (bi) {
              nm1--;
              nr1++;
            } else {
              nm0--;
              nr0++;
            }
            if (Ao.commit) {
              const int fo = Ao.g.b.first[m_out];
              if (lane < natoms) {
                Ao.x[fo + lane] = S.x[lane];
                Ao.y[fo + lane] = S.y[lane];
                Ao.z[fo + lane] = S.z[lane];
              }
              if (lane == 0) Ao.comd[m_out] = S.com;
            }
          }
        }
      }
    }
    if (lane < 64 && !stop) {
      done = st + 1;
      wave_sync();
      for (int b = 0; b < 2; ++b) {
        const GcmcBoxArgs &a = A[b];
        if (lane == 0) {
          if (a.kind) a.kind[st] = (uint8_t)bo;
          if (a.accepted) a.accepted[st] = (uint8_t)acc;
          if (a.rec_nmols) a.rec_nmols[st] = b ? nm1 : nm0;
          if (a.rec_energy) a.rec_energy[st] = E[b][kE_total];
        }
        if (a.rec_rng && lane < 5) a.rec_rng[5 * st + lane] = S.rw[lane][G.rpos & (kRing - 1)];
      }
    }
  }
  if (lane < 64) {
    wave_sync();
    for (int b = 0; b < 2; ++b) {
      const GcmcBoxArgs &a = A[b];
      if (lane < 5) a.rng[lane] = S.rw[lane][G.rpos & (kRing - 1)];
      if (lane < 14) a.energy[lane] = E[b][lane];
      if (list_cap) {
        copy_slots(a.locate, b ? loc1 : loc0, b ? nm1 : nm0);
        copy_slots(a.reservoir, b ? res1 : res0, b ? nr1 : nr0);
      }
      if (lane < nt) a.nbeads[lane] = b ? nb1 : nb0;
      record_rest(a.kind, done, nsteps);
      record_rest(a.accepted, done, nsteps);
      record_rest(a.rec_nmols, done, nsteps);
      record_rest(a.rec_energy, done, nsteps);
      record_rest(a.rec_rng, 5 * done, 5 * nsteps);
      if (lane == 0) {
        *a.nmols = b ? nm1 : nm0;
        *a.nres = stop ? -1 : (b ? nr1 : nr0);
      }
    }
  }
}

// ------------------------------------------------------------- regrowth
// Per box of the regrowth chain kernel.
struct RegrowBoxArgs {
  GrowArgs g;
  double *x, *y, *z;  // the box's coordinates (the memory of g.b.x/y/z)
  double4 *comd;      // (COM, max_dcom) per slot
  int first_slot, nmols;
  const int *locate;  // [nmols] slot offsets from first_slot
  LiveList list;      // device memory for the live list, where LDS is too small
  // state, in/out
  int64_t *rng;       // 5
  double *energy;     // cass_energy as 14 doubles
  int *status;        // 1: a molecule's own configuration could not be regrown
  // records [nsteps] per box, or null
  uint8_t *kind, *accepted;
  double *rec_energy, *ln_pacc;
  int64_t *rec_rng;
};

// Cut_Regrow's set-up (fragment_growth.f90:1118-1312); the whole of wave 0.
// Outside del_flag: the fragment bond to cut and the side to delete
// (fragment_bond_list%prob_del1), and the dead fragments' order
// (Fragment_Order from frag_dead with frag_live live).  Then every atom
// exists but those of the ordered fragments, the two anchors of the cut
// bond excepted, and the ordered fragments are not placed.
template <int NT>
__device__ __forceinline__ void cut_regrow_setup(const CbmcSpeciesDev &c, GrowLds<NT> &S, GrowReg &G, bool del_flag,
                                        int &frag_live, int &frag_dead) {
  G.ln_pbias = 0.0;
  G.ln_pseq = 0.0;
  const int nfrag = ufi(c.nfrag);
  if (!del_flag) {
    // rranf can round to 1.0 (random_generators.f90:118): the index is clamped
    const int nfb = ufi(c.nfbond);
    const int fb = ufi(min((int)(draw(S, G) * nfb), nfb - 1));
    const int side = ufi(draw(S, G) < c.prob_del1[fb] ? 0 : 1);
    frag_dead = ufi(c.fbond[fb][side]);
    frag_live = ufi(c.fbond[fb][1 - side]);
    G.order = (unsigned)frag_dead;
    G.ntotal = 1;
    fragment_order(c, S, G, frag_dead, (1u << frag_live) | (1u << frag_dead));
  }
  G.ex = (1u << ufi(c.natoms)) - 1u;
  G.placed = (1u << nfrag) - 1u;
  for (int i = 0; i < G.ntotal; ++i) {
    const int f = (int)((G.order >> (4 * i)) & 15u);
    G.placed &= ~(1u << f);
    G.ex &= ~(unsigned)ufi((int)c.frag_mask[f]);
  }
  G.ex |= 1u << ufi(c.frag_anchor[frag_live]);
  G.ex |= 1u << ufi(c.frag_anchor[frag_dead]);
  if (threadIdx.x == 0) {
    S.flag = 0;
    S.ntotal = G.ntotal;
  }
}

// Chains of Cut_N_Grow regrowth moves (move_regrow.f90:22-510), one
// workgroup per box, the box's whole move loop in one launch: per move the
// NVT driver's move draw, the box, species and molecule draws, the forward
// regrowth of the cut-off end (folded into the box), its full-cutoff
// energies, the reverse pass over the molecule's own configuration and the
// acceptance with ln_pfor - ln_prev.  Accepted: the regrown coordinates
// replace the molecule's; rejected after the reverse pass: its re-placed
// coordinates do, as in the reference.  Waves as in k_gcmc_chain.  60 moves
// in 48 pentane boxes (kappa 16): 6.5 ms before, 3.8 ms now.
template <typename P, int NT, bool LJ>
__global__ void __launch_bounds__(NT) k_regrow_chain(const RegrowBoxArgs *__restrict__ boxes, int64_t nsteps,
                                                     int list_cap) {
  __shared__ GrowLds<NT> S;
  __shared__ double E[14];
  __shared__ int q_m, q_state;  // q_state: 0 go on, 1 rejected, 2 stop
  extern __shared__ __align__(16) char dyn[];
  const RegrowBoxArgs &a = boxes[blockIdx.x];
  const CbmcSpeciesDev &c = S.sp;
  const int lane = threadIdx.x;
  const LiveList l = chain_list(dyn, list_cap, 0, a.list);
  load_tables(S, a.g.sp, a.g.tp);
  ring_start(S, a.rng);
  if (lane < 14) E[lane] = vld(a.energy + lane);
  __shared__ int q_nl;
  GrowReg G{};
  if (lane < 64) {
    const int n = build_live_list<NT>(a.g, l);
    if (lane == 0) q_nl = n;
  }
  __syncthreads();
  if (fill_wave<NT>()) ring_fill(S);
  __syncthreads();
  const int nl = ufi(q_nl), natoms = ufi(c.natoms);
  const double beta = a.g.beta;
  int state = 0;
  int64_t done = 0;  // moves recorded
  for (int64_t st = 0; st < nsteps; ++st) {
    int flive = 0, fdead = 0;
    double xo = 0.0, yo = 0.0, zo = 0.0;  // lane k: atom k as it was
    double e_prev0 = 0.0;
    if (lane < 64) {
      (void)draw(S, G);  // the move draw (nvtmc_driver.f90:109): regrowth only
      (void)draw(S, G);  // the box (one box: x_box(1) = 1)
      (void)draw(S, G);  // the species (one regrowable species)
      const int im = ufi(min((int)(draw(S, G) * a.nmols), a.nmols - 1));
      const int m0 = a.first_slot + a.locate[im];
      const int f = a.g.b.first[m0];
      if (lane < natoms) {
        S.x[lane] = xo = vld(a.x + f + lane);
        S.y[lane] = yo = vld(a.y + f + lane);
        S.z[lane] = zo = vld(a.z + f + lane);
      }
      wave_sync();
      cut_regrow_setup(c, S, G, false, flive, fdead);
      e_prev0 = dihedral_wave(c, S, G.ex);  // E_prev of the remaining atoms
      if (lane == 0) {
        q_m = m0;
        S.rpos = G.rpos;
      }
    }
    __syncthreads();
    const int m = ufi(q_m);
    fragment_placement<P, NT, LJ>(a.g, S, G, l, nl, m, false, 0, e_prev0);
    if (lane < 64 && !ufi(S.flag)) whole_molecule(a.g, S, G, true, true, false);
    if (lane == 0) S.rpos = G.rpos;
    if (fill_wave<NT>()) ring_fill(S);
    __syncthreads();
    const int cov = ufi(S.flag);  // cbmc_overlap: the old coordinates stay
    double n_iv = 0.0, n_iq = 0.0, n_ip = 0.0, n_ea = 0.0, n_ed = 0.0;
    if (!cov) {
      if (lane < 64)  // intra_overlap is not acted on
        (void)mol_terms_wave<NT, LJ>(a.g, c, S, n_iv, n_iq, n_ip, n_ea, n_ed);
      stage_full<P, NT, LJ>(a.g, S, l, nl, m);
    }
    __syncthreads();
    double xn = 0.0, yn = 0.0, zn = 0.0, n_ev = 0.0, n_eq = 0.0, lpfor = 0.0;
    double4 ncom = make_double4(0.0, 0.0, 0.0, 0.0);
    if (lane < 64) {
      state = cov ? 1 : 0;
      if (!cov) {
        const bool sov = full_sums<NT>(S, n_ev, n_eq);
        if (sov) {
          state = 1;
        } else {
          n_eq = __dadd_rn(n_eq, n_ip);
          lpfor = G.ln_pbias;
          const int k = min(lane, kCbA - 1);
          xn = S.x[k];
          yn = S.y[k];
          zn = S.z[k];
          ncom = S.com;
          wave_sync();
          if (lane < natoms) {
            S.x[lane] = xo;
            S.y[lane] = yo;
            S.z[lane] = zo;
          }
          wave_sync();
          cut_regrow_setup(c, S, G, true, flive, fdead);
        }
      }
      if (lane == 0) q_state = state;
    }
    __syncthreads();
    int acc = 0;
    double lp = __longlong_as_double(0x7ff8000000000000ll);
    if (ufi(q_state) == 0) {
      // the reverse pass over the molecule's own configuration
      fragment_placement<P, NT, LJ>(a.g, S, G, l, nl, m, true, 0, e_prev0);
      if (lane < 64 && !ufi(S.flag)) whole_molecule(a.g, S, G, true, false, false);
      if (lane == 0) S.rpos = G.rpos;
      if (fill_wave<NT>()) ring_fill(S);
      __syncthreads();
      const int cov2 = ufi(S.flag);
      double iv = 0.0, iq = 0.0, ip = 0.0, ea = 0.0, ed = 0.0;
      if (!cov2) {
        if (lane < 64) (void)mol_terms_wave<NT, LJ>(a.g, c, S, iv, iq, ip, ea, ed);
        stage_full<P, NT, LJ>(a.g, S, l, nl, m);
      }
      __syncthreads();
      if (cov2) {
        state = 2;  // the reference aborts
      } else if (lane < 64) {
        double ev, eq;
        (void)full_sums<NT>(S, ev, eq);
        eq = __dadd_rn(eq, ip);
        double de_intra = __dadd_rn(__dadd_rn(__dadd_rn(__dadd_rn(__dadd_rn(0.0, n_ea), n_ed), 0.0), n_iq), n_iv);
        double de_inter = __dadd_rn(n_eq, n_ev);
        de_intra = __dsub_rn(__dsub_rn(__dsub_rn(__dsub_rn(__dsub_rn(__dsub_rn(de_intra, 0.0), ea), ed), 0.0), iq), iv);
        de_inter = __dsub_rn(__dsub_rn(de_inter, eq), ev);
        const double de = __dadd_rn(de_intra, de_inter);
        const double de_frag = __dsub_rn(__dadd_rn(__dsub_rn(n_ea, ea), 0.0), 0.0);
        lp = __dsub_rn(__dadd_rn(__dmul_rn(beta, __dsub_rn(de, de_frag)), lpfor), G.ln_pbias);
        acc = ufi(accept_or_reject(S, G, lp));
        const int f = a.g.b.first[m];
        const double4 com = acc ? ncom : S.com;
        if (acc && lane == 0) {
          E[kE_total] = __dadd_rn(E[kE_total], de);
          E[kE_intra] = __dadd_rn(E[kE_intra], de_intra);
          E[kE_inter] = __dadd_rn(E[kE_inter], de_inter);
          E[kE_angle] = __dsub_rn(__dadd_rn(E[kE_angle], n_ea), ea);
          E[kE_dihedral] = __dsub_rn(__dadd_rn(E[kE_dihedral], n_ed), ed);
          E[kE_intra_vdw] = __dsub_rn(__dadd_rn(E[kE_intra_vdw], n_iv), iv);
          E[kE_intra_q] = __dsub_rn(__dadd_rn(E[kE_intra_q], n_iq), iq);
          E[kE_inter_vdw] = __dsub_rn(__dadd_rn(E[kE_inter_vdw], n_ev), ev);
          E[kE_inter_q] = __dsub_rn(__dadd_rn(E[kE_inter_q], n_eq), eq);
        }
        if (lane < natoms) {
          a.x[f + lane] = acc ? xn : S.x[lane];
          a.y[f + lane] = acc ? yn : S.y[lane];
          a.z[f + lane] = acc ? zn : S.z[lane];
        }
        if (lane == 0) a.comd[m] = com;
        list_move(l, nl, m, com);
      }
      if (cov2) break;
    }
    if (lane < 64) {
      done = st + 1;
      wave_sync();
      if (lane == 0) {
        if (a.kind) a.kind[st] = 2;
        if (a.accepted) a.accepted[st] = (uint8_t)acc;
        if (a.rec_energy) a.rec_energy[st] = E[kE_total];
        if (a.ln_pacc) a.ln_pacc[st] = lp;
      }
      if (a.rec_rng && lane < 5) a.rec_rng[5 * st + lane] = S.rw[lane][G.rpos & (kRing - 1)];
    }
  }
  if (lane < 64) {
    wave_sync();
    if (lane < 5) a.rng[lane] = S.rw[lane][G.rpos & (kRing - 1)];
    if (lane < 14) a.energy[lane] = E[lane];
    record_rest(a.kind, done, nsteps);
    record_rest(a.accepted, done, nsteps);
    record_rest(a.rec_energy, done, nsteps);
    record_rest(a.ln_pacc, done, nsteps);
    record_rest(a.rec_rng, 5 * done, 5 * nsteps);
    if (lane == 0) *a.status = state == 2 ? 1 : 0;
  }
}

// The growth kernels of one precision and pair style, instantiated by
// cbmc_kernels.hip (one object each): Widom insertions in parallel (256
// lanes) and in sequence (512), the GCMC chain with 128 << k lanes, GEMC and
// regrowth with 512.
struct CbmcKernels {
  void (*widom_par)(WidomCbmcArgs);
  void (*widom_seq)(WidomCbmcArgs);
  void (*gcmc[4])(const GcmcBoxArgs *, int64_t, int);
  void (*gemc)(const GcmcBoxArgs *, int64_t, int);
  void (*regrow)(const RegrowBoxArgs *, int64_t, int);
};
CbmcKernels cbmc_kernels_fp64_lj();
CbmcKernels cbmc_kernels_fp64_any();
CbmcKernels cbmc_kernels_mixed_lj();
CbmcKernels cbmc_kernels_mixed_any();
CbmcKernels cbmc_kernels_fp32_lj();
CbmcKernels cbmc_kernels_fp32_any();

}  // namespace cass
