// cbmc.hip -- the growth kernels' host side (cbmc_grow.h has the kernels):
// species set-up, the batches of CBMC Widom insertions, the GCMC, GEMC and
// regrowth chains, and the est_emax / est_atompair_rminsq estimators.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "cbmc_grow.h"
#include "engine.h"
#include "kernels.h"

namespace cass {

// The frame's live molecules, listed once for all insertions of a batch (one
// wave).
__global__ void __launch_bounds__(64) k_widom_live(GrowArgs g, LiveList l, int *nlive) {
  const int n = build_live_list<64>(g, l);
  if (threadIdx.x == 0) *nlive = n;
}

// Fixed-order sums of the insertions: widom_sum, overlaps and the
// sub-interval sums (widom_insert.f90:481-484).  One workgroup.
__global__ void __launch_bounds__(256) k_widom_cbmc_sum(const double *wvar, const uint8_t *over, int64_t n,
                                                        int nsub, int64_t subint, double *out) {
  __shared__ double sh[256];
  __shared__ long long shn[256];
  const int lane = threadIdx.x;
  // per sub-interval (and the total as interval nsub)
  for (int k = 0; k <= nsub; ++k) {
    const int64_t lo = k < nsub ? (int64_t)k * subint : 0;
    const int64_t hi = k < nsub ? lo + subint : n;
    double s = 0.0;
    long long no = 0;
    for (int64_t i = lo + lane; i < hi; i += 256) {
      s += wvar[i];
      if (k == nsub) no += over[i];
    }
    sh[lane] = s;
    shn[lane] = no;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
      if (lane < o) {
        sh[lane] += sh[lane + o];
        shn[lane] += shn[lane + o];
      }
      __syncthreads();
    }
    if (lane == 0) {
      out[k] = sh[0];
      if (k == nsub) out[nsub + 1] = (double)shn[0];
    }
    __syncthreads();
  }
}

}  // namespace cass

using namespace cass;

// ------------------------------------------------------------------ host
struct CbmcHostSpecies {
  CbmcSpeciesDev h{};
  CbmcSpeciesDev *d = nullptr;
  double *lib = nullptr;
};

static std::vector<CbmcHostSpecies> &cbmc_table(cass_engine *e) {
  // one table per engine, kept beside it (engines are few and long-lived)
  static std::vector<std::pair<cass_engine *, std::vector<CbmcHostSpecies>>> all;
  for (auto &p : all)
    if (p.first == e) return p.second;
  all.emplace_back(e, std::vector<CbmcHostSpecies>());
  return all.back().second;
}

BoxDev cass_box_view(const cass_engine *e, const cass_box_state &b);
TopoDev cass_topo_view(const cass_engine *e);

void cass_cbmc_release(cass_engine *e) {
  auto &t = cbmc_table(e);
  for (auto &s : t) {
    if (s.d) (void)hipFree(s.d);
    if (s.lib) (void)hipFree(s.lib);
  }
  t.clear();
}

extern "C" int cass_cbmc_set_species(cass_engine *e, int32_t species, const cass_cbmc_species *cs) {
  if (!e || !cs || species < 0 || species >= e->nspecies) return CASS_ERR_ARG;
  const int n = e->sp_natoms[species];
  if (n > kCbA || cs->nfrag < 1 || cs->nfrag > kCbF || cs->kappa_ins < 1 || cs->kappa_ins > kCbK ||
      cs->kappa_dih < 0 || cs->kappa_dih > kCbK || (cs->nfrag > 1 && cs->kappa_dih < 1) || cs->nangles > kCbAng ||
      cs->ndihedrals > kCbDih || cs->nangles < 0 || cs->ndihedrals < 0 || e->ntypes > 64)
    return cass_fail(e, CASS_ERR_ARG, "CBMC species beyond the device limits (16 atoms, 8 fragments, "
                                      "32 trials per stage, 32 angles, 32 dihedrals, 64 atom types)");
  CbmcHostSpecies hs;
  CbmcSpeciesDev &c = hs.h;
  c.species = species;
  c.natoms = n;
  c.nfrag = cs->nfrag;
  c.spa0 = e->sp_atom_off[species];
  c.coul_cbmc = e->sp_coul_cbmc[species];
  int k = 0, tot = 0;
  long long lk = 0;
  for (int f = 0; f < cs->nfrag; ++f) {
    const int fa = cs->frag_natoms[f];
    if (fa < 1 || fa > n) return cass_fail(e, CASS_ERR_ARG, "bad fragment size");
    c.frag_natoms[f] = fa;
    for (int j = 0; j < fa; ++j) {
      const int at = cs->frag_atoms[k + j];
      if (at < 0 || at >= n) return cass_fail(e, CASS_ERR_ARG, "bad fragment atom");
      c.frag_atoms[f][j] = at;
    }
    k += fa;
    tot += fa;
    if (cs->frag_nconfig[f] < 1) return cass_fail(e, CASS_ERR_ARG, "empty fragment library");
    c.nconfig[f] = cs->frag_nconfig[f];
    c.lib_off[f] = lk;
    lk += (long long)cs->frag_nconfig[f] * fa * 3;
  }
  // anchors: atoms bonded to two or more atoms of their fragment, each bond
  // of the list counted (input_routines.f90:2760-2820)
  for (int f = 0; f < c.nfrag; ++f) {
    int na = 0;
    c.frag_anchor[f] = -1;
    for (int i = 0; i < c.frag_natoms[f]; ++i) {
      const int ai = c.frag_atoms[f][i];
      int nb = 0;
      for (int j = 0; j < c.frag_natoms[f]; ++j) {
        const int aj = c.frag_atoms[f][j];
        if (ai == aj) continue;
        for (int b = 0; b < cs->nbonds; ++b) {
          const int b1 = cs->bond_atoms[2 * b], b2 = cs->bond_atoms[2 * b + 1];
          if ((ai == b1 && aj == b2) || (ai == b2 && aj == b1)) nb++;
        }
      }
      if (nb >= 2) {
        if (na == 0) c.frag_anchor[f] = ai;
        na++;
      }
    }
    if (na > 1) return cass_fail(e, CASS_ERR_ARG, "ring fragments are not supported by the device growth");
    if (c.nfrag > 1 && na < 1) return cass_fail(e, CASS_ERR_ARG, "fragment without an anchor atom");
  }
  for (int f = 0, cum = 0; f < c.nfrag; ++f) {
    cum += c.frag_natoms[f];
    c.prob_ins[f] = (double)c.frag_natoms[f] / (double)tot;
    c.cum_prob_ins[f] = f == 0 ? c.prob_ins[f] : (double)cum / (double)tot;
  }
  for (int f = 0; f < c.nfrag; ++f) {
    c.frag_nconnect[f] = 0;
    for (int b = 0; b < cs->nfrag_bonds; ++b) {
      const int f1 = cs->frag_bonds[2 * b], f2 = cs->frag_bonds[2 * b + 1];
      if (f1 < 0 || f1 >= c.nfrag || f2 < 0 || f2 >= c.nfrag) return cass_fail(e, CASS_ERR_ARG, "bad fragment bond");
      if (f == f1) c.frag_connect[f][c.frag_nconnect[f]++] = f2;
      else if (f == f2) c.frag_connect[f][c.frag_nconnect[f]++] = f1;
    }
  }
  c.nangles = cs->nangles;
  for (int q = 0; q < cs->nangles; ++q) {
    for (int d = 0; d < 3; ++d) c.angle[q][d] = cs->angle_atoms[3 * q + d];
    c.angle_k[q] = cs->angle_k[q];
    c.angle_t0[q] = cs->angle_theta0[q];
  }
  c.ndihed = cs->ndihedrals;
  for (int q = 0; q < cs->ndihedrals; ++q) {
    for (int d = 0; d < 4; ++d) c.dihed[q][d] = cs->dihedral_atoms[4 * q + d];
    for (int d = 0; d < 6; ++d) c.rb[q][d] = cs->dihedral_rb[6 * q + d];
  }
  c.kappa_ins = cs->kappa_ins;
  c.kappa_rot = cs->kappa_rot;
  c.kappa_dih = cs->kappa_dih;
  // prob_del1 (input_routines.f90:3050-3120): the atoms deleted with each
  // side of a fragment bond, natoms - 2 per fragment reachable from that
  // side without crossing the bond; the smaller side is cut more often
  if (cs->nfrag_bonds < 0 || cs->nfrag_bonds > kCbF) return cass_fail(e, CASS_ERR_ARG, "fragment bonds");
  c.nfbond = cs->nfrag_bonds;
  for (int b = 0; b < c.nfbond; ++b) {
    c.fbond[b][0] = cs->frag_bonds[2 * b];
    c.fbond[b][1] = cs->frag_bonds[2 * b + 1];
    int n_side[2];
    for (int side = 0; side < 2; ++side) {
      int seen[kCbF] = {0}, stack[kCbF], ns = 0, cnt = 0;
      seen[c.fbond[b][1 - side]] = 1;
      seen[c.fbond[b][side]] = 1;
      stack[ns++] = c.fbond[b][side];
      while (ns > 0) {
        const int f = stack[--ns];
        cnt += c.frag_natoms[f] - 2;
        for (int j = 0; j < c.frag_nconnect[f]; ++j) {
          const int g = c.frag_connect[f][j];
          if (!seen[g]) {
            seen[g] = 1;
            stack[ns++] = g;
          }
        }
      }
      n_side[side] = cnt;
    }
    c.prob_del1[b] = n_side[0] + n_side[1] > 0 ? (double)n_side[1] / (double)(n_side[0] + n_side[1]) : 0.5;
  }
  const int o = e->sp_atom_off[species], po = e->sp_pair_off[species];
  for (int a = 0; a < n; ++a) {
    c.type[a] = e->atom_type[o + a];
    c.q[a] = e->atom_charge[o + a];
    c.mass[a] = e->atom_mass[o + a];
  }
  for (int a = 0; a < n * n; ++a) {
    c.vs[a] = e->vdw_scale[po + a];
    c.qs[a] = e->q_scale[po + a];
    c.bonded[a] = e->bonded[po + a];
  }
  for (int f = 0; f < kCbF; ++f) c.frag_mask[f] = 0;
  for (int f = 0; f < c.nfrag; ++f)
    for (int j = 0; j < c.frag_natoms[f]; ++j) c.frag_mask[f] |= 1u << c.frag_atoms[f][j];
  for (int d = 0; d < c.ndihed; ++d) {
    c.dihed_mask[d] = 0;
    for (int q = 0; q < 4; ++q) c.dihed_mask[d] |= 1u << c.dihed[d][q];
  }
  for (int a = 0, p = 0; a < n; ++a) {
    c.intra_mask[a] = 0;
    for (int b = 0; b < n; ++b)
      if (c.vs[a * n + b] > 0.0 || c.qs[a * n + b] > 0.0) c.intra_mask[a] |= 1u << b;
    for (int b = a + 1; b < n; ++b, ++p) {
      c.pair_i[p] = (uint8_t)a;
      c.pair_j[p] = (uint8_t)b;
    }
  }
  HIP_TRY(e, hipSetDevice(e->device));
  if (hipMalloc(&hs.lib, sizeof(double) * std::max<long long>(lk, 1)) != hipSuccess ||
      hipMalloc(&hs.d, sizeof(CbmcSpeciesDev)) != hipSuccess)
    return cass_fail(e, CASS_ERR_NOMEM, "CBMC species");
  c.lib = hs.lib;
  HIP_TRY(e, hipMemcpy(hs.lib, cs->frag_coords, sizeof(double) * lk, hipMemcpyHostToDevice));
  HIP_TRY(e, hipMemcpy(hs.d, &c, sizeof(CbmcSpeciesDev), hipMemcpyHostToDevice));
  auto &t = cbmc_table(e);
  if ((int)t.size() < e->nspecies) t.resize(e->nspecies);
  if (t[species].d) (void)hipFree(t[species].d);
  if (t[species].lib) (void)hipFree(t[species].lib);
  t[species] = hs;
  return CASS_OK;
}

static const CbmcHostSpecies *cbmc_of(cass_engine *e, int species) {
  auto &t = cbmc_table(e);
  if (species < 0 || species >= (int)t.size() || !t[species].d) return nullptr;
  return &t[species];
}

// Compute_Molecule_Angle_Energy (energy_routines.f90:283-347) and
// Compute_Molecule_Dihedral_Energy (:350-447) of one molecule of species s
// on the host, every atom existing; the arithmetic of angle_term and
// dihedral_term.  False: s has no growth description (a rigid species,
// no bonded energy).
bool cass_cbmc_bonded_host(const cass_engine *e, int s, const double *xyz, double *angle, double *dihedral) {
  const CbmcHostSpecies *hs = cbmc_of(const_cast<cass_engine *>(e), s);
  *angle = *dihedral = 0.0;
  if (!hs) return false;
  const CbmcSpeciesDev &c = hs->h;
  auto X = [&](int a, int d) { return xyz[3 * a + d]; };
  double ea_sum = 0.0;
  for (int k = 0; k < c.nangles; ++k) {
    double ea = 0.0;
    if (c.angle_k[k] != 0.0) {
      const int *q = c.angle[k];
      const double rx21 = X(q[1], 0) - X(q[0], 0), ry21 = X(q[1], 1) - X(q[0], 1), rz21 = X(q[1], 2) - X(q[0], 2);
      const double rx32 = X(q[2], 0) - X(q[1], 0), ry32 = X(q[2], 1) - X(q[1], 1), rz32 = X(q[2], 2) - X(q[1], 2);
      const double c23 = (rx21 * rx32 + ry21 * ry32) + rz21 * rz32;
      const double c22 = (rx21 * rx21 + ry21 * ry21) + rz21 * rz21;
      const double c33 = (rx32 * rx32 + ry32 * ry32) + rz32 * rz32;
      const double inv = 1.0 / std::sqrt(c33 * c22);
      double ct = c23 * inv;
      ct = std::fmin(ct, 0.999999);
      ct = std::fmax(ct, -0.999999);
      const double d = (kPi - std::acos(ct)) - c.angle_t0[k];
      ea = c.angle_k[k] * (d * d);
    }
    ea_sum = ea_sum + ea;
  }
  double ed_sum = 0.0;
  for (int dd = 0; dd < c.ndihed; ++dd) {
    const int *q = c.dihed[dd];
    const double rx12 = X(q[0], 0) - X(q[1], 0), ry12 = X(q[0], 1) - X(q[1], 1), rz12 = X(q[0], 2) - X(q[1], 2);
    const double rx32 = X(q[2], 0) - X(q[1], 0), ry32 = X(q[2], 1) - X(q[1], 1), rz32 = X(q[2], 2) - X(q[1], 2);
    const double rx34 = X(q[2], 0) - X(q[3], 0), ry34 = X(q[2], 1) - X(q[3], 1), rz34 = X(q[2], 2) - X(q[3], 2);
    const double mx = ry12 * rz32 - ry32 * rz12, my = -(rx12 * rz32) + rz12 * rx32, mz = rx12 * ry32 - ry12 * rx32;
    const double nx = ry32 * rz34 - rz32 * ry34, ny = -(rx32 * rz34) + rz32 * rx34, nz = rx32 * ry34 - ry32 * rx34;
    const double msq = (mx * mx + my * my) + mz * mz, nsq = (nx * nx + ny * ny) + nz * nz;
    const double mdn = (mx * nx + my * ny) + mz * nz;
    const double c1 = mdn / std::sqrt(msq * nsq);
    const double c2 = c1 * c1, c3 = c1 * c2, c4 = c2 * c2, c5 = c2 * c3;
    const double *rb = c.rb[dd];
    double dot = 1.0 * rb[0];
    dot = dot + c1 * rb[1];
    dot = dot + c2 * rb[2];
    dot = dot + c3 * rb[3];
    dot = dot + c4 * rb[4];
    dot = dot + c5 * rb[5];
    ed_sum = ed_sum + dot;
  }
  *angle = ea_sum;
  *dihedral = ed_sum;
  return true;
}

static bool species_has_charge(const cass_engine *e, int s) {
  for (int a = 0; a < e->sp_natoms[s]; ++a)
    if (e->atom_charge[e->sp_atom_off[s] + a] != 0.0) return true;
  return false;
}

static GrowArgs grow_args(cass_engine *e, cass_box_state &b, const CbmcHostSpecies *hs) {
  GrowArgs g;
  g.b = cass_box_view(e, b);
  g.tp = cass_topo_view(e);
  g.cd = make_pair_const<double>(b.p, e->ntypes);
  g.cf = make_pair_const<float>(b.p, e->ntypes);
  g.sp = hs->d;
  g.beta = b.p.beta;
  return g;
}

// Whether a grown species' pairs in box b are plain LJ (the LJ kernels): LJ
// cut / cut_tail / cut_shift, no CBMC energy table, no q-q terms of the
// species, and a topology within the LDS tables.
static bool lj_growth(const cass_engine *e, const cass_box_state &b, int species) {
  const cass_params &p = b.p;
  return p.vdw_style == CASS_VDW_LJ &&
         (p.vdw_sum_style == CASS_SUM_CUT || p.vdw_sum_style == CASS_SUM_CUT_TAIL ||
          p.vdw_sum_style == CASS_SUM_CUT_SHIFT) &&
         !b.apt && (p.charge_style == CASS_Q_NONE || !species_has_charge(e, species)) && e->nspecies <= kCtSp &&
         e->natoms_total <= kCtAt && e->ntypes <= kCtT;
}

static CbmcKernels growth_kernels(const cass_engine *e, bool lj) {
  if (e->prec == CASS_PREC_MIXED) return lj ? cbmc_kernels_mixed_lj() : cbmc_kernels_mixed_any();
  if (e->prec == CASS_PREC_FP32) return lj ? cbmc_kernels_fp32_lj() : cbmc_kernels_fp32_any();
  return lj ? cbmc_kernels_fp64_lj() : cbmc_kernels_fp64_any();
}

// Index of a GCMC workgroup size (128 << k lanes).
static int lanes_index(int nt) {
  int k = 0;
  while (128 << k < nt) ++k;
  return k;
}

static int widom_cbmc(cass_engine *e, int32_t box, int32_t species, int64_t n_ins, cass_rng *rng, uint64_t seed,
                      int32_t n_sub, double *sub, double *widom_var, cass_widom_result *res, double *eij_max,
                      uint8_t *overlap, double *rsq_min) {
  if (!e || box < 0 || box >= (int)e->boxes.size() || n_ins <= 0 || !res || n_sub < 0 || n_sub > 1024)
    return CASS_ERR_ARG;
  const CbmcHostSpecies *hs = cbmc_of(e, species);
  if (!hs) return cass_fail(e, CASS_ERR_STATE, "no CBMC description for this species (cass_cbmc_set_species)");
  if (eij_max && !(e->nspecies <= kCtSp && e->natoms_total <= kCtAt && e->ntypes <= kCtT))
    return cass_fail(e, CASS_ERR_ARG, "est_emax needs at most 8 species, 128 species sites and 16 atom types");
  cass_box_state &b = e->boxes[box];
  if (b.p.charge_style == CASS_Q_EWALD && species_has_charge(e, species))
    return cass_fail(e, CASS_ERR_ARG, "CBMC Widom of a charged species with Ewald sums is not supported");
  HIP_TRY(e, hipSetDevice(e->device));
  // the insertion-independent constants (widom_insert.f90:212-240)
  double lrc_diff = 0.0, e_self = 0.0;
  if (b.p.vdw_sum_style == CASS_SUM_CUT_TAIL) {
    std::vector<double> nb(e->ntypes, 0.0);
    for (int m = 0; m < b.nmols; ++m) {
      if (!b.live[m]) continue;
      const int s = b.mol_species[m];
      for (int a = 0; a < e->sp_natoms[s]; ++a) {
        const int ty = e->atom_type[e->sp_atom_off[s] + a];
        if (ty >= 0) nb[ty] += 1.0;
      }
    }
    double e0, e1;
    cass_lrc(e, box, nb.data(), &e0);
    for (int a = 0; a < e->sp_natoms[species]; ++a) {
      const int ty = e->atom_type[e->sp_atom_off[species] + a];
      if (ty >= 0) nb[ty] += 1.0;
    }
    cass_lrc(e, box, nb.data(), &e1);
    lrc_diff = e1 - e0;
  }
  if (b.p.charge_style != CASS_Q_NONE && species_has_charge(e, species)) cass_mol_self_energy(e, box, species, &e_self);
  const int nsub = n_sub > 0 ? n_sub : 1;
  const int64_t rsq_stride = rsq_min ? (int64_t)e->natoms_total * e->sp_natoms[species] : 0;
  const size_t live_bytes = (kCentre + sizeof(LiveMol)) * (size_t)b.nmols + 64;
  const size_t need = (size_t)n_ins * (2 * sizeof(double) + 1) + sizeof(double) * (nsub + 2) + 64 +
                      5 * sizeof(int64_t) + sizeof(double) * (size_t)(n_ins * rsq_stride) + live_bytes;
  char *s = (char *)cass_scratch(e, need);
  if (!s) return cass_fail(e, CASS_ERR_NOMEM, "scratch");
  // the frame's live molecules, then the per-insertion arrays
  double *d_lcom = (double *)s;
  LiveMol *d_lmol = (LiveMol *)(d_lcom + 4 * (size_t)b.nmols);
  int *d_nlive = (int *)(d_lmol + b.nmols);
  double *d_w = (double *)(s + (live_bytes & ~(size_t)15));
  double *d_em = d_w + n_ins;
  double *d_rsq = d_em + n_ins;
  double *d_out = d_rsq + n_ins * rsq_stride;
  int64_t *d_rng = (int64_t *)(d_out + nsub + 2);
  uint8_t *d_ov = (uint8_t *)(d_rng + 5);
  WidomCbmcArgs w;
  w.g = grow_args(e, b, hs);
  w.n_ins = n_ins;
  w.seed = seed;
  w.sequential = rng != nullptr;
  w.rng = d_rng;
  // E_inter_constant = lrc_diff + E_self - E_recip_in (no reciprocal term here)
  w.e_const = (lrc_diff + e_self) - 0.0;
  w.wvar = d_w;
  w.over = d_ov;
  w.eij_max = eij_max ? d_em : nullptr;
  w.rsq_min = rsq_min ? d_rsq : nullptr;
  w.rsq_rows = e->natoms_total;
  w.live = LiveList{d_lmol, d_lcom, b.nmols};
  w.nlive = d_nlive;
  if (rng) HIP_TRY(e, hipMemcpyAsync(d_rng, rng->s, sizeof(int64_t) * 5, hipMemcpyHostToDevice, e->stream));
  HIP_TRY(e, hipEventRecord(e->ev0, e->stream));
  const int grid = rng ? 1 : (int)n_ins;
  if (rng ? false : (int64_t)grid != n_ins) return cass_fail(e, CASS_ERR_ARG, "too many insertions for one batch");
  hipLaunchKernelGGL(k_widom_live, dim3(1), dim3(64), 0, e->stream, w.g, w.live, d_nlive);
  HIP_TRY(e, hipGetLastError());
  const bool lj = lj_growth(e, b, species);
  // One insertion of the parallel mode per workgroup of 4 waves: the LDS
  // holds three of them a CU, and 3001 pentane insertions (kappa 12 / 24) took
  // 0.45, 0.44 and 0.62 ms with 2, 4 and 8 waves.  Insertions in
  // sequence have one CU to themselves: 8 waves.
  const int nt = rng ? 512 : 256;
  const CbmcKernels kt = growth_kernels(e, lj);
  hipLaunchKernelGGL(rng ? kt.widom_seq : kt.widom_par, dim3(grid), dim3(nt), 0, e->stream, w);
  HIP_TRY(e, hipGetLastError());
  const int64_t subint = n_ins / nsub;
  hipLaunchKernelGGL(k_widom_cbmc_sum, dim3(1), dim3(256), 0, e->stream, d_w, d_ov, n_ins, n_sub > 0 ? n_sub : 0,
                     subint, d_out);
  HIP_TRY(e, hipGetLastError());
  HIP_TRY(e, hipEventRecord(e->ev1, e->stream));
  std::vector<double> out(nsub + 2);
  HIP_TRY(e, hipMemcpyAsync(out.data(), d_out, sizeof(double) * (nsub + 2), hipMemcpyDeviceToHost, e->stream));
  if (rng) HIP_TRY(e, hipMemcpyAsync(rng->s, d_rng, sizeof(int64_t) * 5, hipMemcpyDeviceToHost, e->stream));
  if (widom_var) HIP_TRY(e, hipMemcpyAsync(widom_var, d_w, sizeof(double) * n_ins, hipMemcpyDeviceToHost, e->stream));
  if (eij_max) HIP_TRY(e, hipMemcpyAsync(eij_max, d_em, sizeof(double) * n_ins, hipMemcpyDeviceToHost, e->stream));
  if (overlap) HIP_TRY(e, hipMemcpyAsync(overlap, d_ov, n_ins, hipMemcpyDeviceToHost, e->stream));
  if (rsq_min)
    HIP_TRY(e, hipMemcpyAsync(rsq_min, d_rsq, sizeof(double) * n_ins * rsq_stride, hipMemcpyDeviceToHost, e->stream));
  HIP_TRY(e, hipStreamSynchronize(e->stream));
  float ms = 0.f;
  if (hipEventElapsedTime(&ms, e->ev0, e->ev1) == hipSuccess) e->last_kernel_ms = ms;
  const int ns = n_sub > 0 ? n_sub : 0;
  if (sub)
    for (int k = 0; k < ns; ++k) sub[k] = out[k];
  res->widom_sum = out[ns];
  res->n_overlaps = (int64_t)out[ns + 1];
  res->n_insertions = n_ins;
  res->e_const = w.e_const;
  return CASS_OK;
}

extern "C" int cass_widom_cbmc_batch(cass_engine *e, int32_t box, int32_t species, int64_t n_ins, cass_rng *rng,
                                     uint64_t seed, int32_t n_sub, double *sub, double *widom_var,
                                     cass_widom_result *res) {
  return widom_cbmc(e, box, species, n_ins, rng, seed, n_sub, sub, widom_var, res, nullptr, nullptr, nullptr);
}

extern "C" int cass_widom_cbmc_emax(cass_engine *e, int32_t box, int32_t species, int64_t n_ins, cass_rng *rng,
                                    uint64_t seed, double *widom_var, double *eij_max, uint8_t *overlap,
                                    double *rsq_min, cass_widom_result *res) {
  if (!widom_var || !eij_max || !overlap) return CASS_ERR_ARG;
  return widom_cbmc(e, box, species, n_ins, rng, seed, 0, nullptr, widom_var, res, eij_max, overlap, rsq_min);
}

// ---------------------------------------------------------------- est_emax
// Bins 0..ub merged `by` at a time into bins 0..(ub+1)/by-1 (maximum of the
// weights, counts and weight sums in bin order), the rest cleared: the
// histogram of a factor divided by `by` (coarsen_w_max,
// widom_insert.f90:570-589).
static void emax_merge(int32_t ub, double *w_max, double *w_sum, int64_t *freq, int64_t by) {
  const int64_t groups = ((int64_t)ub + 1) / by;
  for (int64_t g = 0; g < groups; ++g) {
    const int64_t lo = g * by;
    double m = w_max[lo], s = 0.0;
    int64_t f = 0;
    for (int64_t k = lo; k < lo + by; ++k) {
      m = w_max[k] > m ? w_max[k] : m;
      s = s + w_sum[k];
      f += freq[k];
    }
    w_max[g] = m;
    w_sum[g] = s;
    freq[g] = f;
  }
  for (int64_t k = groups; k <= ub; ++k) {
    w_max[k] = 0.0;
    w_sum[k] = 0.0;
    freq[k] = 0;
  }
}

extern "C" int cass_emax_frame(int32_t ub, double *factor, double *w_max, double *w_sum, int64_t *freq, int64_t n,
                               const double *widom_var, const double *eij_max, const uint8_t *overlap,
                               double prefactor) {
  if (ub < 1 || !factor || !(*factor > 0.0) || !w_max || !w_sum || !freq || n < 0 ||
      (n > 0 && (!widom_var || !eij_max || !overlap)))
    return CASS_ERR_ARG;
  for (int64_t i = 0; i < n; ++i)
    if (!overlap[i] && !(eij_max[i] >= 0.0 && std::isfinite(eij_max[i]))) return CASS_ERR_ARG;
  // the frame's own histogram (widom_insert.f90:466-476): an insertion past
  // the top bin halves the frame's factor until it fits
  std::vector<double> fmax(ub + 1, 0.0), fsum(ub + 1, 0.0);
  std::vector<int64_t> fcnt(ub + 1, 0);
  double tf = *factor;
  int64_t merged = 1;
  for (int64_t i = 0; i < n; ++i) {
    if (overlap[i]) continue;
    while (eij_max[i] * tf >= (double)ub + 1.0) {
      emax_merge(ub, fmax.data(), fsum.data(), fcnt.data(), 2);
      tf = tf / 2.0;
      merged *= 2;
    }
    const int b = (int)(eij_max[i] * tf);
    fmax[b] = widom_var[i] > fmax[b] ? widom_var[i] : fmax[b];
    fsum[b] = fsum[b] + widom_var[i];
    fcnt[b] += 1;
  }
  // the running totals follow in one merge (widom_insert.f90:490-520)
  if (merged > 1) {
    emax_merge(ub, w_max, w_sum, freq, merged);
    *factor = *factor / (double)merged;
  }
  for (int k = 0; k <= ub; ++k) {
    const double m = prefactor * fmax[k];
    w_max[k] = m > w_max[k] ? m : w_max[k];
    w_sum[k] = w_sum[k] + prefactor * fsum[k];
    freq[k] += fcnt[k];
  }
  return CASS_OK;
}

extern "C" int cass_emax_estimate(int32_t ub, double factor, const double *w_sum, const int64_t *freq,
                                  double widom_sum, double beta, double *emax, int64_t *nskips, double *w_frac) {
  if (ub < 1 || !(factor > 0.0) || !w_sum || !freq || !emax || !nskips) return CASS_ERR_ARG;
  // Estimate_Pair_Emax (pair_emax_estimation.f90:41-77): the bins' weight
  // fractions added from the top until they pass 1e-10
  int32_t top = ub + 1;
  double tail = 0.0;
  while (top >= 1) {
    tail = tail + w_sum[top - 1] / widom_sum;
    if (tail > 1.0e-10) break;
    --top;
  }
  *emax = (double)top * (beta / factor);
  int64_t skipped = 0;
  for (int32_t k = top; k <= ub; ++k) skipped += freq[k];
  *nskips = skipped;
  if (w_frac)
    for (int32_t k = 0; k <= ub; ++k) w_frac[k] = w_sum[k] / widom_sum;
  return CASS_OK;
}

// ------------------------------------------------------ est_atompair_rminsq
extern "C" int cass_rminsq_frame(int32_t nsolv, const int32_t *rows, int32_t nsolute, int32_t nrows, int32_t res,
                                 double step, double rcut_lowsq, double *w_max, double *w_sum, int64_t *freq,
                                 int64_t n, const double *widom_var, const double *rsq_min, const uint8_t *overlap,
                                 double prefactor) {
  if (nsolv < 1 || nsolute < 1 || nrows < 1 || res < 1 || !rows || !(step > 0.0) || !(rcut_lowsq >= 0.0) ||
      !w_max || !w_sum || !freq || n < 0 || (n > 0 && (!widom_var || !rsq_min || !overlap)))
    return CASS_ERR_ARG;
  for (int32_t k = 0; k < nsolv; ++k)
    if (rows[k] < 0 || rows[k] >= nrows) return CASS_ERR_ARG;
  // bins of width step from rcut_low^2 (atompair_nrg_table_routines.f90:133-135)
  const double top = step * res + rcut_lowsq, shift = rcut_lowsq - step;
  const size_t cells = (size_t)nsolv * nsolute;
  std::vector<double> fmax(cells * res, 0.0), fsum(cells * res, 0.0);
  std::vector<int64_t> fcnt(cells * res, 0);
  for (int64_t i = 0; i < n; ++i) {
    if (overlap[i]) continue;
    const double *m = rsq_min + (size_t)i * nrows * nsolute;
    const double w = widom_var[i];
    for (int32_t k = 0; k < nsolv; ++k)
      for (int32_t a = 0; a < nsolute; ++a) {
        const double r2 = m[(size_t)rows[k] * nsolute + a];
        if (!(r2 < top)) continue;
        // INT((r2 - shift) / step), 1-based, held inside 1..res
        const int b = std::min(std::max((int)((r2 - shift) / step), 1), (int)res) - 1;
        const size_t q = ((size_t)k * nsolute + a) * res + b;
        fmax[q] = w > fmax[q] ? w : fmax[q];
        fsum[q] = fsum[q] + w;
        fcnt[q] += 1;
      }
  }
  for (size_t q = 0; q < cells * res; ++q) {
    freq[q] += fcnt[q];
    w_sum[q] = w_sum[q] + prefactor * fsum[q];
    const double m = prefactor * fmax[q];
    w_max[q] = m > w_max[q] ? m : w_max[q];
  }
  return CASS_OK;
}

extern "C" int cass_rminsq_estimate(int32_t nsolv, int32_t nsolute, int32_t res, const double *w_max,
                                    const double *w_sum, const int64_t *freq, double widom_sum, double tol,
                                    int32_t *ind, int64_t *nskips, double *wmax) {
  if (nsolv < 1 || nsolute < 1 || res < 1 || !w_max || !w_sum || !freq || !ind || !nskips || !wmax)
    return CASS_ERR_ARG;
  // Estimate_Pair_rminsq (pair_emax_estimation.f90:79-168): per pair, the
  // first bin at which the fractions summed outward pass tol
  int64_t sk_all = 0;
  double wm_all = 0.0;
  for (int32_t k = 0; k < nsolv; ++k)
    for (int32_t a = 0; a < nsolute; ++a) {
      const size_t base = ((size_t)k * nsolute + a) * res;
      double frac = 0.0, wm = 0.0;
      int64_t sk = 0;
      int32_t b = 0;
      for (; b < res; ++b) {
        frac = frac + w_sum[base + b] / widom_sum;
        if (frac > tol) break;
        wm = w_max[base + b] > wm ? w_max[base + b] : wm;
        sk += freq[base + b];
      }
      ind[k * nsolute + a] = b + 1;
      sk_all = std::max(sk_all, sk);
      wm_all = wm > wm_all ? wm : wm_all;
    }
  *nskips = sk_all;
  *wmax = wm_all;
  return CASS_OK;
}

// Live lists of up to this many bytes per workgroup stand in the LDS beside
// the chain kernels' own 40 to 60 KB; longer ones in device memory.
constexpr size_t kListLds = (size_t)96 << 10;
static int list_cap_of(int maxm, int per) {
  const int cap = (maxm + 3) & ~3;
  return (size_t)per * cap * kListBytes <= kListLds ? cap : 0;
}

// One launch of a chain kernel with the live lists of `per` boxes in the
// dynamic LDS (cap molecules each; 0: in device memory).
template <typename K, typename A>
static int launch_chain(cass_engine *e, K kern, const A *d_boxes, int grid, int nt, int64_t nsteps, int cap, int per,
                        const char *what) {
  const size_t lds = (size_t)per * cap * kListBytes;
  // the attribute belongs to the process: always the largest, so that engines on
  // other threads never find a smaller one than they launch with
  HIP_TRY(e, hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kListLds));
  hipLaunchKernelGGL(kern, dim3(grid), dim3(nt), lds, e->stream, d_boxes, nsteps, cap);
  return hipGetLastError() == hipSuccess ? CASS_OK : cass_fail(e, CASS_ERR_HIP, what);
}

// workgroup size of the GCMC chain per engine: 0 until cass_gcmc_autotune
// picks one (then 512)
static std::vector<std::pair<cass_engine *, int>> g_gcmc_block;
static int &gcmc_block(cass_engine *e) {
  for (auto &p : g_gcmc_block)
    if (p.first == e) return p.second;
  g_gcmc_block.emplace_back(e, 0);
  return g_gcmc_block.back().second;
}

// One launch of the chain over the given boxes; commit = 0 leaves the boxes
// and the caller's states untouched (a timing run).
static int gcmc_launch(cass_engine *e, int32_t nboxes, const cass_gcmc_box *boxes, cass_gcmc_state *states,
                       int64_t nsteps, cass_gcmc_record *rec, int commit, int nt, double *ms_out, bool gemc = false) {
  if (!e || nboxes <= 0 || !boxes || !states || nsteps < 0) return CASS_ERR_ARG;
  if (nsteps == 0) return CASS_OK;
  if (e->ntypes > 64) return cass_fail(e, CASS_ERR_ARG, "the device GCMC / GEMC chains take up to 64 atom types");
  if (gemc) {
    if (nboxes % 2) return cass_fail(e, CASS_ERR_ARG, "GEMC boxes come in pairs");
    for (int i = 0; i < nboxes; i += 2)
      if (boxes[i].species != boxes[i + 1].species)
        return cass_fail(e, CASS_ERR_ARG, "the boxes of a GEMC pair exchange one species");
  }
  HIP_TRY(e, hipSetDevice(e->device));
  const int ntypes = e->ntypes;
  size_t bytes = 0;
  int maxm = 0;
  bool lj = true;
  ChainRecords recs;
  struct Offs {
    size_t rng, en, cnt, loc, res, nb, kind, acc, nm, ren, rr;
  };
  std::vector<Offs> offs(nboxes);
  auto up = [](size_t n) { return (n + 255) & ~size_t(255); };
  for (int i = 0; i < nboxes; ++i) {
    const cass_gcmc_box &g = boxes[i];
    if (g.box < 0 || g.box >= (int)e->boxes.size()) return cass_fail(e, CASS_ERR_ARG, "bad box");
    for (int j = 0; j < i; ++j)
      if (boxes[j].box == g.box) return cass_fail(e, CASS_ERR_ARG, "a box appears twice");
    cass_box_state &b = e->boxes[g.box];
    const CbmcHostSpecies *hs = cbmc_of(e, g.species);
    if (!hs) return cass_fail(e, CASS_ERR_STATE, "no CBMC description for the sorbate (cass_cbmc_set_species)");
    if (g.first_slot < 0 || g.max_mols < 1 || g.first_slot + g.max_mols > b.nmols)
      return cass_fail(e, CASS_ERR_ARG, "sorbate slots outside the box");
    for (int m = g.first_slot; m < g.first_slot + g.max_mols; ++m)
      if (b.mol_species[m] != g.species) return cass_fail(e, CASS_ERR_ARG, "a sorbate slot holds another species");
    if (b.p.charge_style != CASS_Q_NONE && species_has_charge(e, g.species))
      return cass_fail(e, CASS_ERR_ARG, "GCMC of a charged sorbate is not supported on the device");
    if (b.p.vdw_style == CASS_VDW_MIE && b.p.vdw_sum_style == CASS_SUM_CUT_TAIL)
      return cass_fail(e, CASS_ERR_ARG, "Mie tail corrections are not supported by the device GCMC chain");
    if (b.p.box_shape != CASS_BOX_CUBIC && b.p.box_shape != CASS_BOX_ORTHO)
      return cass_fail(e, CASS_ERR_ARG, "the device GCMC chain places centres in cubic or orthogonal boxes");
    const cass_gcmc_state &s = states[i];
    if (s.nmols < 0 || s.nres < 0 || s.nmols + s.nres != g.max_mols || !s.locate || !s.reservoir)
      return cass_fail(e, CASS_ERR_ARG, "locate / reservoir do not cover the sorbate slots");
    {
      // together they must name every slot once, live slots live and the others dead
      std::vector<char> seen(g.max_mols, 0);
      for (int k = 0; k < s.nmols + s.nres; ++k) {
        const int v = k < s.nmols ? s.locate[k] : s.reservoir[k - s.nmols];
        if (v < 0 || v >= g.max_mols || seen[v]) return cass_fail(e, CASS_ERR_ARG, "locate / reservoir entries");
        seen[v] = 1;
        if ((k < s.nmols) != (b.live[g.first_slot + v] != 0))
          return cass_fail(e, CASS_ERR_ARG, "locate / reservoir disagree with the live flags");
      }
    }
    maxm = std::max(maxm, b.nmols);
    lj = lj && lj_growth(e, b, g.species);
    // the same rounded pieces the layout below takes, one by one
    bytes += up(sizeof(int64_t) * 5) + up(sizeof(double) * 14) + up(sizeof(int) * 2) +
             2 * up(sizeof(int) * g.max_mols) + up(sizeof(double) * ntypes);
    Offs &o = offs[i];
    if (rec) {
      const size_t at = (size_t)i * nsteps;
      o.kind = recs.add(rec->kind + at, nsteps);
      o.acc = recs.add(rec->accepted + at, nsteps);
      o.nm = recs.add(rec->nmols + at, sizeof(int) * nsteps);
      o.ren = recs.add(rec->energy + at, sizeof(double) * nsteps);
      o.rr = recs.add(rec->rng_state + 5 * at, sizeof(int64_t) * 5 * nsteps);
    }
  }
  bytes += up(sizeof(GcmcBoxArgs) * nboxes);
  // the records, then the live lists, which are not copied to or from the host
  const int list_cap = list_cap_of(maxm, gemc ? 2 : 1);
  const size_t state_bytes = bytes;
  bytes += recs.staged();
  const size_t list_at = bytes;
  if (list_cap == 0) bytes += (up(kCentre * maxm) + up(sizeof(LiveMol) * maxm)) * (size_t)nboxes;
  char *s0 = (char *)cass_scratch(e, bytes + 256);
  if (!s0) return cass_fail(e, CASS_ERR_NOMEM, "scratch");
  if (int rrc = recs.place(e, s0 + state_bytes)) return rrc;
  std::vector<char> host(state_bytes, 0);
  size_t off = 0;
  auto take = [&](size_t n) {
    const size_t o = off;
    off += up(n);
    return o;
  };
  std::vector<GcmcBoxArgs> args(nboxes);
  for (int i = 0; i < nboxes; ++i) {
    const cass_gcmc_box &g = boxes[i];
    cass_box_state &b = e->boxes[g.box];
    const cass_gcmc_state &st = states[i];
    Offs &o = offs[i];
    o.rng = take(sizeof(int64_t) * 5);
    o.en = take(sizeof(double) * 14);
    o.cnt = take(sizeof(int) * 2);
    o.loc = take(sizeof(int) * g.max_mols);
    o.res = take(sizeof(int) * g.max_mols);
    o.nb = take(sizeof(double) * ntypes);
    std::memcpy(host.data() + o.rng, st.rng.s, sizeof(int64_t) * 5);
    std::memcpy(host.data() + o.en, &st.energy, sizeof(double) * 14);
    int cnt[2] = {st.nmols, st.nres};
    std::memcpy(host.data() + o.cnt, cnt, sizeof(cnt));
    std::memcpy(host.data() + o.loc, st.locate, sizeof(int) * st.nmols);
    std::memcpy(host.data() + o.res, st.reservoir, sizeof(int) * st.nres);
    // bead counts per type of the live molecules (Compute_Beads)
    std::vector<double> nb(ntypes, 0.0);
    std::vector<int64_t> count(e->nspecies, 0);
    for (int m = 0; m < b.nmols; ++m)
      if (b.live[m]) ++count[b.mol_species[m]];
    for (int sp = 0; sp < e->nspecies; ++sp)
      for (int a = 0; a < e->sp_natoms[sp]; ++a) {
        const int ty = e->atom_type[e->sp_atom_off[sp] + a];
        if (ty >= 0) nb[ty] += (double)count[sp];
      }
    std::memcpy(host.data() + o.nb, nb.data(), sizeof(double) * ntypes);
    GcmcBoxArgs &a = args[i];
    a.g = grow_args(e, b, cbmc_of(e, g.species));
    a.x = b.x;
    a.y = b.y;
    a.z = b.z;
    a.comd = b.comd;
    a.live = b.d_live;
    a.first_slot = g.first_slot;
    a.max_mols = g.max_mols;
    a.prob_insert = g.prob_insert;
    a.mu = g.mu;
    a.lambda = g.de_broglie;
    a.log_volume = std::log(b.p.volume);
    a.rng = (int64_t *)(s0 + o.rng);
    a.energy = (double *)(s0 + o.en);
    a.nmols = (int *)(s0 + o.cnt);
    a.nres = a.nmols + 1;
    a.locate = (int *)(s0 + o.loc);
    a.reservoir = (int *)(s0 + o.res);
    a.nbeads = (double *)(s0 + o.nb);
    a.volume = b.p.volume;
    a.rcut3 = b.p.rcut3;
    a.rcut9 = b.p.rcut9;
    a.rcut_vdw = b.p.rcut_vdw;
    a.vdw_style = b.p.vdw_style;
    a.tail = b.p.vdw_sum_style == CASS_SUM_CUT_TAIL;
    a.commit = commit;
    a.kind = rec ? recs.at<uint8_t>(o.kind) : nullptr;
    a.accepted = rec ? recs.at<uint8_t>(o.acc) : nullptr;
    a.rec_nmols = rec ? recs.at<int>(o.nm) : nullptr;
    a.rec_energy = rec ? recs.at<double>(o.ren) : nullptr;
    a.rec_rng = rec ? recs.at<int64_t>(o.rr) : nullptr;
    const size_t o_list = list_at + (up(kCentre * maxm) + up(sizeof(LiveMol) * maxm)) * (size_t)i;
    a.list = list_cap ? LiveList{nullptr, nullptr, 0}
                      : LiveList{(LiveMol *)(s0 + o_list + up(kCentre * maxm)), (double *)(s0 + o_list), maxm};
  }
  const size_t o_args = take(sizeof(GcmcBoxArgs) * nboxes);
  if (off != state_bytes) return cass_fail(e, CASS_ERR_STATE, "GCMC state layout differs from its buffer");
  MirrorPull mirrors;
  std::vector<int> ids(commit ? nboxes : 0);
  for (size_t i = 0; i < ids.size(); ++i) ids[i] = boxes[i].box;
  if (int mrc = mirrors.reserve(e, ids, true, off + recs.staged())) return mrc;
  std::memcpy(host.data() + o_args, args.data(), sizeof(GcmcBoxArgs) * nboxes);
  HIP_TRY(e, hipMemcpyAsync(s0, host.data(), off, hipMemcpyHostToDevice, e->stream));
  HIP_TRY(e, hipEventRecord(e->ev0, e->stream));
  // 8 waves unless the autotuner picked otherwise.  us a move of pentane boxes
  // (FP64) with 2 / 4 / 8 / 16 waves:
  //     8 molecules,  48 boxes    59.6 / 50.7 / 45.8 / 47.8
  //    60 molecules,  48 boxes    87.5 / 68.0 / 56.9 / 54.6
  //    60 molecules, 300 boxes     203 /  190 /  204 /  201
  //    60 molecules, 900 boxes     950 /  923 /  958 /  964
  //   500 molecules,  48 boxes     238 /  159 /  123 /  101
  //  3000 molecules,   8 boxes     954 /  525 /  343 /  210
  // and LJ switch, 60 molecules, 48 boxes: 113 / 85 / 69 / 84.  16 waves leave
  // 128 registers a lane, and the kernels then spill.
  if (nt <= 0) nt = gcmc_block(e) > 0 ? gcmc_block(e) : 512;
  const GcmcBoxArgs *d_args = (const GcmcBoxArgs *)(s0 + o_args);
  if (gemc) nt = 512;  // 30 transfers of 96 pentane pairs: 3.0 ms with 4 waves, 2.4 ms with 8
  if (nt != 128 && nt != 256 && nt != 512 && nt != 1024) return cass_fail(e, CASS_ERR_ARG, "workgroup size");
  const CbmcKernels kt = growth_kernels(e, lj);
  const int rc = gemc ? launch_chain(e, kt.gemc, d_args, nboxes / 2, nt, nsteps, list_cap, 2,
                                     "k_gemc_chain launch")
                      : launch_chain(e, kt.gcmc[lanes_index(nt)], d_args, nboxes, nt, nsteps, list_cap, 1,
                                     "k_gcmc_chain launch");
  if (rc) return rc;
  HIP_TRY(e, hipEventRecord(e->ev1, e->stream));
  // the states and, unless this is a timing run, coordinates, live flags and
  // centres of every box come back behind one synchronisation
  if (int mrc = mirrors.queue(e)) return mrc;
  HIP_TRY(e, hipMemcpyAsync(mirrors.host, s0, off + recs.staged(), hipMemcpyDeviceToHost, e->stream));
  if (int mrc = recs.queue(e)) return mrc;
  HIP_TRY(e, hipStreamSynchronize(e->stream));
  float ms = 0.f;
  if (hipEventElapsedTime(&ms, e->ev0, e->ev1) == hipSuccess) e->last_kernel_ms = ms;
  if (ms_out) *ms_out = ms;
  if (!commit) return CASS_OK;
  mirrors.end(e);
  recs.end(mirrors.host + off);
  const char *back = mirrors.host;
  int bad = 0;
  for (int i = 0; i < nboxes; ++i) {
    const cass_gcmc_box &g = boxes[i];
    cass_gcmc_state &st = states[i];
    const Offs &o = offs[i];
    std::memcpy(st.rng.s, back + o.rng, sizeof(int64_t) * 5);
    std::memcpy(&st.energy, back + o.en, sizeof(double) * 14);
    int cnt[2];
    std::memcpy(cnt, back + o.cnt, sizeof(cnt));
    if (cnt[1] < 0) bad = 1;
    st.nmols = cnt[0];
    st.nres = cnt[1] < 0 ? g.max_mols - cnt[0] : cnt[1];
    std::memcpy(st.locate, back + o.loc, sizeof(int) * g.max_mols);
    std::memcpy(st.reservoir, back + o.res, sizeof(int) * g.max_mols);
  }
  ++e->gen;
  if (bad)
    return cass_fail(e, CASS_ERR_STATE, gemc ? "a box had no free slot, or a molecule to transfer could not be regrown"
                                             : "a box reached max_molecules or could not regrow a molecule to delete");
  return CASS_OK;
}

extern "C" int cass_gcmc_run_device(cass_engine *e, int32_t nboxes, const cass_gcmc_box *boxes,
                                    cass_gcmc_state *states, int64_t nsteps, cass_gcmc_record *rec) {
  return gcmc_launch(e, nboxes, boxes, states, nsteps, rec, 1, 0, nullptr);
}

extern "C" int cass_gemc_run_device(cass_engine *e, int32_t npairs, const cass_gcmc_box *boxes,
                                    cass_gcmc_state *states, int64_t nsteps, cass_gcmc_record *rec) {
  if (npairs <= 0 || npairs > (1 << 29)) return CASS_ERR_ARG;
  return gcmc_launch(e, 2 * npairs, boxes, states, nsteps, rec, 1, 0, nullptr, true);
}

extern "C" int cass_regrow_run_device(cass_engine *e, int32_t nboxes, const cass_regrow_box *boxes, cass_rng *rngs,
                                      int64_t nsteps, cass_energy *energies, cass_nvt_record *recs) {
  if (!e || nboxes <= 0 || !boxes || !rngs || !energies || nsteps < 0) return CASS_ERR_ARG;
  if (nsteps == 0) return CASS_OK;
  HIP_TRY(e, hipSetDevice(e->device));
  auto up = [](size_t n) { return (n + 255) & ~size_t(255); };
  size_t bytes = 0;
  int maxm = 0;
  bool lj = true;
  ChainRecords pull;
  struct Offs {
    size_t rng, en, st, loc, kind, acc, ren, lp, rr;
  };
  std::vector<Offs> offs(nboxes);
  for (int i = 0; i < nboxes; ++i) {
    const cass_regrow_box &g = boxes[i];
    if (g.box < 0 || g.box >= (int)e->boxes.size()) return cass_fail(e, CASS_ERR_ARG, "bad box");
    for (int j = 0; j < i; ++j)
      if (boxes[j].box == g.box) return cass_fail(e, CASS_ERR_ARG, "a box appears twice");
    cass_box_state &b = e->boxes[g.box];
    const CbmcHostSpecies *hs = cbmc_of(e, g.species);
    if (!hs) return cass_fail(e, CASS_ERR_STATE, "no CBMC description for the species (cass_cbmc_set_species)");
    if (hs->h.nfrag < 2 || hs->h.nfbond < 1)
      return cass_fail(e, CASS_ERR_ARG, "regrowth needs a species of two or more fragments");
    if (g.nmols < 1 || !g.locate) return cass_fail(e, CASS_ERR_ARG, "no molecules to regrow");
    for (int k = 0; k < g.nmols; ++k) {
      const int m = g.first_slot + g.locate[k];
      if (g.first_slot < 0 || g.locate[k] < 0 || m >= b.nmols || b.mol_species[m] != g.species || !b.live[m])
        return cass_fail(e, CASS_ERR_ARG, "locate names a slot that is not a live molecule of the species");
    }
    if (b.p.charge_style != CASS_Q_NONE && species_has_charge(e, g.species))
      return cass_fail(e, CASS_ERR_ARG, "regrowth of a charged species is not supported on the device");
    maxm = std::max(maxm, b.nmols);
    lj = lj && lj_growth(e, b, g.species);
    bytes += up(sizeof(int64_t) * 5) + up(sizeof(double) * 14) + up(sizeof(int)) + up(sizeof(int) * g.nmols);
    if (recs) {
      const cass_nvt_record &r = recs[i];
      Offs &o = offs[i];
      if (r.kind) o.kind = pull.add(r.kind, nsteps);
      if (r.accepted) o.acc = pull.add(r.accepted, nsteps);
      if (r.energy) o.ren = pull.add(r.energy, sizeof(double) * nsteps);
      if (r.ln_pacc) o.lp = pull.add(r.ln_pacc, sizeof(double) * nsteps);
      if (r.rng_state) o.rr = pull.add(r.rng_state, sizeof(int64_t) * 5 * nsteps);
    }
  }
  bytes += up(sizeof(RegrowBoxArgs) * nboxes);
  const int list_cap = list_cap_of(maxm, 1);
  const size_t state_bytes = bytes;
  bytes += pull.staged();
  const size_t list_at = bytes;
  if (list_cap == 0) bytes += (up(kCentre * maxm) + up(sizeof(LiveMol) * maxm)) * (size_t)nboxes;
  char *s0 = (char *)cass_scratch(e, bytes + 256);
  if (!s0) return cass_fail(e, CASS_ERR_NOMEM, "scratch");
  if (int prc = pull.place(e, s0 + state_bytes)) return prc;
  std::vector<char> host(state_bytes, 0);
  size_t off = 0;
  auto take = [&](size_t n) {
    const size_t o = off;
    off += up(n);
    return o;
  };
  std::vector<RegrowBoxArgs> args(nboxes);
  for (int i = 0; i < nboxes; ++i) {
    const cass_regrow_box &g = boxes[i];
    cass_box_state &b = e->boxes[g.box];
    Offs &o = offs[i];
    o.rng = take(sizeof(int64_t) * 5);
    o.en = take(sizeof(double) * 14);
    o.st = take(sizeof(int));
    o.loc = take(sizeof(int) * g.nmols);
    std::memcpy(host.data() + o.rng, rngs[i].s, sizeof(int64_t) * 5);
    std::memcpy(host.data() + o.en, &energies[i], sizeof(double) * 14);
    std::memcpy(host.data() + o.loc, g.locate, sizeof(int) * g.nmols);
    RegrowBoxArgs &a = args[i];
    a.g = grow_args(e, b, cbmc_of(e, g.species));
    a.x = b.x;
    a.y = b.y;
    a.z = b.z;
    a.comd = b.comd;
    a.first_slot = g.first_slot;
    a.nmols = g.nmols;
    a.locate = (const int *)(s0 + o.loc);
    a.rng = (int64_t *)(s0 + o.rng);
    a.energy = (double *)(s0 + o.en);
    a.status = (int *)(s0 + o.st);
    const cass_nvt_record *r = recs ? recs + i : nullptr;
    a.kind = r && r->kind ? pull.at<uint8_t>(o.kind) : nullptr;
    a.accepted = r && r->accepted ? pull.at<uint8_t>(o.acc) : nullptr;
    a.rec_energy = r && r->energy ? pull.at<double>(o.ren) : nullptr;
    a.ln_pacc = r && r->ln_pacc ? pull.at<double>(o.lp) : nullptr;
    a.rec_rng = r && r->rng_state ? pull.at<int64_t>(o.rr) : nullptr;
    const size_t o_list = list_at + (up(kCentre * maxm) + up(sizeof(LiveMol) * maxm)) * (size_t)i;
    a.list = list_cap ? LiveList{nullptr, nullptr, 0}
                      : LiveList{(LiveMol *)(s0 + o_list + up(kCentre * maxm)), (double *)(s0 + o_list), maxm};
  }
  const size_t o_args = take(sizeof(RegrowBoxArgs) * nboxes);
  if (off != state_bytes) return cass_fail(e, CASS_ERR_STATE, "regrowth state layout differs from its buffer");
  MirrorPull mirrors;
  std::vector<int> ids(nboxes);
  for (int i = 0; i < nboxes; ++i) ids[i] = boxes[i].box;
  if (int mrc = mirrors.reserve(e, ids, false, off + pull.staged())) return mrc;
  std::memcpy(host.data() + o_args, args.data(), sizeof(RegrowBoxArgs) * nboxes);
  HIP_TRY(e, hipMemcpyAsync(s0, host.data(), off, hipMemcpyHostToDevice, e->stream));
  HIP_TRY(e, hipEventRecord(e->ev0, e->stream));
  const RegrowBoxArgs *d_args = (const RegrowBoxArgs *)(s0 + o_args);
  const int nt = 512;  // 60 moves of 48 pentane boxes: 5.6 ms with 4 waves, 3.8 ms with 8
  const int rc = launch_chain(e, growth_kernels(e, lj).regrow, d_args, nboxes, nt, nsteps, list_cap,
                              1, "k_regrow_chain launch");
  if (rc) return rc;
  HIP_TRY(e, hipEventRecord(e->ev1, e->stream));
  if (int mrc = mirrors.queue(e)) return mrc;
  HIP_TRY(e, hipMemcpyAsync(mirrors.host, s0, off + pull.staged(), hipMemcpyDeviceToHost, e->stream));
  if (int prc = pull.queue(e)) return prc;
  HIP_TRY(e, hipStreamSynchronize(e->stream));
  mirrors.end(e);
  pull.end(mirrors.host + off);
  const char *back = mirrors.host;
  float ms = 0.f;
  if (hipEventElapsedTime(&ms, e->ev0, e->ev1) == hipSuccess) e->last_kernel_ms = ms;
  int bad = 0;
  for (int i = 0; i < nboxes; ++i) {
    const Offs &o = offs[i];
    std::memcpy(rngs[i].s, back + o.rng, sizeof(int64_t) * 5);
    std::memcpy(&energies[i], back + o.en, sizeof(double) * 14);
    int st;
    std::memcpy(&st, back + o.st, sizeof(int));
    bad |= st;
  }
  ++e->gen;
  if (bad) return cass_fail(e, CASS_ERR_STATE, "a molecule's own configuration could not be regrown (the reference aborts)");
  return CASS_OK;
}

// Times the chain with 128, 256, 512 and 1024 lanes per box on timing runs
// of nsteps moves that leave every box untouched, and keeps the fastest for
// the engine's later cass_gcmc_run_device calls.
extern "C" int cass_gcmc_autotune(cass_engine *e, int32_t nboxes, const cass_gcmc_box *boxes,
                                  cass_gcmc_state *states, int64_t nsteps, int32_t *block) {
  if (!e || nsteps <= 0) return CASS_ERR_ARG;
  const int cand[4] = {128, 256, 512, 1024};
  double best = 1e300;
  int best_nt = 256;
  for (int nt : cand) {
    double ms = 0.0;
    if (int rc = gcmc_launch(e, nboxes, boxes, states, nsteps, nullptr, 0, nt, &ms)) return rc;
    if (ms < best) {
      best = ms;
      best_nt = nt;
    }
  }
  gcmc_block(e) = best_nt;
  if (block) *block = best_nt;
  return CASS_OK;
}
