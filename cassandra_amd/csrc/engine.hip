// engine.hip -- host side of the C ABI (include/cass_gpu.h): device state,
// uploads and kernel launches.  One HIP stream per engine; every entry point
// that returns values synchronises on it.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "engine.h"
#include "kernels.h"

using namespace cass;


int cass_fail(cass_engine *e, int code, const std::string &msg) {
  if (e) e->err = msg;
  return code;
}

int cass_check_hip(cass_engine *e, hipError_t st, const char *what) {
  if (st == hipSuccess) return CASS_OK;
  return cass_fail(e, st == hipErrorOutOfMemory ? CASS_ERR_NOMEM : CASS_ERR_HIP,
                   std::string(what) + ": " + hipGetErrorString(st));
}

void *cass_scratch(cass_engine *e, size_t bytes) {
  if (bytes <= e->scratch_bytes) return e->scratch;
  if (e->scratch) {
    (void)hipStreamSynchronize(e->stream);
    (void)hipFree(e->scratch);
  }
  e->scratch = nullptr;
  e->scratch_bytes = 0;
  size_t want = std::max(bytes, (size_t)1 << 20);
  if (hipMalloc(&e->scratch, want) != hipSuccess) return nullptr;
  e->scratch_bytes = want;
  return e->scratch;
}

// For tests of a failed allocation: pinned staging beyond `bytes` is refused.
extern "C" void cass_test_pinned_limit(cass_engine *e, size_t bytes) { e->pinned_limit = bytes; }

void *cass_pinned(cass_engine *e, size_t bytes) {
  if (bytes > e->pinned_limit) return nullptr;
  if (bytes <= e->pinned_bytes) return e->pinned;
  if (e->pinned) {
    (void)hipStreamSynchronize(e->stream);
    (void)hipHostFree(e->pinned);
  }
  e->pinned = nullptr;
  e->pinned_bytes = 0;
  size_t want = std::max(bytes, (size_t)1 << 16);
  if (hipHostMalloc(&e->pinned, want, hipHostMallocDefault) != hipSuccess) return nullptr;
  e->pinned_bytes = want;
  return e->pinned;
}

void *cass_io(cass_engine *e, size_t bytes) {
  if (bytes <= e->io_bytes) return e->io;
  if (e->io) {
    (void)hipStreamSynchronize(e->stream);
    (void)hipFree(e->io);
  }
  e->io = nullptr;
  e->io_bytes = 0;
  size_t want = std::max(bytes, (size_t)1 << 16);
  if (hipMalloc(&e->io, want) != hipSuccess) return nullptr;
  e->io_bytes = want;
  return e->io;
}

template <typename X>
static hipError_t dalloc(X **p, size_t n) {
  return hipMalloc((void **)p, std::max<size_t>(n, 1) * sizeof(X));
}

template <typename X>
static hipError_t upload(cass_engine *e, X *dst, const X *src, size_t n) {
  if (n == 0) return hipSuccess;
  return hipMemcpyAsync(dst, src, n * sizeof(X), hipMemcpyHostToDevice, e->stream);
}

static BoxDev box_view(const cass_engine *e, const cass_box_state &b) {
  BoxDev v;
  v.x = b.x;
  v.y = b.y;
  v.z = b.z;
  v.first = b.d_first;
  v.species = b.d_species;
  v.live = b.d_live;
  v.comd = b.comd;
  v.nmols = b.nmols;
  v.cubic = b.p.box_shape == CASS_BOX_CUBIC;
  v.vdw_minimum = b.p.vdw_sum_style == CASS_SUM_MINIMUM;
  for (int k = 0; k < 3; ++k) {
    v.L[k] = b.p.cell[4 * k];
    v.hL[k] = b.p.hlength[k];
  }
  for (int k = 0; k < 9; ++k) {
    v.Li[k] = b.p.length_inv[k];
    v.Lc[k] = b.p.cell[k];
  }
  v.rcut_max = b.p.rcut_max;
  v.rcut_cbmc = b.p.rcut_cbmc;
  v.apt = b.apt;
  v.apt_res = b.apt ? b.apt_res : 0;
  v.apt_step = b.apt_step;
  v.apt_shift = b.apt_shift;
  v.apt_rcs = b.apt_rcs;
  (void)e;
  return v;
}

static TopoDev topo_view(const cass_engine *e) {
  TopoDev t;
  t.eps = e->d_eps;
  t.sig = e->d_sig;
  t.mn = e->d_mn;
  t.mm = e->d_mm;
  t.atom_type = e->d_atom_type;
  t.atom_charge = e->d_atom_charge;
  t.atom_mass = e->d_atom_mass;
  t.sp_natoms = e->d_sp_natoms;
  t.sp_atom_off = e->d_sp_atom_off;
  t.sp_coul_cbmc = e->d_sp_coul_cbmc;
  t.ntypes = e->ntypes;
  t.nspecies = e->nspecies;
  t.natoms_total = e->natoms_total;
  return t;
}

static EwaldDev ewald_view(const cass_box_state &b, const int *row_k0) {
  EwaldDev w;
  w.nvecs = b.nvecs;
  w.nrows = b.nrows;
  w.hx = b.hx;
  w.hy = b.hy;
  w.hz = b.hz;
  w.cn = b.cn;
  w.cs = b.cs;
  w.sn = b.sn;
  w.cmol = b.cmol;
  w.smol = b.smol;
  w.cs_new = b.cs_new;
  w.sn_new = b.sn_new;
  w.cm_new = b.cm_new;
  w.sm_new = b.sm_new;
  w.rows = b.rows;
  w.row_k0 = row_k0;
  w.kperm = row_k0 ? row_k0 + b.nrows : nullptr;
  w.segs = b.segs();
  w.nsegs = b.nsegs;
  w.tx = std::max(2, b.kmax[0] + 1);
  w.ty = b.kmax[1] + 1;
  w.tz = b.kmax[2] + 1;
  return w;
}

// traversal position of each k row's first vector, stored after the rows
static const int *row_k0_of(const cass_box_state &b) { return (const int *)(b.rows + b.nrows + b.nsegs); }
BoxDev cass_box_view(const cass_engine *e, const cass_box_state &b) { return box_view(e, b); }
TopoDev cass_topo_view(const cass_engine *e) { return topo_view(e); }
EwaldDev cass_ewald_view(const cass_box_state &b) {
  return ewald_view(b, b.rows ? row_k0_of(b) : nullptr);
}

static bool species_charged(const cass_engine *e, int s) {
  for (int a = 0; a < e->sp_natoms[s]; ++a)
    if (e->atom_charge[e->sp_atom_off[s] + a] != 0.0) return true;
  return false;
}

// Workgroups that share one molecule's structure-factor sums in
// ewald_mol_block: one where the molecules of the call alone fill the chip, else
// as many as bring them to 512, and at most one per 256 segments.  With one
// each, 4 waters and 56000 vectors took 100 us a call (31 shared), 128 took 130
// (81); 512 waters take the same 53 us either way.
static int ewald_parts(const cass_box_state &b, int call_mols) {
  return std::max(1, std::min((b.nsegs + kMaxBlock - 1) / kMaxBlock, 512 / std::max(1, call_mols)));
}

// Whether a box has molecules of the two ways to take those sums.
static void ewald_ways(const cass_engine *e, const cass_box_state &b, const EwaldDev &ew, bool &tabled, bool &direct) {
  tabled = direct = false;
  for (int m = 0; m < b.nmols; ++m)
    (ewald_direct(ew, b.nmols, e->sp_natoms[b.mol_species[m]]) ? direct : tabled) = true;
}

// ------------------------------------------------------------------ setup
static int noalloc_init(cass_engine *e);

extern "C" int cass_engine_create(int32_t device, const cass_topology *t, int32_t max_boxes,
                                  cass_engine **out) {
  if (!t || !out || max_boxes <= 0 || t->ntypes < 1 || t->nspecies < 1) return CASS_ERR_ARG;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return CASS_ERR_NODEVICE;
  if (device < 0 || device >= ndev) return CASS_ERR_ARG;
  if (hipSetDevice(device) != hipSuccess) return CASS_ERR_HIP;
  cass_engine *e = new cass_engine();
  e->device = device;
  e->max_boxes = max_boxes;
  if (hipStreamCreateWithFlags(&e->stream, hipStreamNonBlocking) != hipSuccess ||
      hipStreamCreateWithFlags(&e->side, hipStreamNonBlocking) != hipSuccess ||
      hipEventCreateWithFlags(&e->ev_join, hipEventDisableTiming) != hipSuccess ||
      hipEventCreate(&e->ev0) != hipSuccess || hipEventCreate(&e->ev1) != hipSuccess ||
      hipEventCreate(&e->evs[0]) != hipSuccess || hipEventCreate(&e->evs[1]) != hipSuccess ||
      hipEventCreate(&e->evs[2]) != hipSuccess || hipEventCreate(&e->evs[3]) != hipSuccess) {
    delete e;
    return CASS_ERR_HIP;
  }
  e->ntypes = t->ntypes;
  e->nspecies = t->nspecies;
  const size_t nt2 = (size_t)t->ntypes * t->ntypes;
  e->eps.assign(t->eps, t->eps + nt2);
  e->sig.assign(t->sig, t->sig + nt2);
  e->mie_n = t->mie_n ? std::vector<double>(t->mie_n, t->mie_n + nt2) : std::vector<double>(nt2, 0.0);
  e->mie_m = t->mie_m ? std::vector<double>(t->mie_m, t->mie_m + nt2) : std::vector<double>(nt2, 0.0);
  e->sp_natoms.assign(t->species_natoms, t->species_natoms + t->nspecies);
  e->sp_atom_off.assign(t->species_atom_offset, t->species_atom_offset + t->nspecies);
  e->sp_pair_off.assign(t->species_pair_offset, t->species_pair_offset + t->nspecies);
  e->sp_coul_cbmc.assign(t->species_coul_cbmc, t->species_coul_cbmc + t->nspecies);
  int na = 0, np = 0;
  for (int s = 0; s < t->nspecies; ++s) {
    if (t->species_natoms[s] > kMaxSites) {
      delete e;
      return CASS_ERR_ARG;
    }
    na = std::max(na, t->species_atom_offset[s] + t->species_natoms[s]);
    np = std::max(np, t->species_pair_offset[s] + t->species_natoms[s] * t->species_natoms[s]);
  }
  e->natoms_total = na;
  e->atom_type.assign(t->atom_type, t->atom_type + na);
  e->atom_charge.assign(t->atom_charge, t->atom_charge + na);
  e->atom_mass.assign(t->atom_mass, t->atom_mass + na);
  e->vdw_scale.assign(t->vdw_intra_scale, t->vdw_intra_scale + np);
  e->q_scale.assign(t->charge_intra_scale, t->charge_intra_scale + np);
  e->bonded.assign(t->bonded, t->bonded + np);
  HIP_TRY(e, dalloc(&e->d_eps, nt2));
  HIP_TRY(e, dalloc(&e->d_sig, nt2));
  HIP_TRY(e, dalloc(&e->d_mn, nt2));
  HIP_TRY(e, dalloc(&e->d_mm, nt2));
  HIP_TRY(e, dalloc(&e->d_atom_type, na));
  HIP_TRY(e, dalloc(&e->d_atom_charge, na));
  HIP_TRY(e, dalloc(&e->d_atom_mass, na));
  HIP_TRY(e, dalloc(&e->d_sp_natoms, t->nspecies));
  HIP_TRY(e, dalloc(&e->d_sp_atom_off, t->nspecies));
  HIP_TRY(e, dalloc(&e->d_sp_coul_cbmc, t->nspecies));
  HIP_TRY(e, upload(e, e->d_eps, e->eps.data(), nt2));
  HIP_TRY(e, upload(e, e->d_sig, e->sig.data(), nt2));
  HIP_TRY(e, upload(e, e->d_mn, e->mie_n.data(), nt2));
  HIP_TRY(e, upload(e, e->d_mm, e->mie_m.data(), nt2));
  HIP_TRY(e, upload(e, e->d_atom_type, e->atom_type.data(), na));
  HIP_TRY(e, upload(e, e->d_atom_charge, e->atom_charge.data(), na));
  HIP_TRY(e, upload(e, e->d_atom_mass, e->atom_mass.data(), na));
  HIP_TRY(e, upload(e, e->d_sp_natoms, e->sp_natoms.data(), t->nspecies));
  HIP_TRY(e, upload(e, e->d_sp_atom_off, e->sp_atom_off.data(), t->nspecies));
  HIP_TRY(e, upload(e, e->d_sp_coul_cbmc, e->sp_coul_cbmc.data(), t->nspecies));
  HIP_TRY(e, hipStreamSynchronize(e->stream));
  e->boxes.reserve(max_boxes);
  if (int rc = noalloc_init(e)) return rc;
  *out = e;
  return CASS_OK;
}

static void free_box(cass_box_state &b) {
  void *ps[] = {b.x, b.y, b.z, b.site_spa, b.d_first, b.d_species, b.d_live, b.comd, b.hx, b.hy, b.hz,
                b.cn, b.cs, b.sn, b.cmol, b.smol, b.cs_new, b.sn_new, b.cm_new, b.sm_new, b.rows, b.apt};
  for (void *p : ps)
    if (p) (void)hipFree(p);
}

extern "C" int cass_engine_destroy(cass_engine *e) {
  if (!e) return CASS_OK;
  (void)hipSetDevice(e->device);
  (void)hipStreamSynchronize(e->stream);
  cass_cbmc_release(e);
  for (auto &b : e->boxes) free_box(b);
  void *ps[] = {e->d_eps, e->d_sig, e->d_mn, e->d_mm, e->d_atom_type, e->d_atom_charge, e->d_atom_mass,
                e->d_sp_natoms, e->d_sp_atom_off, e->d_sp_coul_cbmc, e->scratch, e->io, e->wtab.dev,
                e->adjf.dev};
  for (void *p : ps)
    if (p) (void)hipFree(p);
  if (e->pinned) (void)hipHostFree(e->pinned);
  (void)hipEventDestroy(e->ev0);
  (void)hipEventDestroy(e->ev1);
  for (hipEvent_t ev : e->evs)
    if (ev) (void)hipEventDestroy(ev);
  if (e->ev_join) (void)hipEventDestroy(e->ev_join);
  if (e->side) (void)hipStreamDestroy(e->side);
  (void)hipStreamDestroy(e->stream);
  delete e;
  return CASS_OK;
}

// AtomPair_VdW_Energy_Vector (energy_routines.f90:1733-1829) at one r^2 for
// type pair k, in the reference's operation order.
static double vdw_table_entry(const cass_engine *e, const cass_params &p, int k, double r2) {
  const double eps = e->eps[k], sig = e->sig[k];
  if (p.vdw_style == CASS_VDW_LJ) {
    const double s2 = (sig * sig) / r2, s6 = s2 * s2 * s2, s12 = s6 * s6;
    double v = 4.0 * eps * (s12 - s6);
    if (p.vdw_sum_style == CASS_SUM_CUT_SHIFT) {
      const double c2 = sig * sig / p.rcut_vdwsq, c6 = c2 * c2 * c2, c12 = c6 * c6;
      v = v - 4.0 * eps * (c12 - c6);
    } else if (p.vdw_sum_style == CASS_SUM_CUT_SWITCH) {
      if (r2 < p.ron_switch_sq) {
      } else if (r2 > p.roff_switch_sq) {
        v = 0.0;
      } else {
        const double d = p.roff_switch_sq - r2;
        v = d * d * (p.switch_factor2 + 2.0 * r2) * p.switch_factor1 * v;
      }
    } else if (p.vdw_sum_style == CASS_SUM_CHARMM) {
      v = eps * (s12 - 2.0 * s6);
    } else if (p.vdw_sum_style == CASS_SUM_CUT_SHIFT_FORCE) {
      const double c2 = sig * sig / p.rcut_vdwsq, c6 = c2 * c2 * c2, c12 = c6 * c6;
      const double rc = std::sqrt(p.rcut_vdwsq);
      const double de = -(24.0 * eps * (2.0 * c12 - c6) / rc);
      v = v - 4.0 * eps * (c12 - c6) - (std::sqrt(r2) - rc) * de;
    }
    return v;
  }
  if (p.vdw_style == CASS_VDW_MIE) {
    const double n = e->mie_n[k], m = e->mie_m[k];
    const double rc = std::sqrt(p.rcut_vdwsq);
    const double coeff = n / (n - m) * std::pow(n / m, m / (n - m));
    const double sr = sig / std::sqrt(r2);
    double v = coeff * eps * (std::pow(sr, n) - std::pow(sr, m));
    if (p.vdw_sum_style == CASS_SUM_CUT_SHIFT) {
      const double sc = sig / rc;
      v = v - coeff * eps * (std::pow(sc, n) - std::pow(sc, m));
    }
    return v;
  }
  return 0.0;
}

// Create_Atompair_Nrg_table (atompair_nrg_table_routines.f90:149-261) for
// one box: bins of width rsq_step = (max rcut_cbmc^2 - rcut_low^2) / res from
// rsq_shifter = rcut_low^2 - rsq_step, each evaluated at its midpoint; the
// vdW of every type pair and the charge factor f2 of the box's charge style
// (libm erfc, which the Fortran ERFC intrinsic calls).  The q_i q_j factor is
// applied at lookup.  Every species acts as both solute and solvent.
static int build_energy_table(cass_engine *e, cass_box_state &b) {
  const cass_params &p = b.p;
  const int res = b.apt_res, nt = e->ntypes;
  const double rsq_step = (b.apt_rcsq_max - p.rcut_lowsq) / res;
  const double rsq_shifter = p.rcut_lowsq - rsq_step;
  std::vector<double> mp(res), h((size_t)(nt * nt + 1) * res);
  for (int i = 1; i <= res; ++i) {
    const double lb = rsq_shifter + rsq_step * i;
    mp[i - 1] = lb + 0.5 * rsq_step;
  }
  for (int k = 0; k < nt * nt; ++k)
    for (int i = 0; i < res; ++i) h[(size_t)k * res + i] = vdw_table_entry(e, p, k, mp[i]);
  double *f2 = h.data() + (size_t)nt * nt * res;
  for (int i = 0; i < res; ++i) {
    const double rij = std::sqrt(mp[i]);
    if (p.charge_style == CASS_Q_EWALD) {
      f2[i] = std::erfc(p.alpha_ewald * rij) / rij;
    } else if (p.charge_style == CASS_Q_DSF) {
      f2[i] = p.dsf_factor2 * (rij - p.rcut_coul) - p.dsf_factor1 + std::erfc(p.alpha_dsf * rij) / rij;
    } else if (p.charge_style == CASS_Q_CUT) {
      f2[i] = 1.0 / rij;
    } else {
      f2[i] = 0.0;
    }
  }
  if (!b.apt) HIP_TRY(e, hipMalloc((void **)&b.apt, sizeof(double) * h.size()));
  HIP_TRY(e, hipMemcpy(b.apt, h.data(), sizeof(double) * h.size(), hipMemcpyHostToDevice));
  b.apt_step = rsq_step;
  b.apt_shift = rsq_shifter;
  b.apt_rcs = p.rcut_cbmcsq - rsq_shifter;
  return CASS_OK;
}

extern "C" int cass_set_energy_table(cass_engine *e, int32_t box, int32_t res, double rcut_cbmcsq_max) {
  if (!e || box < 0 || box >= (int32_t)e->boxes.size() || res < 0) return CASS_ERR_ARG;
  HIP_TRY(e, hipSetDevice(e->device));
  HIP_TRY(e, hipStreamSynchronize(e->stream));
  cass_box_state &b = e->boxes[box];
  if (res == 0) {
    if (b.apt) HIP_TRY(e, hipFree(b.apt));
    b.apt = nullptr;
    b.apt_res = 0;
    return CASS_OK;
  }
  const double rmax = rcut_cbmcsq_max > 0.0 ? rcut_cbmcsq_max : b.p.rcut_cbmcsq;
  if (!(rmax >= b.p.rcut_cbmcsq) || !(rmax > b.p.rcut_lowsq))
    return cass_fail(e, CASS_ERR_ARG, "energy table: need max rcut_cbmc^2 >= this box's and > rcut_low^2");
  if (b.apt && b.apt_res != res) {
    HIP_TRY(e, hipFree(b.apt));
    b.apt = nullptr;
  }
  b.apt_res = res;
  b.apt_rcsq_max = rmax;
  return build_energy_table(e, b);
}

// The type-pair core radii^2 of calc_rmin (create_nonbond_table.f90:285-301,
// 398-417): rcut_low^2 unless the pair's eps > 0, then sig^2 / lambda^(1/3)
// with lambda = (1 + sqrt(1 + U_max / eps)) / 2, the r where the LJ energy
// reaches U_max = max(U_max_base - min_U_q, 0); min_U_q is the most negative
// Coulomb energy the two types' charge ranges allow (at rcut_low for
// opposite signs, at sigma otherwise).  Charge ranges per type over every
// species' atoms (:143-152).
extern "C" int cass_rminsq_table(cass_engine *e, int32_t box, double u_max_base, double *rminsq) {
  if (!e || box < 0 || box >= (int32_t)e->boxes.size() || !rminsq) return CASS_ERR_ARG;
  const cass_params &p = e->boxes[box].p;
  const int nt = e->ntypes;
  std::vector<double> cmin(nt, 0.0), cmax(nt, 0.0);
  std::vector<bool> seen(nt, false);
  for (int a = 0; a < e->natoms_total; ++a) {
    const int t = e->atom_type[a];
    if (t < 0) continue;
    const double q = e->atom_charge[a];
    cmin[t] = seen[t] ? std::min(cmin[t], q) : q;
    cmax[t] = seen[t] ? std::max(cmax[t], q) : q;
    seen[t] = true;
  }
  const double rcut_low = std::sqrt(p.rcut_lowsq);
  for (int i = 0; i < nt; ++i)
    for (int j = 0; j < nt; ++j) {
      const size_t k = (size_t)i * nt + j;
      rminsq[k] = p.rcut_lowsq;
      const double eps = e->eps[k], sig = e->sig[k];
      if (!(eps > 0.0)) continue;
      double min_u_q = 0.0;
      if (p.charge_style != CASS_Q_NONE) {
        double qp = std::min(cmin[i] * cmax[j], cmax[i] * cmin[j]);
        if (qp <= 0.0) {
          min_u_q = qp * kChargeFactor / rcut_low;
        } else {
          qp = std::min(cmin[i] * cmin[j], cmax[i] * cmax[j]);
          min_u_q = qp * kChargeFactor / sig;
        }
      }
      const double u_max = std::max(u_max_base - min_u_q, 0.0);
      const double lambda = 0.5 * (1.0 + std::sqrt(1.0 + u_max / eps));
      rminsq[k] = sig * sig / std::pow(lambda, 1.0 / 3.0);
    }
  return CASS_OK;
}

extern "C" int cass_widom_set_rminsq(cass_engine *e, int32_t box, const double *rminsq) {
  if (!e || box < 0 || box >= (int32_t)e->boxes.size()) return CASS_ERR_ARG;
  cass_box_state &b = e->boxes[box];
  if (rminsq)
    b.rminsq.assign(rminsq, rminsq + (size_t)e->ntypes * e->ntypes);
  else
    b.rminsq.clear();
  ++e->gen;
  return CASS_OK;
}

extern "C" int cass_set_nonbond_params(cass_engine *e, const double *eps, const double *sig,
                                       const double *atom_charge) {
  if (!e) return CASS_ERR_ARG;
  HIP_TRY(e, hipSetDevice(e->device));
  HIP_TRY(e, hipStreamSynchronize(e->stream));
  const size_t nt2 = (size_t)e->ntypes * e->ntypes;
  if (eps) {
    e->eps.assign(eps, eps + nt2);
    HIP_TRY(e, upload(e, e->d_eps, e->eps.data(), nt2));
  }
  if (sig) {
    e->sig.assign(sig, sig + nt2);
    HIP_TRY(e, upload(e, e->d_sig, e->sig.data(), nt2));
  }
  if (atom_charge) {
    e->atom_charge.assign(atom_charge, atom_charge + e->natoms_total);
    HIP_TRY(e, upload(e, e->d_atom_charge, e->atom_charge.data(), e->natoms_total));
  }
  HIP_TRY(e, hipStreamSynchronize(e->stream));
  for (auto &b : e->boxes) {
    b.ewald_ready = b.ewald_ready && !atom_charge;
    if (b.apt) {
      const int rc = build_energy_table(e, b);
      if (rc != CASS_OK) return rc;
    }
  }
  ++e->gen;
  return CASS_OK;
}

extern "C" int cass_set_precision(cass_engine *e, int32_t prec) {
  if (!e || (prec != CASS_PREC_FP64 && prec != CASS_PREC_MIXED && prec != CASS_PREC_FP32)) return CASS_ERR_ARG;
  e->prec = prec;
  ++e->gen;
  return CASS_OK;
}

extern "C" int cass_set_overlap(cass_engine *e, int32_t on) {
  if (!e) return CASS_ERR_ARG;
  e->overlap = on ? 1 : 0;
  return CASS_OK;
}

extern "C" const char *cass_last_error(cass_engine *e) { return e ? e->err.c_str() : "no engine"; }

extern "C" int cass_last_kernel_ms(cass_engine *e, double *ms) {
  if (!e || !ms) return CASS_ERR_ARG;
  *ms = e->last_kernel_ms;
  return CASS_OK;
}

extern "C" int cass_last_stage_ms(cass_engine *e, double *ms) {
  if (!e || !ms) return CASS_ERR_ARG;
  for (int k = 0; k < 4; ++k) ms[k] = e->last_stage_ms[k];
  return CASS_OK;
}

// The checks the reference makes on a box's cell and cutoffs: the shape
// keyword against the cell matrix (cubic: equal diagonal, no off-diagonal
// entries; orthogonal: no off-diagonal entries), and every cutoff against
// half the box, as Get_Pair_Style does at start-up
// (input_routines.f90:466-471, 491-496) and Volume_Change after a volume
// move (move_volume.f90:283-292: rcut_vdw, rcut_coul, the CHARMM and switch
// outer radii).
static int check_box_params(cass_engine *e, const cass_params &p) {
  if (p.box_shape != CASS_BOX_CUBIC && p.box_shape != CASS_BOX_ORTHO && p.box_shape != CASS_BOX_CELL)
    return cass_fail(e, CASS_ERR_ARG, "unknown box shape");
  if (p.box_shape != CASS_BOX_CELL) {
    const double *c = p.cell;  // column-major 3x3
    if (c[1] != 0.0 || c[2] != 0.0 || c[3] != 0.0 || c[5] != 0.0 || c[6] != 0.0 || c[7] != 0.0)
      return cass_fail(e, CASS_ERR_ARG, "cubic/orthogonal box with off-diagonal cell entries");
    if (p.box_shape == CASS_BOX_CUBIC && (c[0] != c[4] || c[0] != c[8]))
      return cass_fail(e, CASS_ERR_ARG, "cubic box with unequal edges");
  }
  const double half = 0.5 * std::min({p.basis_length[0], p.basis_length[1], p.basis_length[2]}) * (1 + 1e-12);
  if (!(half > 0.0)) return cass_fail(e, CASS_ERR_ARG, "box lengths not derived (cass_params_derive)");
  if (p.vdw_style != CASS_VDW_NONE && p.vdw_sum_style != CASS_SUM_MINIMUM && p.rcut_vdw > half)
    return cass_fail(e, CASS_ERR_CUTOFF, "vdW cutoff exceeds half the box");
  if ((p.vdw_sum_style == CASS_SUM_CUT_SWITCH || p.vdw_sum_style == CASS_SUM_CHARMM) && p.roff_switch > half)
    return cass_fail(e, CASS_ERR_CUTOFF, "switch outer radius exceeds half the box");
  if ((p.charge_style == CASS_Q_EWALD || p.charge_style == CASS_Q_DSF || p.charge_style == CASS_Q_CUT) &&
      p.rcut_coul > half)
    return cass_fail(e, CASS_ERR_CUTOFF, "Coulomb cutoff exceeds half the box");
  return CASS_OK;
}

extern "C" int cass_box_create(cass_engine *e, const cass_params *p, int32_t max_mols, int32_t *box) {
  if (!e || !p || !box || max_mols <= 0) return CASS_ERR_ARG;
  if ((int)e->boxes.size() >= e->max_boxes) return cass_fail(e, CASS_ERR_ARG, "max_boxes reached");
  if (int rc = check_box_params(e, *p)) return rc;
  HIP_TRY(e, hipSetDevice(e->device));
  e->boxes.emplace_back();
  ++e->gen;
  cass_box_state &b = e->boxes.back();
  b.p = *p;
  b.cap_mols = max_mols;
  int maxn = *std::max_element(e->sp_natoms.begin(), e->sp_natoms.end());
  b.cap_sites = max_mols * maxn;
  HIP_TRY(e, dalloc(&b.x, b.cap_sites));
  HIP_TRY(e, dalloc(&b.y, b.cap_sites));
  HIP_TRY(e, dalloc(&b.z, b.cap_sites));
  HIP_TRY(e, dalloc(&b.site_spa, b.cap_sites));
  HIP_TRY(e, dalloc(&b.d_first, max_mols));
  HIP_TRY(e, dalloc(&b.d_species, max_mols));
  HIP_TRY(e, dalloc(&b.d_live, max_mols));
  HIP_TRY(e, dalloc(&b.comd, max_mols));
  *box = (int32_t)e->boxes.size() - 1;
  return CASS_OK;
}

// A box's geometry after a volume change (move_volume.f90:374-426 scales the
// cell, then recomputes the cell dimensions, the k vectors and the total
// energy).  The reciprocal sums become stale until cass_ewald_setup; the
// caller uploads the rescaled coordinates with cass_box_upload.
extern "C" int cass_box_set_params(cass_engine *e, int32_t box, const cass_params *p) {
  if (!e || !p || box < 0 || box >= (int32_t)e->boxes.size()) return CASS_ERR_ARG;
  if (int rc = check_box_params(e, *p)) return rc;
  HIP_TRY(e, hipSetDevice(e->device));
  HIP_TRY(e, hipStreamSynchronize(e->stream));
  cass_box_state &b = e->boxes[box];
  if (b.apt && !(b.apt_rcsq_max >= p->rcut_cbmcsq && b.apt_rcsq_max > p->rcut_lowsq))
    return cass_fail(e, CASS_ERR_ARG, "the pair table's range no longer covers rcut_cbmc; reset it first");
  b.p = *p;
  b.ewald_ready = false;
  ++e->gen;
  return b.apt ? build_energy_table(e, b) : CASS_OK;
}

static int box_of(cass_engine *e, int32_t box, cass_box_state **out) {
  if (!e) return CASS_ERR_ARG;
  if (box < 0 || box >= (int)e->boxes.size()) return cass_fail(e, CASS_ERR_ARG, "bad box index");
  *out = &e->boxes[box];
  return hipSetDevice(e->device) == hipSuccess ? CASS_OK : CASS_ERR_HIP;
}

double4 cass_host_com(const cass_engine *e, int s, const double *xyz) {
  const int o = e->sp_atom_off[s], n = e->sp_natoms[s];
  double tm = 0, cx = 0, cy = 0, cz = 0;
  for (int a = 0; a < n; ++a) {
    const double m = e->atom_mass[o + a];
    tm = tm + m;
    cx = cx + m * xyz[3 * a];
    cy = cy + m * xyz[3 * a + 1];
    cz = cz + m * xyz[3 * a + 2];
  }
  cx = cx / tm;
  cy = cy / tm;
  cz = cz / tm;
  double dmax = 0;
  for (int a = 0; a < n; ++a) {
    const double dx = xyz[3 * a] - cx, dy = xyz[3 * a + 1] - cy, dz = xyz[3 * a + 2] - cz;
    dmax = std::max(dmax, dx * dx + dy * dy + dz * dz);
  }
  return make_double4(cx, cy, cz, std::sqrt(dmax));
}

extern "C" int cass_box_upload(cass_engine *e, int32_t box, int32_t nmols, const int32_t *mol_species,
                               const int32_t *live, const double *xyz, const double *com,
                               const double *max_dcom) {
  cass_box_state *b;
  int rc = box_of(e, box, &b);
  if (rc) return rc;
  if (nmols < 0 || nmols > b->cap_mols) return cass_fail(e, CASS_ERR_ARG, "nmols exceeds box capacity");
  ++e->gen;
  b->nmols = nmols;
  b->mol_species.assign(mol_species, mol_species + nmols);
  b->live.assign(live, live + nmols);
  b->mol_first.resize(nmols);
  int ns = 0;
  for (int m = 0; m < nmols; ++m) {
    if (mol_species[m] < 0 || mol_species[m] >= e->nspecies) return cass_fail(e, CASS_ERR_ARG, "bad species");
    b->mol_first[m] = ns;
    ns += e->sp_natoms[mol_species[m]];
  }
  b->nsites = ns;
  for (size_t k = 0; k < 3 * (size_t)ns; ++k)
    if (!std::isfinite(xyz[k])) return cass_fail(e, CASS_ERR_ARG, "non-finite coordinate");
  b->xyz_h.assign(xyz, xyz + 3 * (size_t)ns);
  std::vector<double> xs(ns), ys(ns), zs(ns);
  std::vector<int32_t> spa(ns);
  std::vector<double4> cd(nmols);
  for (int m = 0; m < nmols; ++m) {
    const int s = mol_species[m], f = b->mol_first[m];
    for (int a = 0; a < e->sp_natoms[s]; ++a) {
      xs[f + a] = xyz[3 * (f + a)];
      ys[f + a] = xyz[3 * (f + a) + 1];
      zs[f + a] = xyz[3 * (f + a) + 2];
      spa[f + a] = e->sp_atom_off[s] + a;
    }
    double4 c = cass_host_com(e, s, xyz + 3 * f);
    if (com) c = make_double4(com[3 * m], com[3 * m + 1], com[3 * m + 2], c.w);
    if (max_dcom) c.w = max_dcom[m];
    cd[m] = c;
  }
  HIP_TRY(e, upload(e, b->x, xs.data(), ns));
  HIP_TRY(e, upload(e, b->y, ys.data(), ns));
  HIP_TRY(e, upload(e, b->z, zs.data(), ns));
  HIP_TRY(e, upload(e, b->site_spa, spa.data(), ns));
  HIP_TRY(e, upload(e, b->d_first, b->mol_first.data(), nmols));
  HIP_TRY(e, upload(e, b->d_species, b->mol_species.data(), nmols));
  HIP_TRY(e, upload(e, b->d_live, b->live.data(), nmols));
  HIP_TRY(e, upload(e, b->comd, cd.data(), nmols));
  HIP_TRY(e, hipStreamSynchronize(e->stream));
  b->comd_h = cd;
  b->ewald_ready = false;
  return CASS_OK;
}

extern "C" int cass_mol_update(cass_engine *e, int32_t box, int32_t mol, int32_t live, const double *xyz,
                               const double *com, const double *max_dcom) {
  cass_box_state *b;
  int rc = box_of(e, box, &b);
  if (rc) return rc;
  if (mol < 0 || mol >= b->nmols) return cass_fail(e, CASS_ERR_ARG, "bad molecule index");
  const int s = b->mol_species[mol], n = e->sp_natoms[s], f = b->mol_first[mol];
  ++e->gen;
  // one pinned staging buffer: x[n], y[n], z[n], comd, live
  double *h = (double *)cass_pinned(e, sizeof(double) * (3 * n + 4) + 16);
  if (!h) return cass_fail(e, CASS_ERR_NOMEM, "pinned staging");
  HIP_TRY(e, hipStreamSynchronize(e->stream));
  if (xyz)
    for (int k = 0; k < 3 * n; ++k)
      if (!std::isfinite(xyz[k])) return cass_fail(e, CASS_ERR_ARG, "non-finite coordinate");
  if (xyz) {
    std::memcpy(b->xyz_h.data() + 3 * (size_t)f, xyz, sizeof(double) * 3 * n);
    for (int a = 0; a < n; ++a) {
      h[a] = xyz[3 * a];
      h[n + a] = xyz[3 * a + 1];
      h[2 * n + a] = xyz[3 * a + 2];
    }
    double4 c = cass_host_com(e, s, xyz);
    if (com) c = make_double4(com[0], com[1], com[2], c.w);
    if (max_dcom) c.w = *max_dcom;
    std::memcpy(h + 3 * n, &c, sizeof(double4));
    b->comd_h[mol] = c;
    HIP_TRY(e, upload(e, b->x + f, h, n));
    HIP_TRY(e, upload(e, b->y + f, h + n, n));
    HIP_TRY(e, upload(e, b->z + f, h + 2 * n, n));
    HIP_TRY(e, upload(e, b->comd + mol, (const double4 *)(h + 3 * n), 1));
  }
  b->live[mol] = live;
  int32_t *hl = (int32_t *)(h + 3 * n + 4);
  *hl = live;
  HIP_TRY(e, upload(e, b->d_live + mol, hl, 1));
  HIP_TRY(e, hipStreamSynchronize(e->stream));
  return CASS_OK;
}

extern "C" int cass_box_download(cass_engine *e, int32_t box, double *xyz) {
  cass_box_state *b;
  int rc = box_of(e, box, &b);
  if (rc) return rc;
  std::vector<double> xs(b->nsites), ys(b->nsites), zs(b->nsites);
  HIP_TRY(e, hipMemcpyAsync(xs.data(), b->x, sizeof(double) * b->nsites, hipMemcpyDeviceToHost, e->stream));
  HIP_TRY(e, hipMemcpyAsync(ys.data(), b->y, sizeof(double) * b->nsites, hipMemcpyDeviceToHost, e->stream));
  HIP_TRY(e, hipMemcpyAsync(zs.data(), b->z, sizeof(double) * b->nsites, hipMemcpyDeviceToHost, e->stream));
  HIP_TRY(e, hipStreamSynchronize(e->stream));
  for (int i = 0; i < b->nsites; ++i) {
    xyz[3 * i] = xs[i];
    xyz[3 * i + 1] = ys[i];
    xyz[3 * i + 2] = zs[i];
  }
  return CASS_OK;
}

// ------------------------------------------------------------- mirrors
namespace {
struct MirrorBox {
  const double *x, *y, *z;
  const double4 *comd;
  const int *live;  // null: not packed
  int nsites, nmols;
  size_t xyz, com, flags;  // byte offsets in the packed buffer
};
}  // namespace

// One box per blockIdx.x, its entries over blockIdx.y and the lanes.  The
// copies of a batch of boxes cost a launch each, some 3 us: 64 water boxes
// took 17 ms in 3800 of them beside 1.2 ms of chain kernel; packed here and
// copied once, 3 MB take 0.1 ms.
static __global__ void __launch_bounds__(256) k_pack_mirrors(const MirrorBox *__restrict__ boxes,
                                                             char *__restrict__ out) {
  const MirrorBox &m = boxes[blockIdx.x];
  double *xyz = (double *)(out + m.xyz);
  double4 *com = (double4 *)(out + m.com);
  int *flags = (int *)(out + m.flags);
  const int step = gridDim.y * blockDim.x, t0 = blockIdx.y * blockDim.x + threadIdx.x;
  for (int i = t0; i < 3 * m.nsites; i += step) {
    const int s = i / 3, d = i - 3 * s;
    xyz[i] = d == 0 ? m.x[s] : (d == 1 ? m.y[s] : m.z[s]);
  }
  for (int i = t0; i < m.nmols; i += step) {
    com[i] = m.comd[i];
    if (m.live) flags[i] = m.live[i];
  }
}

int MirrorPull::reserve(cass_engine *e, const std::vector<int> &ids, bool live, size_t extra) {
  auto up = [](size_t n) { return (n + 255) & ~size_t(255); };
  base = up(extra);
  bytes = 0;
  parts.clear();
  with_live = live;
  for (int id : ids) {
    const cass_box_state &b = e->boxes[id];
    Part p{id, bytes, 0, 0};
    bytes += up(sizeof(double) * 3 * b.nsites);
    p.com = bytes;
    bytes += up(sizeof(double4) * b.nmols);
    p.live = bytes;
    if (live) bytes += up(sizeof(int32_t) * b.nmols);
    parts.push_back(p);
  }
  const size_t table = up(sizeof(MirrorBox) * std::max<size_t>(1, parts.size()));
  host = (char *)cass_pinned(e, base + bytes + table);
  dev = (char *)cass_io(e, bytes + table);
  return host && dev ? CASS_OK : cass_fail(e, CASS_ERR_NOMEM, "mirror staging");
}

int MirrorPull::queue(cass_engine *e) {
  if (parts.empty()) return CASS_OK;
  // the box table goes through the tail of the staging
  MirrorBox *table = (MirrorBox *)(host + base + bytes);
  int most = 1;
  for (size_t i = 0; i < parts.size(); ++i) {
    const Part &p = parts[i];
    const cass_box_state &b = e->boxes[p.box];
    table[i] = MirrorBox{b.x,   b.y,   b.z,   b.comd, with_live ? b.d_live : nullptr, b.nsites,
                         b.nmols, p.xyz, p.com, p.live};
    most = std::max(most, 3 * b.nsites);
  }
  HIP_TRY(e, hipMemcpyAsync(dev + bytes, table, sizeof(MirrorBox) * parts.size(), hipMemcpyHostToDevice, e->stream));
  const unsigned ny = (unsigned)std::min(64, (most + 1023) / 1024);
  hipLaunchKernelGGL(k_pack_mirrors, dim3((unsigned)parts.size(), ny), dim3(256), 0, e->stream,
                     (const MirrorBox *)(dev + bytes), dev);
  HIP_TRY(e, hipGetLastError());
  if (bytes) HIP_TRY(e, hipMemcpyAsync(host + base, dev, bytes, hipMemcpyDeviceToHost, e->stream));
  return CASS_OK;
}

void MirrorPull::end(cass_engine *e) {
  for (const Part &p : parts) {
    cass_box_state &b = e->boxes[p.box];
    const char *h = host + base;
    std::memcpy(b.xyz_h.data(), h + p.xyz, sizeof(double) * 3 * b.nsites);
    std::memcpy(b.comd_h.data(), h + p.com, sizeof(double4) * b.nmols);
    if (with_live) std::memcpy(b.live.data(), h + p.live, sizeof(int32_t) * b.nmols);
  }
}

// -------------------------------------------------------------- records
ChainRecords::~ChainRecords() {
  if (owner) (void)hipFreeAsync(dev, owner->stream);
}

size_t ChainRecords::add(void *dst, size_t bytes) {
  const size_t off = total;
  parts.push_back(Part{off, bytes, dst});
  total += (bytes + 255) & ~size_t(255);
  return off;
}

int ChainRecords::place(cass_engine *e, char *room) {
  if (total == 0) return CASS_OK;
  dev = room;
  if (!staged()) {
    if (hipMallocAsync((void **)&dev, total, e->stream) != hipSuccess) {
      (void)hipGetLastError();
      return cass_fail(e, CASS_ERR_NOMEM, "per-move records");
    }
    owner = e;
  }
  return CASS_OK;
}

int ChainRecords::queue(cass_engine *e) {
  if (staged()) return CASS_OK;
  for (const Part &p : parts)
    if (p.bytes) HIP_TRY(e, hipMemcpyAsync(p.dst, dev + p.off, p.bytes, hipMemcpyDeviceToHost, e->stream));
  return CASS_OK;
}

void ChainRecords::end(const char *pinned) {
  if (staged())
    for (const Part &p : parts) std::memcpy(p.dst, pinned + p.off, p.bytes);
}

// ------------------------------------------------------- trial energies
// Launches k_trials + k_finalize_trials; results (E_vdw, E_qq, overlap)
// land in dev_out[2*t], dev_ov[t] (device) -- the caller copies back.
static int trial_blocks(const cass_box_state &b) { return std::max(1, (b.nmols + kMaxBlock - 1) / kMaxBlock); }

// part / part_ov: ntrial * trial_blocks(b) partials (E_vdw, E_qq) and flags.
static int launch_trials_into(cass_engine *e, cass_box_state &b, int species, int ntrial, const double *d_txyz,
                              int cbmc, int exclude, double *part, int *part_ov, double *dev_out, int *dev_ov) {
  const int ni = e->sp_natoms[species];
  const int blk = kMaxBlock;
  const int nblk = trial_blocks(b);
  BoxDev bv = box_view(e, b);
  TopoDev tv = topo_view(e);
  PairConst<double> cd = make_pair_const<double>(b.p, e->ntypes);
  dim3 grid(nblk, ntrial);
  PairConst<float> cf = make_pair_const<float>(b.p, e->ntypes);
  auto kern = e->prec == CASS_PREC_MIXED  ? k_trials<PrecMixed>
              : e->prec == CASS_PREC_FP32 ? k_trials<PrecFP32>
                                          : k_trials<PrecFP64>;
  hipLaunchKernelGGL(kern, grid, dim3(blk), 0, e->stream, bv, tv, cd, cf, species, ni, d_txyz, exclude, cbmc, part,
                     part_ov);
  HIP_TRY(e, hipGetLastError());
  hipLaunchKernelGGL(k_finalize_trials, dim3((ntrial + 255) / 256), dim3(256), 0, e->stream, part, part_ov,
                     nblk, ntrial, dev_out, dev_ov);
  HIP_TRY(e, hipGetLastError());
  return CASS_OK;
}

static int launch_trials(cass_engine *e, cass_box_state &b, int species, int ntrial, const double *d_txyz,
                         int cbmc, int exclude, double *dev_out, int *dev_ov) {
  const size_t np = (size_t)ntrial * trial_blocks(b);
  char *s = (char *)cass_scratch(e, np * (2 * sizeof(double) + sizeof(int)) + 64);
  if (!s) return cass_fail(e, CASS_ERR_NOMEM, "scratch");
  return launch_trials_into(e, b, species, ntrial, d_txyz, cbmc, exclude, (double *)s,
                            (int *)(s + np * 2 * sizeof(double)), dev_out, dev_ov);
}

extern "C" int cass_trial_energies(cass_engine *e, int32_t box, int32_t species, int32_t ntrial,
                                   const double *trial_xyz, int32_t cbmc_flag, int32_t exclude_mol,
                                   double *nrg, int32_t *overlap) {
  cass_box_state *b;
  int rc = box_of(e, box, &b);
  if (rc) return rc;
  if (species < 0 || species >= e->nspecies || ntrial <= 0 || !trial_xyz)
    return cass_fail(e, CASS_ERR_ARG, "bad trial arguments");
  const int ni = e->sp_natoms[species];
  const size_t nxyz = (size_t)ntrial * ni * 3;
  // io buffers live in their own allocation (scratch holds partials)
  double *d_io = (double *)cass_io(e, sizeof(double) * (nxyz + 3 * (size_t)ntrial) + 16);
  if (!d_io) return cass_fail(e, CASS_ERR_NOMEM, "io buffer");
  double *d_out = d_io + nxyz;
  int *d_ov = (int *)(d_out + 2 * (size_t)ntrial);
  HIP_TRY(e, hipMemcpyAsync(d_io, trial_xyz, sizeof(double) * nxyz, hipMemcpyHostToDevice, e->stream));
  rc = launch_trials(e, *b, species, ntrial, d_io, cbmc_flag, exclude_mol, d_out, d_ov);
  if (rc) return rc;
  std::vector<double> out(2 * (size_t)ntrial);
  std::vector<int> ov(ntrial);
  HIP_TRY(e, hipMemcpyAsync(out.data(), d_out, sizeof(double) * 2 * ntrial, hipMemcpyDeviceToHost, e->stream));
  HIP_TRY(e, hipMemcpyAsync(ov.data(), d_ov, sizeof(int) * ntrial, hipMemcpyDeviceToHost, e->stream));
  HIP_TRY(e, hipStreamSynchronize(e->stream));
  for (int t = 0; t < ntrial; ++t) {
    nrg[t] = out[2 * t] + out[2 * t + 1];
    overlap[t] = ov[t];
  }
  return CASS_OK;
}

// ------------------------------------------- trial energies, no allocation
// The variant of cass_trial_energies for callers that cannot allocate: every
// device buffer it needs (the trial coordinates, the per-block partials and
// flags, the results) is carved from one file-scope device array of
// kNoAllocBytes, resolved per device at engine creation.  Calls on one GPU
// share the array, so calls that overlap on a GPU (two host threads, two
// engines on one device) race.  Nothing in it needs clearing: every partial
// is written by the trial kernel before it is read.
namespace {
constexpr size_t kNoAllocBytes = size_t(8) << 20;  // 8 MiB per GPU
constexpr int kNoAllocMaxDevices = 64;
void *g_noalloc_ptr[kNoAllocMaxDevices] = {};
}  // namespace

static __device__ __align__(256) char scratch[kNoAllocBytes];

__global__ void k_sum_pair_results(const double *out2, int ntrial, double *nrg) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < ntrial) nrg[t] = out2[2 * t] + out2[2 * t + 1];
}

// The device address of `scratch` on the current device (once per device).
static int noalloc_init(cass_engine *e) {
  if (e->device < 0 || e->device >= kNoAllocMaxDevices) return cass_fail(e, CASS_ERR_ARG, "device index");
  if (g_noalloc_ptr[e->device]) return CASS_OK;
  void *ptr = nullptr;
  const hipError_t st = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
  if (st != hipSuccess || !ptr) return cass_check_hip(e, st != hipSuccess ? st : hipErrorInvalidSymbol,
                                                      "hipGetSymbolAddress(scratch)");
  g_noalloc_ptr[e->device] = ptr;
  return CASS_OK;
}

extern "C" int cass_trial_energies_noalloc(cass_engine *e, int32_t box, int32_t species, int32_t ntrial,
                                           const double *trial_xyz, int32_t cbmc_flag, int32_t exclude_mol,
                                           double *nrg, int32_t *overlap) {
  cass_box_state *b;
  int rc = box_of(e, box, &b);
  if (rc) return rc;
  if (species < 0 || species >= e->nspecies || ntrial <= 0 || !trial_xyz || !nrg || !overlap)
    return cass_fail(e, CASS_ERR_ARG, "bad trial arguments");
  char *base = (char *)g_noalloc_ptr[e->device];
  if (!base) return cass_fail(e, CASS_ERR_STATE, "no-allocation scratch not resolved on this device");
  const size_t ni = (size_t)e->sp_natoms[species];
  const size_t np = (size_t)ntrial * trial_blocks(*b);
  auto up = [](size_t n) { return (n + 255) & ~size_t(255); };
  const size_t o_xyz = 0, n_xyz = up(sizeof(double) * ntrial * ni * 3);
  const size_t o_part = o_xyz + n_xyz, n_part = up(sizeof(double) * 2 * np);
  const size_t o_pov = o_part + n_part, n_pov = up(sizeof(int) * np);
  const size_t o_out = o_pov + n_pov, n_out = up(sizeof(double) * 2 * ntrial);
  const size_t o_ov = o_out + n_out, n_ov = up(sizeof(int) * ntrial);
  const size_t o_nrg = o_ov + n_ov, n_nrg = up(sizeof(double) * ntrial);
  if (o_nrg + n_nrg > kNoAllocBytes)
    return cass_fail(e, CASS_ERR_ARG, "trial set exceeds the 8 MiB no-allocation scratch (ntrial * (24 * natoms "
                                      "+ 20 * ceil(nmols / 256) + 20) bytes)");
  double *d_xyz = (double *)(base + o_xyz);
  double *d_out = (double *)(base + o_out);
  double *d_nrg = (double *)(base + o_nrg);
  int *d_ov = (int *)(base + o_ov);
  HIP_TRY(e, hipMemcpyAsync(d_xyz, trial_xyz, sizeof(double) * ntrial * ni * 3, hipMemcpyHostToDevice, e->stream));
  rc = launch_trials_into(e, *b, species, ntrial, d_xyz, cbmc_flag, exclude_mol, (double *)(base + o_part),
                          (int *)(base + o_pov), d_out, d_ov);
  if (rc) return rc;
  hipLaunchKernelGGL(k_sum_pair_results, dim3((ntrial + 255) / 256), dim3(256), 0, e->stream, d_out, ntrial, d_nrg);
  HIP_TRY(e, hipGetLastError());
  HIP_TRY(e, hipMemcpyAsync(nrg, d_nrg, sizeof(double) * ntrial, hipMemcpyDeviceToHost, e->stream));
  HIP_TRY(e, hipMemcpyAsync(overlap, d_ov, sizeof(int32_t) * ntrial, hipMemcpyDeviceToHost, e->stream));
  HIP_TRY(e, hipStreamSynchronize(e->stream));
  return CASS_OK;
}

// Energies of up to two placements of molecule `mol` in one launch (used by
// cass_mol_inter_energy and by the NVT chain for old + new positions).
int cass_mol_pair_trials(cass_engine *e, int32_t box, int32_t mol, int32_t cbmc, int32_t ntrial,
                         const double *xyz2, double *ev, double *eq, int32_t *ov) {
  cass_box_state *b;
  int rc = box_of(e, box, &b);
  if (rc) return rc;
  const int s = b->mol_species[mol], n = e->sp_natoms[s];
  const size_t nx = (size_t)ntrial * n * 3;
  char *h = (char *)cass_pinned(e, sizeof(double) * (nx + 3 * ntrial) + 64);
  double *d_io = (double *)cass_io(e, sizeof(double) * (nx + 3 * ntrial) + 64);
  if (!h || !d_io) return cass_fail(e, CASS_ERR_NOMEM, "staging");
  HIP_TRY(e, hipStreamSynchronize(e->stream));
  std::memcpy(h, xyz2, sizeof(double) * nx);
  HIP_TRY(e, hipMemcpyAsync(d_io, h, sizeof(double) * nx, hipMemcpyHostToDevice, e->stream));
  double *d_out = d_io + nx;
  int *d_ov = (int *)(d_out + 2 * ntrial);
  rc = launch_trials(e, *b, s, ntrial, d_io, cbmc, mol, d_out, d_ov);
  if (rc) return rc;
  double *ho = (double *)(h + sizeof(double) * nx);
  HIP_TRY(e, hipMemcpyAsync(ho, d_out, sizeof(double) * 2 * ntrial + sizeof(int) * ntrial,
                            hipMemcpyDeviceToHost, e->stream));
  HIP_TRY(e, hipStreamSynchronize(e->stream));
  const int *hov = (const int *)(ho + 2 * ntrial);
  for (int t = 0; t < ntrial; ++t) {
    ev[t] = ho[2 * t];
    eq[t] = ho[2 * t + 1];
    ov[t] = hov[t];
  }
  return CASS_OK;
}

const double *cass_box_xyz(cass_engine *e, int32_t box, int32_t mol) {
  cass_box_state &b = e->boxes[box];
  return b.xyz_h.data() + 3 * (size_t)b.mol_first[mol];
}

extern "C" int cass_mol_inter_energy(cass_engine *e, int32_t box, int32_t mol, int32_t cbmc_flag,
                                     const double *xyz, const double *com, const double *max_dcom,
                                     double *e_vdw, double *e_qq, int32_t *overlap) {
  cass_box_state *b;
  int rc = box_of(e, box, &b);
  if (rc) return rc;
  if (mol < 0 || mol >= b->nmols) return cass_fail(e, CASS_ERR_ARG, "bad molecule index");
  (void)com;
  (void)max_dcom;
  const double *src = xyz ? xyz : cass_box_xyz(e, box, mol);
  return cass_mol_pair_trials(e, box, mol, cbmc_flag, 1, src, e_vdw, e_qq, overlap);
}

// ----------------------------------------------------------- total energy
int cass_intra_host(const cass_engine *e, const cass_params &p, int s, int cbmc, const double *xyz,
                    double *ev, double *eq, double *eqi);  // host.cpp

// Intramolecular terms of Compute_System_Total_Energy on the host (n_m^2
// pairs per molecule), with the angle and dihedral energies of species that
// have a growth description, summed per molecule in the reference's order
// (energy_routines.f90:2722-2745); false: an intramolecular overlap.
static bool total_intra(const cass_engine *e, const cass_box_state *b, cass_energy *out) {
  const std::vector<double> &xyz = b->xyz_h;
  for (int s = 0; s < e->nspecies; ++s) {
    double vi = 0, vq = 0, vqi = 0, va = 0, vd = 0;
    for (int m = 0; m < b->nmols; ++m) {
      if (b->mol_species[m] != s || !b->live[m]) continue;
      double a, q, qi, ang, dih;
      const double *mx = xyz.data() + 3 * b->mol_first[m];
      cass_cbmc_bonded_host(e, s, mx, &ang, &dih);
      if (cass_intra_host(e, b->p, s, 0, mx, &a, &q, &qi)) return false;
      vi = vi + 0.0 + ang + dih + 0.0 + q + a;
      va = va + ang;
      vd = vd + dih;
      vq = vq + q;
      vqi = vqi + qi;
      out->intra_vdw += a;
    }
    out->intra += vi;
    out->angle += va;
    out->dihedral += vd;
    out->intra_q += vq;
    out->inter_q += vqi;
  }
  return true;
}

// The intermolecular pair partials (E_vdw, E_qq per partial, in order) and
// their overlap flags into out; false: an overlap.
static bool total_pair_sums(const double *hp, const int *ho, size_t np, cass_energy *out) {
  bool ov = false;
  double sum[2] = {0.0, 0.0}, low[2] = {0.0, 0.0};
  for (size_t i = 0; i < np; ++i) {
    for (int k = 0; k < 2; ++k) {
      // each addition's rounding error is kept (Knuth's two-sum)
      const double v = hp[2 * i + k], t = sum[k] + v, w = t - sum[k];
      if (std::isfinite(t)) low[k] += (sum[k] - (t - w)) + (v - w);
      sum[k] = t;
    }
    if (ho[i]) ov = true;
  }
  out->inter_vdw += sum[0] + low[0];
  out->inter_q += sum[1] + low[1];
  return !ov;
}

// The reciprocal energy (already in out->reciprocal), the self energy and
// the tail correction, then the totals.
static int total_finish(cass_engine *e, int32_t box, const cass_box_state *b, cass_energy *out) {
  out->inter = out->inter_q + out->inter_vdw;
  const cass_params &p = b->p;
  int rc;
  if (p.charge_style != CASS_Q_NONE) {
    if (p.charge_style == CASS_Q_EWALD) out->inter += out->reciprocal;
    double qq = 0.0;
    for (int s2 = 0; s2 < e->nspecies; ++s2)
      for (int m = 0; m < b->nmols; ++m) {
        if (b->mol_species[m] != s2 || !b->live[m]) continue;
        for (int a = 0; a < e->sp_natoms[s2]; ++a) {
          const double q = e->atom_charge[e->sp_atom_off[s2] + a];
          qq = qq + q * q;
        }
      }
    if (p.charge_style == CASS_Q_EWALD) out->self = -qq * kChargeFactor * p.alpha_ewald / kRootPi;
    else if (p.charge_style == CASS_Q_DSF)
      out->self = -(qq * (p.alpha_dsf / kRootPi + p.dsf_factor1 / 2.0)) * kChargeFactor;
    out->inter += out->self;
  }
  if (p.vdw_sum_style == CASS_SUM_CUT_TAIL) {
    std::vector<double> nb(e->ntypes, 0.0);
    for (int m = 0; m < b->nmols; ++m) {
      if (!b->live[m]) continue;
      const int s2 = b->mol_species[m];
      for (int a = 0; a < e->sp_natoms[s2]; ++a) {
        const int t = e->atom_type[e->sp_atom_off[s2] + a];
        if (t >= 0) nb[t] += 1.0;
      }
    }
    double lrc;
    if ((rc = cass_lrc(e, box, nb.data(), &lrc))) return rc;
    out->lrc = lrc;
    out->inter += lrc;
  }
  out->total = out->intra + out->inter;
  return CASS_OK;
}

extern "C" int cass_total_energy(cass_engine *e, int32_t box, int32_t intra_flag, cass_energy *out,
                                 int32_t *overlap) {
  cass_box_state *b;
  int rc = box_of(e, box, &b);
  if (rc) return rc;
  std::memset(out, 0, sizeof(*out));
  *overlap = 0;
  if (intra_flag && !total_intra(e, b, out)) {
    *overlap = 1;
    return CASS_OK;
  }
  // intermolecular pairs on the device
  const size_t np = (size_t)std::max(1, b->nmols);
  char *s = (char *)cass_scratch(e, np * (2 * sizeof(double) + sizeof(int)) + 256);
  if (!s) return cass_fail(e, CASS_ERR_NOMEM, "scratch");
  double *part = (double *)s;
  int *part_ov = (int *)(s + np * 2 * sizeof(double));
  if (b->nmols > 0) {
    BoxDev bv = box_view(e, *b);
    TopoDev tv = topo_view(e);
    PairConst<double> cd = make_pair_const<double>(b->p, e->ntypes);
    PairConst<float> cf = make_pair_const<float>(b->p, e->ntypes);
    auto kern = e->prec == CASS_PREC_MIXED  ? k_total_pairs<PrecMixed>
                : e->prec == CASS_PREC_FP32 ? k_total_pairs<PrecFP32>
                                            : k_total_pairs<PrecFP64>;
    hipLaunchKernelGGL(kern, dim3((b->nmols + kPairMols - 1) / kPairMols), dim3(64 * kPairMols), 0, e->stream, bv, tv,
                       cd, cf, part, part_ov);
    HIP_TRY(e, hipGetLastError());
    std::vector<double> hp(2 * np);
    std::vector<int> ho(np);
    HIP_TRY(e, hipMemcpyAsync(hp.data(), part, sizeof(double) * 2 * np, hipMemcpyDeviceToHost, e->stream));
    HIP_TRY(e, hipMemcpyAsync(ho.data(), part_ov, sizeof(int) * np, hipMemcpyDeviceToHost, e->stream));
    HIP_TRY(e, hipStreamSynchronize(e->stream));
    if (!total_pair_sums(hp.data(), ho.data(), np, out)) {
      *overlap = 1;
      return CASS_OK;
    }
  }
  if (b->p.charge_style == CASS_Q_EWALD) {
    if (!b->ewald_ready) {
      int32_t nv;
      if ((rc = cass_ewald_setup(e, box, &nv))) return rc;
    }
    double er;
    if ((rc = cass_ewald_full(e, box, &er))) return rc;
    out->reciprocal = er;
  }
  return total_finish(e, box, b, out);
}

// Compute_System_Total_Energy for several boxes in one set of launches
// (move_vol_swap.f90:322-383 recomputes both boxes of a GEMC volume swap;
// batches of volume moves recompute many): every box's pair partials in
// one k_total_pairs_multi grid, every Ewald box's structure factors in one
// k_ewald_mol_multi and one k_ewald_box_multi grid, the per-box k sums in
// one k_sum_multi; the host reductions and terms are those of
// cass_total_energy, so each box's result equals its own call bit for bit.
extern "C" int cass_total_energy_batch(cass_engine *e, int32_t nboxes, const int32_t *boxes, int32_t intra_flag,
                                       cass_energy *out, int32_t *overlap) {
  if (!e || nboxes < 0 || (nboxes > 0 && (!boxes || !out || !overlap))) return CASS_ERR_ARG;
  std::vector<cass_box_state *> bs(nboxes);
  for (int i = 0; i < nboxes; ++i) {
    int rc = box_of(e, boxes[i], &bs[i]);
    if (rc) return rc;
    for (int k = 0; k < i; ++k)
      if (boxes[k] == boxes[i]) return cass_fail(e, CASS_ERR_ARG, "a box appears twice in the batch");
  }
  int rc;
  for (int i = 0; i < nboxes; ++i)
    if (bs[i]->p.charge_style == CASS_Q_EWALD && !bs[i]->ewald_ready) {
      int32_t nv;
      if ((rc = cass_ewald_setup(e, boxes[i], &nv))) return rc;
    }
  const int blk = kMaxBlock;
  std::vector<RecomputeBox> rb(nboxes);
  std::vector<int2> items, kitems_box, kitems_mol, kitems_direct;
  int64_t np = 0, nk = 0;
  std::vector<char> direct;
  int kmols = 0;  // molecules of the Ewald boxes
  for (int i = 0; i < nboxes; ++i)
    if (bs[i]->p.charge_style == CASS_Q_EWALD) kmols += bs[i]->nmols;
  for (int i = 0; i < nboxes; ++i) {
    const cass_box_state &b = *bs[i];
    RecomputeBox &r = rb[i];
    r.b = box_view(e, b);
    r.cd = make_pair_const<double>(b.p, e->ntypes);
    r.cf = make_pair_const<float>(b.p, e->ntypes);
    r.part_off = np;
    for (int m = 0; m < b.nmols; m += kPairMols) items.push_back(make_int2(i, m));
    np += std::max(1, b.nmols);
    const bool ewald = b.p.charge_style == CASS_Q_EWALD;
    r.ew = ewald ? ewald_view(b, row_k0_of(b)) : EwaldDev{};
    r.kblk = ewald ? box_blocks(b.nvecs, b.nmols) : 0;
    r.kparts = ewald ? ewald_parts(b, kmols) : 1;
    r.kdirect = std::max(1, (b.nvecs + blk - 1) / blk);
    r.kpart_off = nk;
    if (ewald) {
      // which species take which way first: tests per molecule took 15 us of
      // a call of 24 boxes of 512
      bool any = false, all = true;
      direct.resize(e->nspecies);
      for (int sp = 0; sp < e->nspecies; ++sp) {
        direct[sp] = ewald_direct(r.ew, b.nmols, e->sp_natoms[sp]);
        any = any || direct[sp];
        all = all && direct[sp];
      }
      auto items_of = [&](std::vector<int2> &to, int parts, bool way, bool every) {
        for (int m = 0; m < b.nmols; ++m)
          if (every || direct[b.mol_species[m]] == way)
            for (int k = 0; k < parts; ++k) to.push_back(make_int2(i, m * parts + k));
      };
      if (b.nvecs > 0 && !all) items_of(kitems_mol, r.kparts, false, !any);
      if (b.nvecs > 0 && any) items_of(kitems_direct, r.kdirect, true, all);
      for (int kb = 0; kb < r.kblk; ++kb) kitems_box.push_back(make_int2(i, kb));
      nk += r.kblk;
    }
  }
  // device layout: box views, items, pair partials, k partials, k sums
  size_t off = 0;
  auto take = [&](size_t bytes) {
    const size_t o = off;
    off = (off + bytes + 255) & ~(size_t)255;
    return o;
  };
  const size_t o_rb = take(sizeof(RecomputeBox) * std::max(1, nboxes)),
               o_it = take(sizeof(int2) * std::max<size_t>(1, items.size())),
               o_km = take(sizeof(int2) * std::max<size_t>(1, kitems_mol.size())),
               o_kd = take(sizeof(int2) * std::max<size_t>(1, kitems_direct.size())),
               o_kb = take(sizeof(int2) * std::max<size_t>(1, kitems_box.size())),
               o_part = take(2 * sizeof(double) * std::max<int64_t>(1, np)),
               o_pov = take(sizeof(int) * std::max<int64_t>(1, np)),
               o_kp = take(sizeof(double) * std::max<int64_t>(1, nk)),
               o_ks = take(sizeof(double) * std::max(1, nboxes));
  char *s = (char *)cass_scratch(e, off);
  if (!s) return cass_fail(e, CASS_ERR_NOMEM, "scratch");
  HIP_TRY(e, hipMemcpyAsync(s + o_rb, rb.data(), sizeof(RecomputeBox) * nboxes, hipMemcpyHostToDevice, e->stream));
  if (!items.empty())
    HIP_TRY(e, hipMemcpyAsync(s + o_it, items.data(), sizeof(int2) * items.size(), hipMemcpyHostToDevice, e->stream));
  if (!kitems_mol.empty())
    HIP_TRY(e, hipMemcpyAsync(s + o_km, kitems_mol.data(), sizeof(int2) * kitems_mol.size(), hipMemcpyHostToDevice,
                              e->stream));
  if (!kitems_direct.empty())
    HIP_TRY(e, hipMemcpyAsync(s + o_kd, kitems_direct.data(), sizeof(int2) * kitems_direct.size(),
                              hipMemcpyHostToDevice, e->stream));
  if (!kitems_box.empty())
    HIP_TRY(e, hipMemcpyAsync(s + o_kb, kitems_box.data(), sizeof(int2) * kitems_box.size(), hipMemcpyHostToDevice,
                              e->stream));
  const RecomputeBox *d_rb = (const RecomputeBox *)(s + o_rb);
  double *d_part = (double *)(s + o_part), *d_kp = (double *)(s + o_kp), *d_ks = (double *)(s + o_ks);
  int *d_pov = (int *)(s + o_pov);
  const TopoDev tv = topo_view(e);
  HIP_TRY(e, hipEventRecord(e->ev0, e->stream));
  if (!items.empty()) {
    auto kern = e->prec == CASS_PREC_MIXED  ? k_total_pairs_multi<PrecMixed>
                : e->prec == CASS_PREC_FP32 ? k_total_pairs_multi<PrecFP32>
                                            : k_total_pairs_multi<PrecFP64>;
    hipLaunchKernelGGL(kern, dim3((unsigned)items.size()), dim3(64 * kPairMols), 0, e->stream, d_rb, tv,
                       (const int2 *)(s + o_it), d_part, d_pov);
    HIP_TRY(e, hipGetLastError());
  }
  if (!kitems_mol.empty()) {
    hipLaunchKernelGGL(k_ewald_mol_multi, dim3((unsigned)kitems_mol.size()), dim3(blk), 0, e->stream, d_rb, tv,
                       (const int2 *)(s + o_km));
    HIP_TRY(e, hipGetLastError());
  }
  if (!kitems_direct.empty()) {
    hipLaunchKernelGGL(k_ewald_direct_multi, dim3((unsigned)kitems_direct.size()), dim3(blk), 0, e->stream, d_rb, tv,
                       (const int2 *)(s + o_kd));
    HIP_TRY(e, hipGetLastError());
  }
  if (!kitems_box.empty()) {
    hipLaunchKernelGGL(k_ewald_box_multi, dim3((unsigned)kitems_box.size()), dim3(blk), 0, e->stream, d_rb,
                       (const int2 *)(s + o_kb), d_kp);
    HIP_TRY(e, hipGetLastError());
    hipLaunchKernelGGL(k_sum_multi, dim3(nboxes), dim3(256), 0, e->stream, d_rb, d_kp, d_ks);
    HIP_TRY(e, hipGetLastError());
  }
  HIP_TRY(e, hipEventRecord(e->ev1, e->stream));
  std::vector<double> hp(2 * std::max<int64_t>(1, np)), hks(std::max(1, nboxes));
  std::vector<int> ho(std::max<int64_t>(1, np));
  HIP_TRY(e, hipMemcpyAsync(hp.data(), d_part, sizeof(double) * 2 * np, hipMemcpyDeviceToHost, e->stream));
  HIP_TRY(e, hipMemcpyAsync(ho.data(), d_pov, sizeof(int) * np, hipMemcpyDeviceToHost, e->stream));
  if (!kitems_box.empty())
    HIP_TRY(e, hipMemcpyAsync(hks.data(), d_ks, sizeof(double) * nboxes, hipMemcpyDeviceToHost, e->stream));
  HIP_TRY(e, hipStreamSynchronize(e->stream));
  float ms = 0.0f;
  if (hipEventElapsedTime(&ms, e->ev0, e->ev1) == hipSuccess) e->last_kernel_ms = ms;
  for (int i = 0; i < nboxes; ++i) {
    cass_box_state *b = bs[i];
    cass_energy *o = out + i;
    std::memset(o, 0, sizeof(*o));
    overlap[i] = 0;
    // the reciprocal sums are refreshed whatever the rest finds
    if (b->p.charge_style == CASS_Q_EWALD) {
      b->e_recip = hks[i] * kChargeFactor;
      b->staged_mol = -1;
    }
    if (intra_flag && !total_intra(e, b, o)) {
      overlap[i] = 1;
      continue;
    }
    if (b->nmols > 0 &&
        !total_pair_sums(hp.data() + 2 * rb[i].part_off, ho.data() + rb[i].part_off, (size_t)b->nmols, o)) {
      overlap[i] = 1;
      continue;
    }
    if (b->p.charge_style == CASS_Q_EWALD) o->reciprocal = b->e_recip;
    if ((rc = total_finish(e, boxes[i], b, o))) return rc;
  }
  return CASS_OK;
}

// ------------------------------------------------------------------ Ewald
extern "C" int cass_ewald_setup(cass_engine *e, int32_t box, int32_t *nvecs) {
  cass_box_state *b;
  int rc = box_of(e, box, &b);
  if (rc) return rc;
  const cass_params &p = b->p;
  if (p.charge_style != CASS_Q_EWALD) return cass_fail(e, CASS_ERR_STATE, "box is not Ewald");
  // Ewald_Reciprocal_Lattice_Vector_Setup (energy_routines.f90:2170-2323)
  const double cv = 1.0 / (4.0 * p.alpha_ewald * p.alpha_ewald);
  const double hc2 = p.h_ewald_cut * p.h_ewald_cut;
  std::vector<double> hx, hy, hz, cn;
  std::vector<int32_t> kn;
  auto add = [&](int nx, int ny, int nz, double a, double bb, double c) {
    const double h2 = a * a + bb * bb + c * c;
    if (h2 < hc2) {
      hx.push_back(a);
      hy.push_back(bb);
      hz.push_back(c);
      cn.push_back((nx == 0 ? kTwoPi : 2.0 * kTwoPi) / p.volume * std::exp(-h2 * cv) / h2);
      kn.push_back(nx);
      kn.push_back(ny);
      kn.push_back(nz);
    }
  };
  if (p.box_shape != CASS_BOX_CUBIC) {
    const double *Li = p.length_inv;
    for (int nz = -20; nz <= 20; ++nz)
      for (int ny = -20; ny <= 20; ++ny)
        for (int nx = 0; nx <= 20; ++nx) {
          if (nx == 0 && ny == 0 && nz == 0) continue;
          const double X = nx, Y = ny, Z = nz;
          add(nx, ny, nz, kTwoPi * (Li[0] * X + Li[1] * Y + Li[2] * Z),
              kTwoPi * (Li[3] * X + Li[4] * Y + Li[5] * Z), kTwoPi * (Li[6] * X + Li[7] * Y + Li[8] * Z));
        }
  } else {
    const int kz = (int)(p.h_ewald_cut * p.basis_length[2] / kTwoPi) + 1;
    const int ky = (int)(p.h_ewald_cut * p.basis_length[1] / kTwoPi) + 1;
    const int kx = (int)(p.h_ewald_cut * p.basis_length[0] / kTwoPi) + 1;
    int count = 1;
    for (int nz = -kz; nz <= kz; ++nz)
      for (int ny = -ky; ny <= ky; ++ny)
        for (int nx = 0; nx <= kx; ++nx) {
          if (count > 100000) return cass_fail(e, CASS_ERR_KVEC, "Total number of k vectors exceeded");
          if (nx == 0 && ny == 0 && nz == 0) continue;
          const size_t before = hx.size();
          add(nx, ny, nz, kTwoPi * (double)nx / p.basis_length[0], kTwoPi * (double)ny / p.basis_length[1],
              kTwoPi * (double)nz / p.basis_length[2]);
          count += (int)(hx.size() - before);
        }
  }
  const int K = (int)hx.size();
  if (K > 100000) return cass_fail(e, CASS_ERR_KVEC, "Total number of k vectors exceeded");
  // Traversal of the k set for the phase recurrences of the Widom kernels:
  // at fixed (nz, nx), runs of consecutive ny that start next to ny = 0 and
  // walk away from it (ny >= 0 upwards, ny < 0 downwards); rows ordered by
  // nz, then nx.  kperm maps a traversal position to its k index.
  std::vector<int4> rows;
  std::vector<int32_t> k0, kperm;
  {
    std::vector<int> ord(K);
    for (int k = 0; k < K; ++k) ord[k] = k;
    std::sort(ord.begin(), ord.end(), [&](int a, int c) {
      const int *na = &kn[3 * a], *nc = &kn[3 * c];
      if (na[2] != nc[2]) return na[2] < nc[2];
      if (na[0] != nc[0]) return na[0] < nc[0];
      return na[1] < nc[1];
    });
    size_t g = 0;
    while (g < ord.size()) {
      size_t h = g;
      const int nz = kn[3 * ord[g] + 2], nx = kn[3 * ord[g]];
      while (h < ord.size() && kn[3 * ord[h] + 2] == nz && kn[3 * ord[h]] == nx) ++h;
      // [g, h): one (nz, nx) set in increasing ny; split at ny = 0
      size_t mid = g;
      while (mid < h && kn[3 * ord[mid] + 1] < 0) ++mid;
      for (int dir = 1; dir >= -1; dir -= 2) {
        std::vector<int> part;
        if (dir > 0)
          for (size_t i = mid; i < h; ++i) part.push_back(ord[i]);
        else
          for (size_t i = mid; i > g; --i) part.push_back(ord[i - 1]);
        for (size_t i = 0; i < part.size(); ++i) {
          const int ny = kn[3 * part[i] + 1];
          if (i > 0 && ny == kn[3 * part[i - 1] + 1] + dir) {
            rows.back().w += dir;
          } else {
            rows.push_back(make_int4(nx, nz, ny, dir));
            k0.push_back((int32_t)kperm.size());
          }
          kperm.push_back(part[i]);
        }
      }
      g = h;
    }
  }
  // the segments of consecutive vectors along nx, in k order
  std::vector<int4> tables = rows;
  int kmax[3] = {0, 0, 0};
  for (int k = 0; k < K; ++k) {
    const int *c = &kn[3 * k];
    for (int d = 0; d < 3; ++d) kmax[d] = std::max(kmax[d], std::abs(c[d]));
    const bool follows = k > 0 && c[0] == c[-3] + 1 && c[1] == c[-2] && c[2] == c[-1];
    if (follows && (tables.back().x >> 20) < kKSeg)
      tables.back().x += 1 << 20;
    else
      tables.push_back(make_int4(k | 1 << 20, c[0], c[1], c[2]));
  }
  const size_t nsegs = tables.size() - rows.size();
  // (re)allocate the k-space arrays of this box
  void *old[] = {b->hx, b->hy, b->hz, b->cn, b->cs, b->sn, b->cmol, b->smol, b->cs_new, b->sn_new,
                 b->cm_new, b->sm_new, b->rows};
  HIP_TRY(e, hipStreamSynchronize(e->stream));
  for (void *q : old)
    if (q) (void)hipFree(q);
  HIP_TRY(e, dalloc(&b->hx, K));
  HIP_TRY(e, dalloc(&b->hy, K));
  HIP_TRY(e, dalloc(&b->hz, K));
  HIP_TRY(e, dalloc(&b->cn, K));
  HIP_TRY(e, dalloc(&b->cs, K));
  HIP_TRY(e, dalloc(&b->sn, K));
  HIP_TRY(e, dalloc(&b->cs_new, K));
  HIP_TRY(e, dalloc(&b->sn_new, K));
  HIP_TRY(e, dalloc(&b->cm_new, K));
  HIP_TRY(e, dalloc(&b->sm_new, K));
  HIP_TRY(e, dalloc(&b->cmol, (size_t)K * b->cap_mols));
  HIP_TRY(e, dalloc(&b->smol, (size_t)K * b->cap_mols));
  // rows, segments, the rows' first positions and the k permutation share one
  // allocation and one copy
  const size_t head = tables.size();
  tables.resize(head + (k0.size() + kperm.size() + 3) / 4 + 1);
  std::memcpy((void *)(tables.data() + head), k0.data(), sizeof(int32_t) * k0.size());
  std::memcpy((int32_t *)(tables.data() + head) + k0.size(), kperm.data(), sizeof(int32_t) * kperm.size());
  HIP_TRY(e, dalloc(&b->rows, tables.size()));
  HIP_TRY(e, upload(e, b->hx, hx.data(), K));
  HIP_TRY(e, upload(e, b->hy, hy.data(), K));
  HIP_TRY(e, upload(e, b->hz, hz.data(), K));
  HIP_TRY(e, upload(e, b->cn, cn.data(), K));
  HIP_TRY(e, upload(e, b->rows, tables.data(), tables.size()));
  HIP_TRY(e, hipMemsetAsync(b->cs, 0, sizeof(double) * std::max(K, 1), e->stream));
  HIP_TRY(e, hipMemsetAsync(b->sn, 0, sizeof(double) * std::max(K, 1), e->stream));
  HIP_TRY(e, hipStreamSynchronize(e->stream));
  b->nvecs = K;
  b->nrows = (int)rows.size();
  b->nsegs = (int)nsegs;
  std::copy(kmax, kmax + 3, b->kmax);
  b->hx_h = hx;
  b->hy_h = hy;
  b->hz_h = hz;
  b->cn_h = cn;
  b->kn_h = kn;
  b->rows_h = rows;
  b->ewald_ready = true;
  b->staged_mol = -1;
  *nvecs = K;
  return CASS_OK;
}


extern "C" int cass_ewald_full(cass_engine *e, int32_t box, double *e_recip) {
  cass_box_state *b;
  int rc = box_of(e, box, &b);
  if (rc) return rc;
  if (!b->ewald_ready) return cass_fail(e, CASS_ERR_STATE, "call cass_ewald_setup first");
  const int K = b->nvecs;
  BoxDev bv = box_view(e, *b);
  TopoDev tv = topo_view(e);
  EwaldDev ew = ewald_view(*b, row_k0_of(*b));
  if (b->nmols > 0 && K > 0) {
    bool tabled, direct;
    ewald_ways(e, *b, ew, tabled, direct);
    if (tabled)
      hipLaunchKernelGGL(k_ewald_mol, dim3(b->nmols, ewald_parts(*b, b->nmols)), dim3(kMaxBlock), 0, e->stream, bv,
                         tv, ew);
    if (direct)
      hipLaunchKernelGGL(k_ewald_direct, dim3((K + kMaxBlock - 1) / kMaxBlock, b->nmols), dim3(kMaxBlock), 0,
                         e->stream, bv, tv, ew);
    HIP_TRY(e, hipGetLastError());
  }
  const int nb = box_blocks(K, b->nmols);
  double *part = (double *)cass_scratch(e, sizeof(double) * (nb + 1));
  if (!part) return cass_fail(e, CASS_ERR_NOMEM, "scratch");
  hipLaunchKernelGGL(k_ewald_box, dim3(nb), dim3(kMaxBlock), 0, e->stream, bv, ew, part);
  HIP_TRY(e, hipGetLastError());
  hipLaunchKernelGGL(k_sum, dim3(1), dim3(256), 0, e->stream, part, (size_t)nb, 1, 0, part + nb);
  HIP_TRY(e, hipGetLastError());
  double E;
  HIP_TRY(e, hipMemcpyAsync(&E, part + nb, sizeof(double), hipMemcpyDeviceToHost, e->stream));
  HIP_TRY(e, hipStreamSynchronize(e->stream));
  b->e_recip = E * kChargeFactor;
  b->staged_mol = -1;
  *e_recip = b->e_recip;
  return CASS_OK;
}

extern "C" int cass_ewald_move(cass_engine *e, int32_t box, int32_t mol, int32_t move_flag, const double *xyz,
                               double *e_recip_total, double *de_recip) {
  cass_box_state *b;
  int rc = box_of(e, box, &b);
  if (rc) return rc;
  if (!b->ewald_ready) return cass_fail(e, CASS_ERR_STATE, "call cass_ewald_setup first");
  if (mol < 0 || mol >= b->cap_mols) return cass_fail(e, CASS_ERR_ARG, "bad molecule index");
  if (move_flag < CASS_MOVE_TRANSLATION || move_flag > CASS_MOVE_DELETION) return CASS_ERR_ARG;
  if (move_flag != CASS_MOVE_DELETION && !xyz) return CASS_ERR_ARG;
  const int s = mol < b->nmols ? b->mol_species[mol] : 0;
  const int n = e->sp_natoms[s];
  const int K = b->nvecs;
  const int nb = std::max(1, (K + 255) / 256);
  char *h = (char *)cass_pinned(e, sizeof(double) * (3 * n + 4));
  if (!h) return cass_fail(e, CASS_ERR_NOMEM, "pinned staging");
  HIP_TRY(e, hipStreamSynchronize(e->stream));
  double *part = (double *)cass_scratch(e, sizeof(double) * (2 * nb + 3 * n + 8));
  if (!part) return cass_fail(e, CASS_ERR_NOMEM, "scratch");
  double *d_xyz = part + 2 * nb + 4;
  if (xyz) {
    std::memcpy(h, xyz, sizeof(double) * 3 * n);
    HIP_TRY(e, hipMemcpyAsync(d_xyz, h, sizeof(double) * 3 * n, hipMemcpyHostToDevice, e->stream));
  }
  TopoDev tv = topo_view(e);
  EwaldDev ew = ewald_view(*b, row_k0_of(*b));
  hipLaunchKernelGGL(k_ewald_move, dim3(nb), dim3(256), 0, e->stream, tv, ew, mol, s, move_flag, n, d_xyz, part);
  HIP_TRY(e, hipGetLastError());
  hipLaunchKernelGGL(k_sum, dim3(1), dim3(256), 0, e->stream, part, (size_t)nb, 2, 0, part + 2 * nb);
  hipLaunchKernelGGL(k_sum, dim3(1), dim3(256), 0, e->stream, part, (size_t)nb, 2, 1, part + 2 * nb + 1);
  HIP_TRY(e, hipGetLastError());
  double *ho = (double *)h;
  HIP_TRY(e, hipMemcpyAsync(ho, part + 2 * nb, sizeof(double) * 2, hipMemcpyDeviceToHost, e->stream));
  HIP_TRY(e, hipStreamSynchronize(e->stream));
  b->e_recip_staged = ho[0] * kChargeFactor;
  b->staged_mol = mol;
  b->staged_flag = move_flag;
  if (e_recip_total) *e_recip_total = b->e_recip_staged;
  if (de_recip) *de_recip = ho[1] * kChargeFactor;
  return CASS_OK;
}

extern "C" int cass_ewald_commit(cass_engine *e, int32_t box) {
  cass_box_state *b;
  int rc = box_of(e, box, &b);
  if (rc) return rc;
  if (b->staged_mol < 0) return cass_fail(e, CASS_ERR_STATE, "no staged Ewald move");
  EwaldDev ew = ewald_view(*b, row_k0_of(*b));
  hipLaunchKernelGGL(k_ewald_commit, dim3(std::max(1, (b->nvecs + 255) / 256)), dim3(256), 0, e->stream, ew,
                     b->staged_mol);
  HIP_TRY(e, hipGetLastError());
  b->e_recip = b->e_recip_staged;
  b->staged_mol = -1;
  return CASS_OK;
}

extern "C" int cass_ewald_revert(cass_engine *e, int32_t box) {
  cass_box_state *b;
  int rc = box_of(e, box, &b);
  if (rc) return rc;
  b->staged_mol = -1;  // the staged sums are simply dropped
  return CASS_OK;
}

extern "C" int cass_ewald_widom(cass_engine *e, int32_t box, int32_t species, int32_t ntrial,
                                const double *trial_xyz, double *e_recip) {
  cass_box_state *b;
  int rc = box_of(e, box, &b);
  if (rc) return rc;
  if (!b->ewald_ready) return cass_fail(e, CASS_ERR_STATE, "call cass_ewald_setup first");
  if (species < 0 || species >= e->nspecies || ntrial <= 0) return CASS_ERR_ARG;
  const int n = e->sp_natoms[species];
  const int K = b->nvecs;
  const int nbk = std::max(1, std::min(8, (K + 255) / 256));
  const size_t nxyz = (size_t)ntrial * n * 3;
  double *d_io = nullptr;
  HIP_TRY(e, hipMallocAsync((void **)&d_io, sizeof(double) * (nxyz + (size_t)ntrial * nbk) + 16, e->stream));
  double *part = d_io + nxyz;
  HIP_TRY(e, hipMemcpyAsync(d_io, trial_xyz, sizeof(double) * nxyz, hipMemcpyHostToDevice, e->stream));
  TopoDev tv = topo_view(e);
  EwaldDev ew = ewald_view(*b, row_k0_of(*b));
  hipLaunchKernelGGL(k_ewald_widom, dim3(nbk, ntrial), dim3(256), 0, e->stream, tv, ew, species, n, d_io, part);
  HIP_TRY(e, hipGetLastError());
  std::vector<double> hp((size_t)ntrial * nbk);
  HIP_TRY(e, hipMemcpyAsync(hp.data(), part, sizeof(double) * hp.size(), hipMemcpyDeviceToHost, e->stream));
  HIP_TRY(e, hipFreeAsync(d_io, e->stream));
  HIP_TRY(e, hipStreamSynchronize(e->stream));
  for (int t = 0; t < ntrial; ++t) {
    double s = 0.0;
    for (int k = 0; k < nbk; ++k) s += hp[(size_t)t * nbk + k];
    e_recip[t] = s * kChargeFactor;
  }
  return CASS_OK;
}

// ----------------------------------------------------------------- Widom
int cass_widom_prepare(cass_engine *e, cass_box_state &b, int species, WidomArgs &w);  // host.cpp

int cass_run_widom(cass_engine *e, int32_t box, int32_t species, int64_t n_ins, uint64_t seed, const double *place,
                   double *widom_var, double *eout, cass_widom_result *res, double *eij_max = nullptr,
                   double *rsq_min = nullptr);  // widom.hip

extern "C" int cass_widom_batch(cass_engine *e, int32_t box, int32_t species, int64_t n_ins, uint64_t seed,
                                double *widom_var, cass_widom_result *res) {
  if (!res) return CASS_ERR_ARG;
  return cass_run_widom(e, box, species, n_ins, seed, nullptr, widom_var, nullptr, res);
}

// Per-insertion body of Widom_Insert at explicit placements (test entry: the
// same kernel as cass_widom_batch).  eout[4*i] = {E_inter, E_cbmc,
// dE_recip, overlap}.
extern "C" int cass_widom_placements(cass_engine *e, int32_t box, int32_t species, int64_t n,
                                     const double *xyz, double *widom_var, double *eout,
                                     cass_widom_result *res) {
  if (!res || !xyz) return CASS_ERR_ARG;
  return cass_run_widom(e, box, species, n, 0, xyz, widom_var, eout, res);
}

// est_emax / est_atompair_rminsq of a rigid Widom batch (widom_insert.f90:
// 178-186, 325, 388, 450-476): the insertions of cass_widom_batch (xyz NULL)
// or of explicit placements, with each one's widom_var, overlap flag,
// Eij_max and, with rsq_min, closest r^2 per (species site, probe atom).
extern "C" int cass_widom_emax(cass_engine *e, int32_t box, int32_t species, int64_t n, uint64_t seed,
                               const double *xyz, double *widom_var, double *eij_max, uint8_t *overlap,
                               double *rsq_min, cass_widom_result *res) {
  if (!e || !res || !widom_var || !eij_max || !overlap || n <= 0) return CASS_ERR_ARG;
  if (box < 0 || box >= (int)e->boxes.size()) return CASS_ERR_ARG;
  std::vector<double> eout((size_t)4 * n);
  int rc = cass_run_widom(e, box, species, n, seed, xyz, widom_var, eout.data(), res, eij_max, rsq_min);
  if (rc) return rc;
  // the batch's overlap (widom_finish): a core overlap, or a CBMC-cutoff
  // energy at or above max_kBT (fragment_growth.f90:536-539)
  const double beta = e->boxes[box].p.beta;
  for (int64_t i = 0; i < n; ++i) {
    const bool ov = eout[4 * i + 3] != 0.0 || beta * eout[4 * i + 1] >= kMaxKBT;
    overlap[i] = (uint8_t)ov;
    if (ov) eij_max[i] = 0.0;
  }
  return CASS_OK;
}
