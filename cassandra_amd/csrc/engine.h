// engine.h -- internal state of libcassgpu (not part of the C ABI).
#pragma once

#include <hip/hip_runtime.h>

#include <string>
#include <vector>

#include "../../include/cass_gpu.h"

struct cass_box_state {
  cass_params p{};
  int32_t cap_mols = 0, cap_sites = 0;
  int32_t nmols = 0, nsites = 0;
  std::vector<int32_t> mol_species, mol_first, live;  // host mirrors
  std::vector<double> xyz_h;        // host mirror of the coordinates (3*nsites)
  // device: sites (SoA, FP64 master) and molecules
  double *x = nullptr, *y = nullptr, *z = nullptr;
  int32_t *site_spa = nullptr;      // species-atom index of each site
  int32_t *d_first = nullptr, *d_species = nullptr, *d_live = nullptr;
  double4 *comd = nullptr;          // (xcom, ycom, zcom, max_dcom)
  std::vector<double4> comd_h;      // host mirror of comd
  // Ewald (k order of Ewald_Reciprocal_Lattice_Vector_Setup)
  int32_t nvecs = 0;
  std::vector<double> hx_h, hy_h, hz_h, cn_h;
  std::vector<int32_t> kn_h;        // (nx, ny, nz) per k, 3 ints
  std::vector<int4> rows_h;         // k traversal rows: (nx, nz, ny0, +-count)
  double *hx = nullptr, *hy = nullptr, *hz = nullptr, *cn = nullptr;
  double *cs = nullptr, *sn = nullptr;            // box structure factor
  double *cmol = nullptr, *smol = nullptr;        // [cap_mols][nvecs]
  double *cs_new = nullptr, *sn_new = nullptr;    // staged box sums of a move
  double *cm_new = nullptr, *sm_new = nullptr;    // staged molecule sums of a move
  int4 *rows = nullptr;             // traversal rows, then the k segments, then the rows' positions and kperm
  int32_t nrows = 0, nsegs = 0;
  const int4 *segs() const { return rows + nrows; }  // runs of up to kKSeg vectors along nx: (k0 | len << 20, nx, ny, nz)
  int32_t kmax[3] = {0, 0, 0};      // largest |nx|, |ny|, |nz|
  int32_t staged_mol = -1, staged_flag = -1;
  bool ewald_ready = false;
  double e_recip = 0.0;             // last full / committed total reciprocal energy
  double e_recip_staged = 0.0;
  // tabulated CBMC pair energies (cass_set_energy_table): apt_res bins of
  // vdW per type pair, then the charge factor f2 per bin
  double *apt = nullptr;
  int32_t apt_res = 0;
  double apt_rcsq_max = 0.0;        // the largest rcut_cbmc^2 over the boxes
  double apt_step = 0.0, apt_shift = 0.0, apt_rcs = 0.0;
  // per type-pair core radii^2 of the Widom overlap pre-screen
  // (cass_widom_set_rminsq); empty: off
  std::vector<double> rminsq;
};

// Device tables of the frame for the Widom kernels (frame molecules and
// sites, per-kind pair tables, image shifts, erfc table), kept between
// batches and rebuilt when the engine generation, the box or the species
// changes.
struct WidomTables {
  uint64_t gen = ~0ull;
  int box = -1, species = -1;
  char *dev = nullptr;
  size_t cap = 0;
  size_t o_fm = 0, o_fs = 0, o_ft = 0, o_tab = 0, o_psite = 0, o_img = 0, o_qtab = 0, o_q = 0, o_rmin = 0;
  bool has_rmin = false;    // per (kind, frame site) overlap radii^2 at o_rmin
  double rmin_max2 = 0.0;   // their largest value
  size_t o_rminf = 0;       // fused path: per (probe site, frame type) radii^2
  bool has_rminf = false;
  double rminf_max2 = 0.0;
  int nmols = 0, ntab = 0;
  bool split_ok = false;  // frame within the split kernels' packing limits
  int64_t ps_stride = 0;
  double tab_inv_h = 0.0, dcom_max = 0.0;
};

// Coordinate frames of one box for the batched adjoint
// (cass_adjoint_set_frames): per frame x[nsites], y[nsites], z[nsites]
// padded to a multiple of 4 doubles, then the molecules' (COM, max_dcom);
// stride doubles per frame.  The molecule table they were stored with is
// kept to refuse a use after the box's molecules changed.
struct AdjFrames {
  int box = -1, nframes = 0, nsites = 0, nmols = 0;
  int64_t stride = 0;
  double *dev = nullptr;
  size_t cap = 0;
  std::vector<int32_t> mol_species, mol_first;
};

struct cass_engine {
  int device = 0;
  // bumped by every call that changes topology, parameters, precision or a
  // box's molecules (invalidates cached device tables)
  uint64_t gen = 0;
  WidomTables wtab;
  AdjFrames adjf;
  hipStream_t stream = nullptr;
  // a second stream (default priority) for kernels that run beside those of
  // `stream`: the reciprocal kernel of a Widom batch beside its real-space one
  hipStream_t side = nullptr;
  hipEvent_t ev_join = nullptr;
  int32_t overlap = 1;
  int32_t prec = CASS_PREC_FP64;
  std::string err;
  // topology (host copies + device)
  int32_t ntypes = 0, nspecies = 0, natoms_total = 0;
  std::vector<double> eps, sig, mie_n, mie_m;
  std::vector<int32_t> sp_natoms, sp_atom_off, sp_pair_off, sp_coul_cbmc;
  std::vector<int32_t> atom_type;
  std::vector<double> atom_charge, atom_mass, vdw_scale, q_scale;
  std::vector<int32_t> bonded;
  double *d_eps = nullptr, *d_sig = nullptr, *d_mn = nullptr, *d_mm = nullptr;
  int32_t *d_atom_type = nullptr;
  double *d_atom_charge = nullptr, *d_atom_mass = nullptr;
  int32_t *d_sp_natoms = nullptr, *d_sp_atom_off = nullptr, *d_sp_coul_cbmc = nullptr;
  std::vector<cass_box_state> boxes;
  // rigid Widom templates per species: site offsets from the COM and the
  // intramolecular energy of the template (cass_widom_set_template)
  std::vector<std::vector<double>> widom_ref;
  std::vector<double> widom_intra;
  int32_t max_boxes = 0;
  // scratch (grown on demand)
  void *scratch = nullptr;
  size_t scratch_bytes = 0;
  void *pinned = nullptr;
  size_t pinned_bytes = 0;
  size_t pinned_limit = ~(size_t)0;  // a request beyond it fails (cass_test_pinned_limit)
  void *io = nullptr;               // device input/output staging of the small calls
  hipEvent_t ev0 = nullptr, ev1 = nullptr;  // brackets the last batched kernel
  double last_kernel_ms = 0.0;
  // stage events of the last Widom batch: start, placed+sorted, real space, end
  hipEvent_t evs[4] = {nullptr, nullptr, nullptr, nullptr};
  double last_stage_ms[4] = {0.0, 0.0, 0.0, 0.0};
  size_t io_bytes = 0;
};

// host helpers shared between translation units
#define HIP_TRY(e, call)                                          \
  do {                                                            \
    hipError_t st_ = (call);                                      \
    if (st_ != hipSuccess) return cass_check_hip((e), st_, #call); \
  } while (0)

int cass_fail(cass_engine *e, int code, const std::string &msg);
int cass_check_hip(cass_engine *e, hipError_t st, const char *what);
void *cass_scratch(cass_engine *e, size_t bytes);
void *cass_pinned(cass_engine *e, size_t bytes);
void *cass_io(cass_engine *e, size_t bytes);
void cass_cbmc_release(cass_engine *e);
// Host mirrors of boxes that a chain kernel moves.  reserve(), before anything
// is launched, obtains the staging, so that a lack of memory leaves the boxes
// untouched; the first `extra` bytes of it are the caller's.  queue(), after
// the launches, packs every box's coordinates (x, y, z together), centres and,
// with live, live flags into one buffer and copies that to the staging; end(),
// after the caller has synchronised the stream, takes them into the mirrors.
struct MirrorPull {
  char *host = nullptr;  // the pinned staging
  int reserve(cass_engine *e, const std::vector<int> &ids, bool live, size_t extra);
  int queue(cass_engine *e);
  void end(cass_engine *e);

 private:
  struct Part {
    int box;
    size_t xyz, com, live;
  };
  std::vector<Part> parts;
  bool with_live = false;
  size_t base = 0, bytes = 0;  // the caller's bytes; the packed ones
  char *dev = nullptr;
};
// Per-move records of a chain batch, on their way from the device to the
// caller's arrays.  Up to kRecordStage bytes of them stand behind the batch's
// states, in its scratch and its pinned staging, and come back in their copy;
// more, from a stream allocation that is given back, are copied straight into
// the caller's arrays, so that the engine keeps no memory that grows with the
// moves of a call.  The kernels write every record of a launch (record_rest).
constexpr size_t kRecordStage = (size_t)16 << 20;
struct ChainRecords {
  ~ChainRecords();
  // one array of `bytes` for dst; returns its place for at()
  size_t add(void *dst, size_t bytes);
  size_t staged() const { return total <= kRecordStage ? total : 0; }
  // device memory: `room`, with staged() bytes of it, or its own
  int place(cass_engine *e, char *room);
  template <typename T>
  T *at(size_t off) const {
    return (T *)(dev + off);
  }
  // queues the copies where the records are not staged; end(), after the
  // synchronisation, takes those that are from `pinned`
  int queue(cass_engine *e);
  void end(const char *pinned);

 private:
  struct Part {
    size_t off, bytes;
    void *dst;
  };
  std::vector<Part> parts;
  size_t total = 0;
  char *dev = nullptr;
  cass_engine *owner = nullptr;  // of a stream allocation
};
bool cass_cbmc_bonded_host(const cass_engine *e, int s, const double *xyz, double *angle, double *dihedral);
double4 cass_host_com(const cass_engine *e, int s, const double *xyz);  // Get_COM and max_dcom of one molecule  // device copies of the CBMC growth descriptions
