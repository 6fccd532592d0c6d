/*
 * cass_gpu.h -- C ABI of the MI355X energy engine for Cassandra's Monte Carlo
 * moves (libcassgpu.so).
 *
 * Every entry point takes plain scalars and pointers, returns an int status
 * (CASS_OK = 0) and replaces one Fortran subroutine of the reference; the
 * replaced routine is cited as file:line into the reference's Src/ tree.
 * Arguments mirror the Fortran ones: int32 for default INTEGER, double for
 * REAL(DP), int32 0/1 for LOGICAL.  Indices (box, molecule, species, atom,
 * type) are 0-based here; the Fortran binding subtracts one.
 *
 * Ownership: the host owns the canonical state (coordinates, molecule
 * lists).  The engine keeps device mirrors and must be told about every
 * mutation (cass_mol_update after an accepted move or a fold,
 * cass_box_upload after a frame load or a volume change).
 *
 * Threading: one engine is driven by one host thread.  Calls are ordered on
 * the engine's HIP stream; calls that return values synchronise.
 */
#ifndef CASS_GPU_H
#define CASS_GPU_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* ---------------------------------------------------------------- status */
enum {
  CASS_OK = 0,
  CASS_ERR_ARG = 1,        /* bad argument (index out of range, bad size) */
  CASS_ERR_HIP = 2,        /* HIP runtime error */
  CASS_ERR_NOMEM = 3,      /* device allocation failed */
  CASS_ERR_KVEC = 4,       /* too many k vectors: energy_routines.f90:2268-2272 */
  CASS_ERR_CHARGE = 5,     /* net charge with Ewald/DSF: main.f90:322-328 */
  CASS_ERR_STATE = 6,      /* call out of order (e.g. Ewald not set up) */
  CASS_ERR_NODEVICE = 7,   /* no GPU visible */
  CASS_ERR_CUTOFF = 8      /* cutoff larger than half the box: input_routines.f90:466-471 */
};

/* ---------------------------------------------------------------- styles */
enum { CASS_VDW_NONE = 0, CASS_VDW_LJ = 1, CASS_VDW_MIE = 2 };
enum {
  CASS_SUM_CUT = 0, CASS_SUM_CUT_TAIL = 1, CASS_SUM_CUT_SHIFT = 2, CASS_SUM_CUT_SWITCH = 3,
  CASS_SUM_CUT_SHIFT_FORCE = 4, CASS_SUM_CHARMM = 5, CASS_SUM_MINIMUM = 6
};
enum { CASS_Q_NONE = 0, CASS_Q_EWALD = 1, CASS_Q_DSF = 2, CASS_Q_CUT = 3, CASS_Q_MINIMUM = 4 };
enum { CASS_BOX_CUBIC = 0, CASS_BOX_ORTHO = 1, CASS_BOX_CELL = 2 };
/* Update_System_Ewald_Reciprocal_Energy move flags (global_variables.f90 int_*) */
enum { CASS_MOVE_TRANSLATION = 0, CASS_MOVE_ROTATION = 1, CASS_MOVE_INTRA = 2,
       CASS_MOVE_INSERTION = 3, CASS_MOVE_DELETION = 4 };
/* arithmetic of the pair and k-space terms */
enum { CASS_PREC_FP64 = 0,     /* plain FP64 everywhere (reference parity) */
       CASS_PREC_MIXED = 1,    /* FP32 real-space q-q pair terms, FP64 LJ/Mie, FP64 sums */
       CASS_PREC_FP32 = 2 };   /* FP32 for both pair terms, FP64 sums (fastest, ~1e-5 rel) */

/* --------------------------------------------------------- box parameters
 * The box geometry and the VDW_Style / Charge_Style / Rcutoff_Low /
 * CBMC_Info settings of one box (input_routines.f90:425-812, 3784-3830,
 * 5931-6104, 6941-7104).  The "derived" block holds what the reference
 * computes from them (compute_cell_dimensions.f90, precalculate.f90:40-90,
 * input_routines.f90:711-757, 4090): cass_params_derive() fills it from the
 * raw block; a Fortran host may copy its own module variables instead. */
typedef struct cass_params {
  int32_t box_shape;        /* CASS_BOX_* */
  int32_t vdw_style;        /* CASS_VDW_* */
  int32_t vdw_sum_style;    /* CASS_SUM_* */
  int32_t charge_style;     /* CASS_Q_* */
  double cell[9];           /* box_list%length(3,3), Fortran column-major */
  double rcut_vdw, rcut_coul, rcut_cbmc, rcut_low;
  double ron_switch, roff_switch;   /* cut_switch / CHARMM on-off radii */
  double ewald_tol;                 /* Ewald accuracy */
  double alpha_dsf_in;              /* DSF damping; <= 0 selects the default */
  double temperature;               /* K */
  /* derived */
  double length_inv[9];     /* box_list%length_inv, column-major */
  double hlength[3];        /* half basis lengths */
  double basis_length[3];
  double volume;
  double rcut_vdwsq, rcut_coulsq, rcut_cbmcsq, rcut_lowsq, rcut_max;
  double ron_switch_sq, roff_switch_sq, switch_factor1, switch_factor2;
  double rcut3, rcut9;
  double alpha_ewald, h_ewald_cut;
  double alpha_dsf, dsf_factor1, dsf_factor2;
  double beta;
} cass_params;

/* ------------------------------------------------------------- topology
 * Force field and species shared by all boxes of an engine: the nonbond
 * tables vdw_param1..4_table (create_nonbond_table.f90:230-440, in internal
 * units), per-atom type/charge/mass (nonbond_list), the intramolecular
 * scaling tables (create_intra_exclusion_table.f90) and l_bonded. */
typedef struct cass_topology {
  int32_t ntypes;
  const double *eps;        /* [ntypes*ntypes] vdw_param1_table */
  const double *sig;        /* [ntypes*ntypes] vdw_param2_table */
  const double *mie_n;      /* [ntypes*ntypes] vdw_param3_table (NULL for LJ) */
  const double *mie_m;      /* [ntypes*ntypes] vdw_param4_table (NULL for LJ) */
  int32_t nspecies;
  const int32_t *species_natoms;      /* [nspecies] */
  const int32_t *species_atom_offset; /* [nspecies] into the per-atom arrays */
  const int32_t *species_pair_offset; /* [nspecies] into the natoms^2 tables */
  const int32_t *species_coul_cbmc;   /* [nspecies] L_Coul_CBMC */
  const int32_t *atom_type;           /* [sum natoms] 0-based type, -1 for none */
  const double *atom_charge;          /* [sum natoms] */
  const double *atom_mass;            /* [sum natoms] */
  const double *vdw_intra_scale;      /* [sum natoms^2] row-major (ia, ja) */
  const double *charge_intra_scale;   /* [sum natoms^2] */
  const int32_t *bonded;              /* [sum natoms^2] l_bonded */
} cass_topology;

/* Energy_Class of one box (type_definitions.f90:487-511), internal units. */
typedef struct cass_energy {
  double total, intra, inter;
  double bond, angle, dihedral, improper, intra_vdw, intra_q;
  double inter_vdw, lrc, inter_q, reciprocal, self;
} cass_energy;

typedef struct cass_engine cass_engine;

/* State of the reference's random-number generator: the five 64-bit
 * components of rranf's L'Ecuyer LFSR (random_generators.f90:51-122). */
typedef struct cass_rng { int64_t s[5]; } cass_rng;

/* ------------------------------------------------------------------ setup */
/* Fills the derived block of *p (compute_cell_dimensions.f90:50-170,
 * precalculate.f90:40-90, input_routines.f90:711-757 and 4090). */
int cass_params_derive(cass_params *p);

/* The start-up charge-neutrality check of main.f90:300-330 for one box:
 * *q_box = sum over species of (live molecules) x (species total charge);
 * returns CASS_ERR_CHARGE when |q_box| > tiny_number with Ewald or DSF sums
 * (the reference aborts there).  Host arithmetic; needs no GPU. */
int cass_net_charge(const cass_params *p, const cass_topology *topo, int32_t nmols,
                    const int32_t *mol_species, const int32_t *live, double *q_box);

/* Creates an engine on HIP device `device` for up to `max_boxes` boxes.
 * The topology is copied. */
int cass_engine_create(int32_t device, const cass_topology *topo, int32_t max_boxes,
                       cass_engine **out);
int cass_engine_destroy(cass_engine *eng);
int cass_set_precision(cass_engine *eng, int32_t prec);   /* CASS_PREC_* */
/* Kernels of one call that do not depend on each other run side by side on
 * a second stream when on (the default): the reciprocal change of a Widom
 * batch beside its real-space sums.  Off runs them one after another on the
 * engine's stream (for timing each on its own).  No reference counterpart:
 * an engine option. */
int cass_set_overlap(cass_engine *eng, int32_t on);

/* Replaces the nonbond tables (vdw_param1/2_table, [ntypes*ntypes]) and/or
 * the per-atom charges ([sum natoms]) of the topology; NULL keeps a table.
 * The Fortran host would call it after Create_Nonbond_Table
 * (create_nonbond_table.f90:10) reruns; force-field fitting calls it between
 * adjoint evaluations.  Ewald sums must be recomputed after a charge change. */
int cass_set_nonbond_params(cass_engine *eng, const double *eps, const double *sig,
                            const double *atom_charge);
const char *cass_last_error(cass_engine *eng);
/* Device time of the last batched kernel (Widom / trial-set), from HIP events
 * recorded on the engine's stream around the launch.  Instrumentation; no
 * counterpart in the reference (whose timers are the CPU clocks of
 * nvtmc_driver.f90:110-232 and widom_insert.f90:322-323). */
int cass_last_kernel_ms(cass_engine *eng, double *ms);
/* Stage times of the last cass_widom_batch / cass_widom_placements, from the
 * same events: ms[0] placement and spatial sort, ms[1] real-space pair
 * kernel, ms[2] reciprocal change and combination, ms[3] the whole batch on
 * the device.  Instrumentation; no counterpart in the reference. */
int cass_last_stage_ms(cass_engine *eng, double *ms);

/* Adds a box able to hold `max_mols` molecules; returns its id in *box. */
int cass_box_create(cass_engine *eng, const cass_params *p, int32_t max_mols, int32_t *box);

/* Replaces a box's geometry and settings, as a volume move leaves them
 * (move_volume.f90:374-426, move_vol_swap.f90:322-383: the cell scaled, then
 * Compute_Cell_Dimensions).  The reciprocal sums are stale afterwards: upload
 * the rescaled coordinates (cass_box_upload), then cass_ewald_setup
 * regenerates the k vectors for the new cell (energy_routines.f90:2170) and
 * cass_total_energy recomputes the box (:2648).  A pair table is rebuilt. */
int cass_box_set_params(cass_engine *eng, int32_t box, const cass_params *p);

/* Mirrors atom_list / molecule_list of a box: nmols molecules of
 * mol_species[m], live flag live[m], coordinates xyz[3*site] (sites of
 * molecule m follow those of m-1), COM com[3*m] and max_dcom[m]
 * (Get_COM / Compute_Max_Com_Distance, get_com.f90:45-121,220-295).  com and
 * max_dcom may be NULL: the engine then computes them as the reference does. */
int cass_box_upload(cass_engine *eng, int32_t box, int32_t nmols, const int32_t *mol_species,
                    const int32_t *live, const double *xyz, const double *com,
                    const double *max_dcom);

/* New coordinates of one molecule (accepted move, fold, insertion);
 * live sets molecule_list%live. com/max_dcom as in cass_box_upload. */
int cass_mol_update(cass_engine *eng, int32_t box, int32_t mol, int32_t live,
                    const double *xyz, const double *com, const double *max_dcom);

/* Reads back the device copy of the coordinates of a box (3*nsites). */
int cass_box_download(cass_engine *eng, int32_t box, double *xyz);

/* --------------------------------------------------------- pair energies */
/* Compute_Molecule_Nonbond_Inter_Energy (energy_routines.f90:1088-1206):
 * molecule `mol` of `box` against every other live molecule, with the COM
 * prefilter of Check_MoleculePair_Cutoff (:3027-3088), the overlap test
 * r^2 < rcut_low^2 (:1676) and the style dispatch of Compute_AtomPair_Energy
 * (:1831-2053).  If xyz is non-NULL the molecule is evaluated at those
 * coordinates (com / max_dcom as in cass_box_upload) instead of its stored
 * ones, which is how a trial position is scored before commit.  cbmc_flag
 * selects the CBMC cutoff (rcut_cbmc, L_Coul_CBMC). */
int cass_mol_inter_energy(cass_engine *eng, int32_t box, int32_t mol, int32_t cbmc_flag,
                          const double *xyz, const double *com, const double *max_dcom,
                          double *e_vdw, double *e_qq, int32_t *overlap);

/* Compute_Molecule_Nonbond_Intra_Energy (energy_routines.f90:980-1085) for a
 * molecule of `species` at xyz (natoms*3): minimum-image intramolecular vdW
 * and q-q with 1-2/1-3/1-4/1-N scaling, the periodic part of Ewald/DSF as
 * e_inter_qq, and the intra overlap test r^2 <= rcut_low^2 for non-bonded
 * pairs.  Host arithmetic (n_m^2 <= 25 pairs). */
int cass_mol_intra_energy(cass_engine *eng, int32_t box, int32_t species, int32_t cbmc_flag,
                          const double *xyz, double *e_intra_vdw, double *e_intra_qq,
                          double *e_inter_qq, int32_t *overlap);

/* Trial energies of a CBMC / Widom trial set in one launch: ntrial
 * placements of a molecule of `species` (trial_xyz[ntrial*natoms*3]) against
 * every live molecule of the box except `exclude_mol` (-1: none).  Each trial
 * is the sum Compute_Molecule_Nonbond_Inter_Energy[_Widom] returns
 * (energy_routines.f90:1088,1209) at cutoff rcut_cbmc when cbmc_flag is set
 * (fragment_growth.f90:519-526) and at the full cutoff otherwise; nrg[t] is
 * E_vdw + E_qq, overlap[t] the overlap flag.  Replaces the serial kappa loops
 * of Build_Molecule (fragment_growth.f90:383-579) and Fragment_Placement
 * (:1926-2058). */
int cass_trial_energies(cass_engine *eng, int32_t box, int32_t species, int32_t ntrial,
                        const double *trial_xyz, int32_t cbmc_flag, int32_t exclude_mol,
                        double *nrg, int32_t *overlap);

/* cass_trial_energies for callers that cannot allocate device memory (code
 * under HIP graph capture, tight serving loops, harnesses that forbid
 * hipMalloc).  No counterpart in the reference.  Same arguments and results
 * as cass_trial_energies, bit for bit; it calls no hipMalloc / hipFree.
 * Its device buffers come from one 8 MiB array per GPU, held until the
 * process ends: a call needs ntrial * (24 natoms + 20 ceil(nmols / 256) + 20)
 * bytes (plus alignment) and sets larger than that are refused with
 * CASS_ERR_ARG.  Calls on one GPU share the array: calls that overlap on a
 * GPU (two threads, two engines on one device) race. */
int cass_trial_energies_noalloc(cass_engine *eng, int32_t box, int32_t species, int32_t ntrial,
                                const double *trial_xyz, int32_t cbmc_flag, int32_t exclude_mol,
                                double *nrg, int32_t *overlap);

/* Tabulated CBMC pair energies, the `energy_table` keyword: replaces
 * Create_Atompair_Nrg_table (atompair_nrg_table_routines.f90:149-261) for
 * one box, res bins (input_routines.f90:6043-6047; 1000 by default there)
 * between rcut_low^2 and rcut_cbmcsq_max, the largest rcut_cbmc^2 over the
 * system's boxes (<= 0: this box's own).  While set, every CBMC-cutoff
 * molecule pair of the trial-set entry points (cass_trial_energies, _multi,
 * plans, cass_mol_inter_energy with cbmc_flag) is scored by the table lookup
 * of Estimate_MoleculePair_Energy (energy_routines.f90:1528-1587), as
 * Compute_Molecule_Nonbond_Inter_Energy does (:1180-1182): vdW and q-q of
 * the table together in e_vdw / nrg, the overlap test r^2 < rcut_low^2.
 * The Widom batch reads its CBMC column from the table too
 * (energy_routines.f90:1275).
 * res = 0 removes the table.  cass_set_nonbond_params rebuilds it. */
int cass_set_energy_table(cass_engine *eng, int32_t box, int32_t res, double rcut_cbmcsq_max);

/* The per type-pair core radii^2 of the `rcut_low` calc_rmin option
 * (create_nonbond_table.f90:285-301, 398-417; U_max_base = 708 / MINVAL(beta)
 * by default there, input_routines.f90:6998-7013): rminsq[ntypes*ntypes]
 * for this box's charge style.  Host arithmetic. */
int cass_rminsq_table(cass_engine *eng, int32_t box, double u_max_base, double *rminsq);

/* The Widom core-overlap pre-screen of the cell lists (l_sectors): an
 * insertion overlaps when a probe site lies closer to any frame site than the
 * pair's rminsq[ntypes*ntypes] (check_overlap, sector_routines.f90:160-233,
 * called from fragment_growth.f90:477), besides the r^2 < rcut_low^2 test.
 * The spatial sort of the batch stands in for the sector grid.  NULL turns it
 * off.  Radii beyond the pair cutoff are refused. */
int cass_widom_set_rminsq(cass_engine *eng, int32_t box, const double *rminsq);

/* Same, for the trial sets of several boxes in one persistent launch:
 * set s has ntrial[s] trials in box box_of_set[s], species species_of_set[s],
 * coordinates at trial_xyz + 3*xyz_offset[s], results at nrg/overlap +
 * out_offset[s]. */
int cass_trial_energies_multi(cass_engine *eng, int32_t nsets, const int32_t *box_of_set,
                              const int32_t *species_of_set, const int32_t *ntrial,
                              const int64_t *xyz_offset, const int64_t *out_offset,
                              const double *trial_xyz, int32_t cbmc_flag,
                              const int32_t *exclude_mol, double *nrg, int32_t *overlap);

/* A reusable trial plan for cass_trial_energies_multi-style launches: the
 * sets (box, species, trial count, excluded molecule) are fixed at creation;
 * every run takes fresh coordinates (sets back to back, trial-major) and
 * returns E_vdw + E_qq and the overlap flag per trial.  With use_graph the
 * run (copy in, trial kernel, finalize, copy out) is captured once in a
 * hipGraph and replayed.  cass_trial_plan_autotune times the molecule-block
 * sizes 64/128/256 on the plan's boxes and keeps the fastest.  The sets
 * replace the per-box kappa loops of Build_Molecule / Fragment_Placement
 * (fragment_growth.f90:383-579, 1926-2058) run for many boxes at once. */
typedef struct cass_trial_plan cass_trial_plan;
int cass_trial_plan_create(cass_engine *eng, int32_t nsets, const int32_t *box_of_set,
                           const int32_t *species_of_set, const int32_t *ntrial,
                           const int32_t *exclude_mol, int32_t cbmc_flag, cass_trial_plan **plan);
int cass_trial_plan_run(cass_trial_plan *plan, const double *trial_xyz, int32_t use_graph,
                        double *nrg, int32_t *overlap);
int cass_trial_plan_autotune(cass_trial_plan *plan, const double *trial_xyz, int32_t *block);
/* Per-set species (same site count) and/or excluded molecule for later runs. */
int cass_trial_plan_update(cass_trial_plan *plan, const int32_t *species_of_set,
                           const int32_t *exclude_mol);
int cass_trial_plan_destroy(cass_trial_plan *plan);

/* Compute_System_Total_Energy (energy_routines.f90:2648-2953): fills *e
 * and *overlap.  The intra terms are the nonbonded ones plus the harmonic
 * angle and dihedral energies of every species with a growth description
 * (cass_cbmc_set_species); species without one are rigid (no bonded
 * energy), and bond and improper energies are zero (fixed bonds, no
 * impropers). */
int cass_total_energy(cass_engine *eng, int32_t box, int32_t intra_flag, cass_energy *e,
                      int32_t *overlap);

/* Compute_System_Total_Energy (energy_routines.f90:2648-2953) of nboxes
 * distinct boxes in one set of launches, as the volume moves need for every
 * box they change (move_volume.f90, move_vol_swap.f90:322-383 for the two
 * boxes of a GEMC volume swap, many boxes at once for batches of NPT or
 * GEMC systems): out[i] and overlap[i] equal what cass_total_energy
 * returns for boxes[i], bit for bit, and each Ewald box's structure factors
 * are refreshed as by cass_ewald_full. */
int cass_total_energy_batch(cass_engine *eng, int32_t nboxes, const int32_t *boxes, int32_t intra_flag,
                            cass_energy *out, int32_t *overlap);

/* Compute_LR_Correction (energy_routines.f90:2956-3023) for the given bead
 * counts per type (nint_beads[ntypes]). */
int cass_lrc(cass_engine *eng, int32_t box, const double *nint_beads, double *e_lrc);

/* Compute_Molecule_Self_Energy (energy_routines.f90:2598-2645). */
int cass_mol_self_energy(cass_engine *eng, int32_t box, int32_t species, double *e_self);

/* ------------------------------------------------------------ reciprocal */
/* Ewald_Reciprocal_Lattice_Vector_Setup (energy_routines.f90:2170-2323):
 * same k set, order (nz, ny, nx) and Cn.  Returns the count in *nvecs. */
int cass_ewald_setup(cass_engine *eng, int32_t box, int32_t *nvecs);

/* Compute_System_Ewald_Reciprocal_Energy (energy_routines.f90:4111-4231):
 * per-molecule cos/sin sums, box sums and the reciprocal energy. */
int cass_ewald_full(cass_engine *eng, int32_t box, double *e_recip);

/* Update_System_Ewald_Reciprocal_Energy (energy_routines.f90:2326-2497) for
 * molecule `mol` at new coordinates xyz (translation / rotation / intra /
 * insertion; NULL for deletion).  The box sums are updated tentatively and
 * the new TOTAL reciprocal energy is returned, as the reference does;
 * *de_recip (may be NULL) gets E_new - E_old computed term by term
 * (sum_k Cn (2 C dC + dC^2 + 2 S dS + dS^2)), which keeps its relative
 * accuracy in mixed precision.  Follow with cass_ewald_commit or
 * cass_ewald_revert (the caller restore of move_translate.f90:296-306). */
int cass_ewald_move(cass_engine *eng, int32_t box, int32_t mol, int32_t move_flag,
                    const double *xyz, double *e_recip_total, double *de_recip);
int cass_ewald_commit(cass_engine *eng, int32_t box);
int cass_ewald_revert(cass_engine *eng, int32_t box);

/* Update_System_Ewald_Reciprocal_Energy_Widom (energy_routines.f90:2500-2550)
 * for ntrial test molecules of `species` at trial_xyz, without mutating the
 * box sums: e_recip[t] is the total reciprocal energy with molecule t added. */
int cass_ewald_widom(cass_engine *eng, int32_t box, int32_t species, int32_t ntrial,
                     const double *trial_xyz, double *e_recip);

/* ----------------------------------------------------------------- Widom */
/* The insertion loop of Widom_Insert (widom_insert.f90:319-489) for a rigid,
 * single-fragment test species with kappa_ins = 1, all insertions in one
 * launch.  Placement u[0..5] per insertion comes from a counter-based stream
 * (seed, insertion index): COM = (u0,u1,u2) - 1/2 in box units and a uniform
 * rotation from (u3,u4,u5).  Per insertion: the inter energy at the full
 * cutoff (and at rcut_cbmc for the max_kBT overlap test of Build_Molecule),
 * the reciprocal energy change dE_recip of adding the molecule, and
 * widom_var = exp(-beta*dE) with dE = E_inter + dE_recip + e_const
 * (e_const = lrc_diff + E_self + intramolecular; the reference's
 * E_reciprocal - E_recip_in is dE_recip).  Insertions are scored in a
 * spatially sorted order; every value is written at its insertion index.
 * Sums are FP64.  If widom_var is non-NULL it receives every insertion's
 * value (n_ins doubles). */
typedef struct cass_widom_result {
  double widom_sum;         /* sum of widom_var (prefactor V/(N Lambda^3) NOT applied) */
  int64_t n_overlaps;       /* insertions rejected by r^2 < rcut_low^2 */
  int64_t n_insertions;
  double e_const;           /* lrc_diff + E_self + intramolecular */
} cass_widom_result;

int cass_widom_batch(cass_engine *eng, int32_t box, int32_t species, int64_t n_ins,
                     uint64_t seed, double *widom_var, cass_widom_result *res);

/* Rigid geometry of the test species (xyz[natoms*3], any position and
 * orientation) used by cass_widom_batch; *e_intra_const receives its
 * intramolecular nonbonded energy (Compute_Molecule_Nonbond_Intra_Energy,
 * energy_routines.f90:980-1085: intra vdW + intra q-q + periodic q-q), which
 * is constant for a rigid molecule and enters widom_var through e_const. */
int cass_widom_set_template(cass_engine *eng, int32_t box, int32_t species, const double *xyz,
                            double *e_intra_const);

/* The per-insertion body of Widom_Insert (widom_insert.f90:378-447) at n
 * explicit placements xyz[n*natoms*3], through the same kernel as
 * cass_widom_batch: eout[4*i..] = {E_inter at the full cutoff, E_inter at
 * rcut_cbmc, reciprocal energy change, overlap}; widom_var[i] as in
 * cass_widom_batch (either pointer may be NULL). */
int cass_widom_placements(cass_engine *eng, int32_t box, int32_t species, int64_t n,
                          const double *xyz, double *widom_var, double *eout,
                          cass_widom_result *res);

/* ------------------------------------------------------ CBMC growth
 * A flexible species grown fragment by fragment, as Build_Molecule grows it
 * (fragment_growth.f90:72-707).  The description mirrors the MCF's
 * Fragment_Info / Fragment_Connectivity sections and the fragment
 * conformation libraries (input_routines.f90:2664-2960, 3466-3480), the
 * bonded terms the trial weights and the acceptance use (Bond_Info,
 * Angle_Info, Dihedral_Info; input_routines.f90:1690-2360), and the kappa
 * counts of CBMC_Info (input_routines.f90:5931-6104).  Atom and fragment
 * indices are 0-based.  Anchors (atoms bonded to two or more atoms of their
 * fragment, input_routines.f90:2760-2820), the first-fragment probabilities
 * (natoms share, :2843-2850) and the fragment connections
 * (Get_Fragment_Connectivity_Info) are derived from these arrays as the
 * reference derives them.  Ring fragments (more than one anchor) are
 * refused. */
typedef struct cass_cbmc_species {
  int32_t nfrag;
  const int32_t *frag_natoms;     /* [nfrag] */
  const int32_t *frag_atoms;      /* [sum frag_natoms] Fragment_Info order (branch point first) */
  int32_t nfrag_bonds;
  const int32_t *frag_bonds;      /* [2*nfrag_bonds] Fragment_Connectivity pairs */
  const int32_t *frag_nconfig;    /* [nfrag] conformations in each fragment's library */
  const double *frag_coords;      /* libraries back to back: nconfig*natoms*3 per fragment,
                                     atoms in Fragment_Info order */
  int32_t nbonds;
  const int32_t *bond_atoms;      /* [2*nbonds] (fixed bonds: no energy) */
  int32_t nangles;
  const int32_t *angle_atoms;     /* [3*nangles] */
  const double *angle_k;          /* [nangles] kboltz*K, internal units; 0 for a fixed angle */
  const double *angle_theta0;     /* [nangles] radians (PI/180 with the truncated PI) */
  int32_t ndihedrals;
  const int32_t *dihedral_atoms;  /* [4*ndihedrals] */
  const double *dihedral_rb;      /* [6*ndihedrals] Ryckaert-Bellemans c0..c5, internal units
                                     (OPLS converted as input_routines.f90:2104-2109) */
  int32_t kappa_ins, kappa_rot, kappa_dih;
} cass_cbmc_species;

/* Registers the growth description of `species` (copied to the device). */
int cass_cbmc_set_species(cass_engine *eng, int32_t species, const cass_cbmc_species *cs);

/* Grand-canonical chains of CBMC insertions and deletions, one box per
 * workgroup, every box's whole move loop in one launch: per move the draws
 * of gcmc_driver.f90:90-200 restricted to insertion and deletion, then
 * Insertion (move_insert.f90:22-424) or Deletion (move_delete.f90:22-416)
 * of the box's sorbate species with Build_Molecule / Fragment_Placement
 * (fragment_growth.f90:72-707, 1449-2132) on the box's own copy of the
 * reference's random stream; the accepted state (coordinates, live flags,
 * the locate order and the reservoir of free molecule slots, bead counts
 * and the Energy_Class) is written back.  Boxes with Ewald sums are
 * refused.  The sorbate's molecule slots of a box are the reference's
 * molecule indices lm = 1..max_molecules; locate lists the live ones in the
 * reference's order and the reservoir the free ones, stack top last. */
typedef struct cass_gcmc_box {
  int32_t box;              /* engine box */
  int32_t species;          /* the sorbate (its slots: first_slot .. first_slot+max_mols-1) */
  int32_t first_slot;
  int32_t max_mols;
  double prob_insert;       /* cut_insertion; deletion takes the rest */
  double mu;                /* chem_potential, internal units (input_routines.f90:4256-4259) */
  double de_broglie;        /* Angstrom (input_routines.f90:4267) */
} cass_gcmc_box;

typedef struct cass_gcmc_state {
  cass_rng rng;
  cass_energy energy;
  int32_t nmols;            /* live sorbate molecules */
  int32_t nres;             /* reservoir size */
  int32_t *locate;          /* [max_mols] 0-based slot offsets, first nmols live */
  int32_t *reservoir;       /* [max_mols] free slot offsets, top = reservoir[nres-1] */
} cass_gcmc_state;

typedef struct cass_gcmc_record {
  uint8_t *kind;            /* [nboxes*nsteps] 0 insertion, 1 deletion */
  uint8_t *accepted;        /* [nboxes*nsteps] */
  int32_t *nmols;           /* [nboxes*nsteps] after the move */
  double *energy;           /* [nboxes*nsteps] running total energy */
  int64_t *rng_state;       /* [nboxes*nsteps*5] */
} cass_gcmc_record;

int cass_gcmc_run_device(cass_engine *eng, int32_t nboxes, const cass_gcmc_box *boxes,
                         cass_gcmc_state *states, int64_t nsteps, cass_gcmc_record *rec);

/* GEMC_Particle_Transfer (move_mol_swap.f90:22-769) in npairs pairs of boxes,
 * one workgroup per pair in one launch, the pair's whole sequence of nsteps
 * moves of the GEMC loop with transfers only (gemc_driver.f90:91-195, one
 * move draw each).  boxes[2p], boxes[2p+1] and states[2p], states[2p+1]
 * describe pair p as for cass_gcmc_run_device: the species (the same in
 * both; one swappable species, no charges), each box's slots of it, their
 * live / free lists and Energy_Class (prob_insert, mu and de_broglie are not
 * used).  Each move takes a molecule out of a box chosen by molecule
 * fraction into the other (a free slot of it), growing it there with
 * Build_Molecule (fragment order drawn) and regrowing it in reverse in the
 * box it leaves with the same order; the acceptance carries both boxes'
 * energy changes at their own beta, ln_pfor - ln_prev and
 * log(P_forward / P_reverse), the same draws and decisions as the reference.
 * The pair's generator is states[2p].rng; on return both states hold it.
 * rec (may be NULL), per box [2*npairs*nsteps]: kind = 0 or 1, the index in
 * its pair of the box the move took a molecule from; accepted; the box's
 * count, running total energy and generator state after the move.
 * CASS_ERR_STATE when a box has no free slot or the molecule to transfer
 * cannot be regrown where it is (the reference aborts). */
int cass_gemc_run_device(cass_engine *eng, int32_t npairs, const cass_gcmc_box *boxes,
                         cass_gcmc_state *states, int64_t nsteps, cass_gcmc_record *rec);

/* Picks the chain's lanes per box (128, 256, 512 or 1024) by timing runs of
 * nsteps moves over the given boxes that change neither the boxes nor the
 * states, and keeps it for the engine's later runs; *block gets it.
 * Instrumentation of the batched path; no counterpart in the reference. */
int cass_gcmc_autotune(cass_engine *eng, int32_t nboxes, const cass_gcmc_box *boxes,
                       cass_gcmc_state *states, int64_t nsteps, int32_t *block);

/* Widom insertions of a CBMC-grown species (Widom_Insert,
 * widom_insert.f90:22-594 with Build_Molecule for every insertion), one
 * workgroup per insertion.  rng != NULL: the reference's single stream, the
 * insertions in sequence as one thread runs them (bit-exact draws; slow);
 * rng == NULL: insertion i draws from its own stream seeded from (seed, i),
 * all insertions in parallel.  widom_sum excludes the prefactor
 * V/(N Lambda^3) as cass_widom_batch does; sub[k] (n_sub >= 1 entries, may be
 * NULL) receives the sub-interval sums of widom_insert.f90:481-484 without
 * prefactor or 1/subinterval scaling. */
int cass_widom_cbmc_batch(cass_engine *eng, int32_t box, int32_t species, int64_t n_ins,
                          cass_rng *rng, uint64_t seed, int32_t n_sub, double *sub,
                          double *widom_var, cass_widom_result *res);

/* cass_widom_cbmc_batch with the per-insertion outputs of est_emax
 * (widom_insert.f90:178-186, 388, 466-476): widom_var[i] (no prefactor),
 * overlap[i] and eij_max[i], the largest pair energy Eij_inter_vdw + bare
 * q-q over the inserted molecule's in-cutoff site pairs in the full-cutoff
 * pass (Eij_max of energy_routines.f90:1702-1705; 0 where overlap[i]).
 * The vdW part has the engine's precision (FP64 with CASS_PREC_FP64).  Needs
 * at most 8 species, 128 species sites and 16 atom types (CASS_ERR_ARG
 * otherwise).  All three arrays hold n_ins entries, host memory.
 * rsq_min (may be NULL; n_ins x S x natoms(species) doubles, S = the
 * topology's species sites, in species order) receives
 * est_atompair_rminsq's closest r^2 of every (species site, inserted atom)
 * over the in-cutoff pairs of the same pass (swi_atompair_rsqmin,
 * energy_routines.f90:1636-1643, 1700), 10000 where no pair was in range
 * (widom_insert.f90:325). */
int cass_widom_cbmc_emax(cass_engine *eng, int32_t box, int32_t species, int64_t n_ins,
                         cass_rng *rng, uint64_t seed, double *widom_var, double *eij_max,
                         uint8_t *overlap, double *rsq_min, cass_widom_result *res);

/* est_emax / est_atompair_rminsq for a rigid test molecule: the insertions
 * of cass_widom_batch (xyz NULL; seed as there) or of explicit placements
 * (xyz, n x natoms x 3, as cass_widom_placements), each with its widom_var
 * (no prefactor), overlap flag, Eij_max (0 where overlap) and, with rsq_min
 * (may be NULL; n x S x natoms, S = the topology's species sites), the
 * closest in-cutoff r^2 of every (species site, probe atom), 10000 where no
 * pair was in range.  Same definitions as cass_widom_cbmc_emax
 * (energy_routines.f90:1636-1643, 1700-1705; widom_insert.f90:325), here
 * for every pair style, Ewald included; FP64.  Host arrays. */
int cass_widom_emax(cass_engine *eng, int32_t box, int32_t species, int64_t n, uint64_t seed,
                    const double *xyz, double *widom_var, double *eij_max, uint8_t *overlap,
                    double *rsq_min, cass_widom_result *res);

/* Host code.  The est_emax histogram of one species in one box, fed one
 * Widom_Insert call (one frame) at a time (widom_insert.f90:466-476 and
 * 490-520, with coarsen_w_max :570-589).  Running totals of ub + 1 bins:
 * w_max (the reference's w_max), w_sum (Eij_w_sum), freq (Eij_freq_total)
 * and *factor (Eij_factor: bin = INT(Eij_max * factor); start it at
 * 2 beta for 0.5 kT bins, ub = 2047 as the reference sizes Eij_ind_ubound,
 * input_routines.f90:5683).  Insertions without overlap are binned; an
 * insertion past bin ub halves the frame's factor, merging bin pairs, and
 * the totals are then merged to match before the frame's bins, scaled by
 * prefactor (V / ((N + 1) Lambda^3)), are added.  CASS_ERR_ARG for a
 * negative or non-finite eij_max of an insertion without overlap. */
int cass_emax_frame(int32_t ub, double *factor, double *w_max, double *w_sum, int64_t *freq,
                    int64_t n, const double *widom_var, const double *eij_max,
                    const uint8_t *overlap, double prefactor);

/* Host code.  Estimate_Pair_Emax (pair_emax_estimation.f90:41-77): the
 * weight fraction w_sum[k] / widom_sum of each bin, added from the top bin
 * down until the sum passes 1e-10; *emax = that bin's upper edge in kT (the
 * recommended U*_max), *nskips = the insertions in the bins above it.
 * widom_sum is the species' prefactor-weighted sum over all frames.
 * w_frac (ub + 1 entries, may be NULL) receives the fractions, the .emax
 * file's w_frac column. */
int cass_emax_estimate(int32_t ub, double factor, const double *w_sum, const int64_t *freq,
                       double widom_sum, double beta, double *emax, int64_t *nskips,
                       double *w_frac);

/* Host code.  The est_atompair_rminsq histograms of one species in one box
 * (`specific write step res`), fed one Widom_Insert call at a time
 * (widom_insert.f90:450-464, 522-539): for each insertion without overlap
 * and each (solvent site k, inserted atom a) whose closest r^2 lies below
 * rcut_low^2 + step * res, bin INT((r^2 - rcut_low^2 + step) / step) of
 * that pair takes widom_var (maximum, sum, count); the totals then take the
 * frame's, scaled by prefactor.  rows[k] (nsolv entries) is solvent site
 * k's row in each insertion's nrows x nsolute block of rsq_min
 * (cass_widom_cbmc_emax); the solvent sites are those of the species with
 * molecules in the frames, in species order (solvent_base,
 * atompair_nrg_table_routines.f90:88-97).  Totals w_max, w_sum, freq are
 * [nsolv][nsolute][res] (the reference's rsqmin_atompair_w_max / _w_sum /
 * _freq).  Bin indices are held in 1..res. */
int cass_rminsq_frame(int32_t nsolv, const int32_t *rows, int32_t nsolute, int32_t nrows,
                      int32_t res, double step, double rcut_lowsq, double *w_max, double *w_sum,
                      int64_t *freq, int64_t n, const double *widom_var, const double *rsq_min,
                      const uint8_t *overlap, double prefactor);

/* Host code.  Estimate_Pair_rminsq (pair_emax_estimation.f90:79-168) at one
 * tolerance: ind[k][a] (nsolv x nsolute) is the first bin (1-based, res + 1
 * if none) at which pair (k, a)'s weight fractions w_sum / widom_sum, summed
 * from the innermost bin out, pass tol: the .rminsq file's table.  *nskips
 * and *wmax are the largest over the pairs of the insertions and of the
 * maximal weight in the bins inside it (Get_rminsq_nskips,
 * Get_rminsq_wmax, as the log prints them). */
int cass_rminsq_estimate(int32_t nsolv, int32_t nsolute, int32_t res, const double *w_max,
                         const double *w_sum, const int64_t *freq, double widom_sum, double tol,
                         int32_t *ind, int64_t *nskips, double *wmax);

/* ---------------------------------------------------------------- adjoint
 * New (no counterpart in the reference): derivatives of the box's total
 * intermolecular pair energy (inter_vdw + inter_q, real-space Ewald/DSF/cut)
 * plus the reciprocal and self energies with respect to the per-type LJ
 * parameters eps[t] and sigma[t] of the diagonal table entries (propagated
 * through Lorentz-Berthelot mixing sigma_ij = (sigma_i+sigma_j)/2,
 * eps_ij = sqrt(eps_i eps_j)) and the per-atom-kind charges, plus forces
 * -dE/dr per site.  Accumulated in FP64.  Arrays: de_deps[ntypes],
 * de_dsig[ntypes], de_dq[sum natoms] (per species atom), forces[3*nsites]. */
int cass_adjoint(cass_engine *eng, int32_t box, double *energy, double *de_deps,
                 double *de_dsig, double *de_dq, double *forces);

/* New (no counterpart in the reference): coordinate frames of a box for the
 * batched adjoint, e.g. the saved configurations of an MC run
 * (write_properties / the .xyz trajectory of the reference).  xyz holds
 * nframes x nsites x 3 coordinates in the box's site order, molecules whole;
 * they are copied to device memory owned by the engine, replacing any frames
 * stored before (one set per engine).  The frames keep the box's current
 * molecule table; the live flags used are the box's at the time of
 * cass_adjoint_frames.  Non-finite coordinates: CASS_ERR_ARG. */
int cass_adjoint_set_frames(cass_engine *eng, int32_t box, int32_t nframes, const double *xyz);

/* cass_adjoint for frames [first, first + count) of the stored set, all in
 * a few launches: per frame energy[f], de_deps[f * ntypes + t],
 * de_dsig[f * ntypes + t], de_dq[f * sum natoms + k] and, if forces is not
 * NULL, forces[(f * nsites + s) * 3 + d].  Any output pointer may be NULL.
 * CASS_ERR_STATE if no frames are stored for this box or its molecules
 * changed since. */
int cass_adjoint_frames(cass_engine *eng, int32_t box, int32_t first, int32_t count, double *energy,
                        double *de_deps, double *de_dsig, double *de_dq, double *forces);

/* -------------------------------------------------------- host-side chain
 * The reference's random-number stream (random_generators.f90:51-122), the
 * Metropolis test (accept_or_reject.f90:22-65) and the NVT move loop of
 * nvtmc_driver.f90:94-152 with Translate (move_translate.f90:23) and Rotate
 * (move_rotate.f90:23) for one box, every energy evaluated by the engine.
 * Per-move record: kind (0 translate, 1 rotate), accepted flag and the
 * running total energy after the move. */
void cass_rng_init(cass_rng *r, int64_t i1, int64_t i3);      /* init_seeds, one thread */
double cass_rng_uniform(cass_rng *r);                         /* rranf */
int64_t cass_rng_int(cass_rng *r);                            /* rranint */
int32_t cass_accept_or_reject(cass_rng *r, double ln_pacc);   /* accept_or_reject */

typedef struct cass_nvt_options {
  double prob_translate;    /* cut_trans; rotation takes the rest */
  double max_disp;          /* max_disp(is, box) */
  double max_rot;           /* max_rot(is, box) */
  int32_t linear;           /* species is linear: Euler rotation (move_rotate.f90:211) */
  int32_t species;          /* the single mobile species */
} cass_nvt_options;

typedef struct cass_nvt_record {
  uint8_t *kind;            /* [nsteps] or NULL */
  uint8_t *accepted;        /* [nsteps] or NULL */
  double *energy;           /* [nsteps] running total, or NULL */
  int64_t *rng_state;       /* [5*nsteps] state after each move, or NULL */
  double *ln_pacc;          /* [nsteps] beta*dE of moves that reached the test, else NaN */
} cass_nvt_record;

/* Runs nsteps moves from the box's current state; *energy holds the
 * Energy_Class on entry (e.g. from cass_total_energy) and is updated. */
int cass_nvt_run(cass_engine *eng, int32_t box, cass_rng *rng, const cass_nvt_options *opt,
                 int64_t nsteps, cass_energy *energy, cass_nvt_record *rec);

/* The same move loop resident on the device: one workgroup runs the moves
 * in sequence (draws, trial coordinates, old/new molecule energies, the
 * staged reciprocal sums, accept_or_reject and the commit) with no host
 * round trip per move; the host mirrors, *rng and *energy are brought up
 * to date at the end.  Same arguments and results as cass_nvt_run
 * (nvtmc_driver.f90:94-152); molecules of at most 64 sites.  A box so large
 * that one workgroup would take longer than cass_nvt_run's launches takes
 * those. */
int cass_nvt_run_device(cass_engine *eng, int32_t box, cass_rng *rng, const cass_nvt_options *opt,
                        int64_t nsteps, cass_energy *energy, cass_nvt_record *rec);

/* cass_nvt_run_device for nboxes distinct boxes at once, one workgroup per
 * box in the same launches: independent chains (replicas of a system, or
 * boxes at other state points), each with its own generator rngs[i],
 * options opts[i], energies energies[i] and records recs[i] (recs may be
 * NULL).  Every chain's results equal those of its own
 * cass_nvt_run_device call. */
int cass_nvt_run_device_batch(cass_engine *eng, int32_t nboxes, const int32_t *boxes, cass_rng *rngs,
                              const cass_nvt_options *opts, int64_t nsteps, cass_energy *energies,
                              cass_nvt_record *recs);

/* Chains of Cut_N_Grow regrowth moves (move_regrow.f90:22-510) on the
 * device, one workgroup per box, every box's whole move loop in one launch:
 * per move the NVT driver's move draw (nvtmc_driver.f90:94-230 with
 * prob_regrowth = 1), the box, species and molecule draws, Cut_Regrow
 * (fragment_growth.f90:1118-1312: the fragment bond cut by prob_del1, the
 * cut-off fragments regrown by Fragment_Placement, :1449-2132), the
 * full-cutoff energies, the reverse pass over the molecule's own
 * configuration and the acceptance; the accepted or re-placed coordinates
 * and the Energy_Class are written back (the host mirrors follow).  The
 * regrown species has a growth description (cass_cbmc_set_species) of two
 * or more fragments and no charges.  rngs[i] and energies[i] are box i's
 * generator and Energy_Class, updated; recs[i] (or recs NULL) takes kind 2
 * per move, the decisions, running total energy, ln_pacc (NaN for moves
 * rejected before the test) and generator states.  CASS_ERR_STATE where
 * the reference aborts (a molecule's own configuration cannot be regrown);
 * that box stops at the move. */
typedef struct cass_regrow_box {
  int32_t box;              /* engine box */
  int32_t species;          /* the regrown species */
  int32_t first_slot;       /* its molecules: first_slot + locate[im] */
  int32_t nmols;            /* nmols(is, ibox) */
  const int32_t *locate;    /* [nmols] slot offsets in the reference's locate order */
} cass_regrow_box;

int cass_regrow_run_device(cass_engine *eng, int32_t nboxes, const cass_regrow_box *boxes, cass_rng *rngs,
                           int64_t nsteps, cass_energy *energies, cass_nvt_record *recs);

#ifdef __cplusplus
}
#endif
#endif /* CASS_GPU_H */
