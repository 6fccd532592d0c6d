"""Python host layer over libcassgpu.so (the C ABI in include/cass_gpu.h).

Mirrors the reference's energy interface one box at a time: the methods are
named after the Fortran subroutines they replace (energy_routines.f90,
fragment_growth.f90, widom_insert.f90) and take the same arguments, with
0-based molecule and species indices.  There is no CPU fallback: if the HIP
library is missing or no GPU is visible, construction raises.
"""
from __future__ import annotations

import ctypes as C
import weakref
import os

import numpy as np

from . import abi
from . import systems as S

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(HERE, "libcassgpu.so")

FP64 = 0
MIXED = 1     # FP32 real-space q-q pair terms, FP64 LJ/Mie and sums
FP32 = 2      # FP32 for both pair terms, FP64 sums

_STATUS = {0: "ok", 1: "bad argument", 2: "HIP error", 3: "out of device memory", 4: "too many k vectors",
           5: "net charge", 6: "call out of order", 7: "no GPU visible", 8: "cutoff exceeds half the box"}


class CassError(RuntimeError):
    def __init__(self, code, msg):
        super().__init__(f"{_STATUS.get(code, code)}: {msg}")
        self.code = code


_LIB = None


def load_library(path=LIB_PATH):
    """Loads libcassgpu.so and declares the C ABI.  Raises if it is missing."""
    global _LIB
    if _LIB is not None:
        return _LIB
    if not os.path.exists(path):
        raise FileNotFoundError(f"{path} is not built; run __graft_entry__.build() or make -C cassandra_amd/csrc")
    lib = C.CDLL(path)
    P = C.POINTER
    d, i32, i64, u64, vp = C.c_double, C.c_int32, C.c_int64, C.c_uint64, C.c_void_p
    sig = {
        "cass_params_derive": (i32, [P(abi.CassParams)]),
        "cass_engine_create": (i32, [i32, P(abi.CassTopology), i32, P(vp)]),
        "cass_engine_destroy": (i32, [vp]),
        "cass_set_precision": (i32, [vp, i32]),
        "cass_set_overlap": (i32, [vp, i32]),
        "cass_last_error": (C.c_char_p, [vp]),
        "cass_last_kernel_ms": (i32, [vp, P(d)]),
        "cass_last_stage_ms": (i32, [vp, P(d)]),
        "cass_box_create": (i32, [vp, P(abi.CassParams), i32, P(i32)]),
        "cass_box_upload": (i32, [vp, i32, i32, P(i32), P(i32), P(d), P(d), P(d)]),
        "cass_mol_update": (i32, [vp, i32, i32, i32, P(d), P(d), P(d)]),
        "cass_box_download": (i32, [vp, i32, P(d)]),
        "cass_mol_inter_energy": (i32, [vp, i32, i32, i32, P(d), P(d), P(d), P(d), P(d), P(i32)]),
        "cass_mol_intra_energy": (i32, [vp, i32, i32, i32, P(d), P(d), P(d), P(d), P(i32)]),
        "cass_trial_energies": (i32, [vp, i32, i32, i32, P(d), i32, i32, P(d), P(i32)]),
        "cass_trial_energies_noalloc": (i32, [vp, i32, i32, i32, P(d), i32, i32, P(d), P(i32)]),
        "cass_cbmc_set_species": (i32, [vp, i32, P(abi.CassCbmcSpecies)]),
        "cass_gcmc_run_device": (i32, [vp, i32, P(abi.CassGcmcBox), P(abi.CassGcmcState), i64,
                                       P(abi.CassGcmcRecord)]),
        "cass_net_charge": (i32, [P(abi.CassParams), P(abi.CassTopology), i32, P(i32), P(i32), P(d)]),
        "cass_gcmc_autotune": (i32, [vp, i32, P(abi.CassGcmcBox), P(abi.CassGcmcState), i64, P(i32)]),
        "cass_widom_cbmc_batch": (i32, [vp, i32, i32, i64, P(abi.CassRng), u64, i32, P(d), P(d),
                                        P(abi.CassWidomResult)]),
        "cass_widom_cbmc_emax": (i32, [vp, i32, i32, i64, P(abi.CassRng), u64, P(d), P(d), P(C.c_uint8), P(d),
                                       P(abi.CassWidomResult)]),
        "cass_rminsq_frame": (i32, [i32, P(i32), i32, i32, i32, d, d, P(d), P(d), P(i64), i64, P(d), P(d),
                                    P(C.c_uint8), d]),
        "cass_rminsq_estimate": (i32, [i32, i32, i32, P(d), P(d), P(i64), d, d, P(i32), P(i64), P(d)]),
        "cass_emax_frame": (i32, [i32, P(d), P(d), P(d), P(i64), i64, P(d), P(d), P(C.c_uint8), d]),
        "cass_emax_estimate": (i32, [i32, d, P(d), P(i64), d, d, P(d), P(i64), P(d)]),
        "cass_gemc_run_device": (i32, [vp, i32, P(abi.CassGcmcBox), P(abi.CassGcmcState), i64,
                                       P(abi.CassGcmcRecord)]),
        "cass_widom_emax": (i32, [vp, i32, i32, i64, u64, P(d), P(d), P(d), P(C.c_uint8), P(d),
                                  P(abi.CassWidomResult)]),
        "cass_set_energy_table": (i32, [vp, i32, i32, d]),
        "cass_box_set_params": (i32, [vp, i32, P(abi.CassParams)]),
        "cass_rminsq_table": (i32, [vp, i32, d, P(d)]),
        "cass_widom_set_rminsq": (i32, [vp, i32, P(d)]),
        "cass_total_energy": (i32, [vp, i32, i32, P(abi.CassEnergy), P(i32)]),
        "cass_total_energy_batch": (i32, [vp, i32, P(i32), i32, P(abi.CassEnergy), P(i32)]),
        "cass_lrc": (i32, [vp, i32, P(d), P(d)]),
        "cass_mol_self_energy": (i32, [vp, i32, i32, P(d)]),
        "cass_ewald_setup": (i32, [vp, i32, P(i32)]),
        "cass_ewald_full": (i32, [vp, i32, P(d)]),
        "cass_ewald_move": (i32, [vp, i32, i32, i32, P(d), P(d), P(d)]),
        "cass_ewald_commit": (i32, [vp, i32]),
        "cass_ewald_revert": (i32, [vp, i32]),
        "cass_ewald_widom": (i32, [vp, i32, i32, i32, P(d), P(d)]),
        "cass_widom_batch": (i32, [vp, i32, i32, i64, u64, P(d), P(abi.CassWidomResult)]),
        "cass_widom_set_template": (i32, [vp, i32, i32, P(d), P(d)]),
        "cass_widom_placements": (i32, [vp, i32, i32, i64, P(d), P(d), P(d), P(abi.CassWidomResult)]),
        "cass_rng_init": (None, [P(abi.CassRng), i64, i64]),
        "cass_rng_uniform": (d, [P(abi.CassRng)]),
        "cass_rng_int": (i64, [P(abi.CassRng)]),
        "cass_accept_or_reject": (i32, [P(abi.CassRng), d]),
        "cass_nvt_run": (i32, [vp, i32, P(abi.CassRng), P(abi.CassNvtOptions), i64, P(abi.CassEnergy),
                               P(abi.CassNvtRecord)]),
        "cass_nvt_run_device": (i32, [vp, i32, P(abi.CassRng), P(abi.CassNvtOptions), i64, P(abi.CassEnergy),
                               P(abi.CassNvtRecord)]),
        "cass_nvt_run_device_batch": (i32, [vp, i32, P(i32), P(abi.CassRng), P(abi.CassNvtOptions), i64,
                                            P(abi.CassEnergy), P(abi.CassNvtRecord)]),
        "cass_regrow_run_device": (i32, [vp, i32, P(abi.CassRegrowBox), P(abi.CassRng), i64, P(abi.CassEnergy),
                                         P(abi.CassNvtRecord)]),
    }
    sig.update({
        "cass_trial_energies_multi": (i32, [vp, i32, P(i32), P(i32), P(i32), P(i64), P(i64), P(d), i32, P(i32),
                                            P(d), P(i32)]),
        "cass_adjoint": (i32, [vp, i32, P(d), P(d), P(d), P(d), P(d)]),
        "cass_adjoint_set_frames": (i32, [vp, i32, i32, P(d)]),
        "cass_adjoint_frames": (i32, [vp, i32, i32, i32, P(d), P(d), P(d), P(d), P(d)]),
        "cass_set_nonbond_params": (i32, [vp, P(d), P(d), P(d)]),
        "cass_trial_plan_create": (i32, [vp, i32, P(i32), P(i32), P(i32), P(i32), i32, P(vp)]),
        "cass_trial_plan_run": (i32, [vp, P(d), i32, P(d), P(i32)]),
        "cass_trial_plan_autotune": (i32, [vp, P(d), P(i32)]),
        "cass_trial_plan_destroy": (i32, [vp]),
        "cass_trial_plan_update": (i32, [vp, P(i32), P(i32)]),
    })
    optional = {}
    for name, (res, args) in list(sig.items()) + list(optional.items()):
        if not hasattr(lib, name):
            if name in optional:
                continue
            raise ImportError(f"{path} does not export {name}")
        fn = getattr(lib, name)
        fn.restype = res
        fn.argtypes = args
    _LIB = lib
    return lib


def derive(system: S.System) -> abi.CassParams:
    """cass_params of a box (raw block from the System, derived block by
    cass_params_derive)."""
    p = abi.raw_params(system)
    rc = load_library().cass_params_derive(C.byref(p))
    if rc:
        raise CassError(rc, "cass_params_derive")
    return p


def _p(a, t=C.c_double):
    return None if a is None else a.ctypes.data_as(C.POINTER(t))


def _at_least(n, **lists):
    """The native call reads and writes n entries of each list: fewer raise."""
    for name, entries in lists.items():
        if len(entries) < n:
            raise ValueError(f"{name}: {len(entries)} entries for {n} boxes")


def _energies_in(energies):
    """A CassEnergy array of energy dicts."""
    ens = (abi.CassEnergy * len(energies))()
    if energies:
        _energy_rows(ens)[:] = [[en.get(f, 0.0) for f in abi.ENERGY_FIELDS] for en in energies]
    return ens


def _energy_rows(ens):
    return np.frombuffer(ens, dtype=np.float64).reshape(len(ens), len(abi.ENERGY_FIELDS))


def _energies_out(ens):
    return [dict(zip(abi.ENERGY_FIELDS, row)) for row in _energy_rows(ens).tolist()] if len(ens) else []


class _NvtRecords:
    """The per-move records of n chains in one array per field, and the
    CassNvtRecord table that points into them."""

    def __init__(self, n, nsteps):
        self.kind, self.acc = np.zeros((n, nsteps), dtype=np.uint8), np.zeros((n, nsteps), dtype=np.uint8)
        self.et, self.lp = np.zeros((n, nsteps)), np.zeros((n, nsteps))
        self.rs = np.zeros((n, nsteps, 5), dtype=np.int64)
        self.table = (abi.CassNvtRecord * n)()
        if n and nsteps:
            fields = (self.kind, self.acc, self.et, self.rs, self.lp)    # the struct's order
            at = np.frombuffer(self.table, dtype=np.uint64).reshape(n, len(fields))
            for f, a in enumerate(fields):
                at[:, f] = a.ctypes.data + np.arange(n, dtype=np.uint64) * np.uint64(a.strides[0])

    def result(self, k, final):
        return dict(kind=self.kind[k], accepted=self.acc[k].astype(bool), energy=self.et[k], ln_pacc=self.lp[k],
                    rng=self.rs[k], final=final)


class Engine:
    """One engine (one GPU, one topology) holding one or more boxes."""

    def __init__(self, system: S.System, max_boxes=1, device=0, precision=FP64):
        self.lib = load_library()
        self.topo = abi.Topology(system)
        self.system = system
        h = C.c_void_p()
        rc = self.lib.cass_engine_create(device, C.byref(self.topo.c), max_boxes, C.byref(h))
        if rc:
            raise CassError(rc, "cass_engine_create (is a GPU visible?)")
        self.h = h
        self.boxes = []
        self._plans = weakref.WeakSet()
        self.set_precision(precision)

    def close(self):
        """Destroys the engine; plans built on it go first (they hold the
        engine's stream and graph executables)."""
        if getattr(self, "h", None):
            for plan in list(getattr(self, "_plans", ())):
                plan.close()
            self.lib.cass_engine_destroy(self.h)
            self.h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    def _chk(self, rc, what):
        if rc:
            raise CassError(rc, f"{what}: {self.lib.cass_last_error(self.h).decode()}")

    def last_kernel_ms(self):
        ms = C.c_double()
        self._chk(self.lib.cass_last_kernel_ms(self.h, C.byref(ms)), "cass_last_kernel_ms")
        return ms.value

    def last_stage_ms(self):
        """(placement + sort, real space, reciprocal + combine, whole batch) of
        the last Widom batch, in ms of device time."""
        ms = (C.c_double * 4)()
        self._chk(self.lib.cass_last_stage_ms(self.h, ms), "cass_last_stage_ms")
        return list(ms)

    def set_precision(self, prec):
        self._chk(self.lib.cass_set_precision(self.h, prec), "cass_set_precision")
        self.precision = prec

    def set_overlap(self, on):
        """cass_set_overlap: independent kernels of a call side by side on a
        second stream (default), or one after another."""
        self._chk(self.lib.cass_set_overlap(self.h, int(bool(on))), "cass_set_overlap")

    def set_nonbond_params(self, eps=None, sig=None, charges=None):
        """cass_set_nonbond_params: full ntypes x ntypes tables (internal units)
        and/or per-atom charges; None keeps the current one."""
        arrs = [None if a is None else np.ascontiguousarray(a, dtype=np.float64).ravel() for a in (eps, sig, charges)]
        self._chk(self.lib.cass_set_nonbond_params(self.h, *[_p(a) for a in arrs]), "cass_set_nonbond_params")

    def trial_plan(self, boxes, species, ntrial, exclude=None, cbmc=True):
        plan = TrialPlan(self, boxes, species, ntrial, exclude, cbmc)
        self._plans.add(plan)
        return plan

    def set_cbmc_species(self, species, cbmc: abi.CbmcSpecies):
        """cass_cbmc_set_species: the growth description of a flexible species."""
        self._cbmc = getattr(self, "_cbmc", {})
        self._cbmc[species] = cbmc
        self._chk(self.lib.cass_cbmc_set_species(self.h, species, C.byref(cbmc.c)), "cass_cbmc_set_species")

    def gemc_run(self, specs, states, nsteps, record=True):
        """cass_gemc_run_device: nsteps GEMC particle transfers in every pair
        of boxes (specs and states as gcmc_run, two consecutive entries per
        pair; prob_insert, mu and de_broglie are not used), one workgroup per
        pair.  The pair's generator is its first state's rng; both states get
        it back.  Returns the records: kind = the index in the pair of the
        box a molecule was taken from, accepted, and per box the molecule
        count, running total energy and generator state ([nboxes, nsteps])."""
        return self.gcmc_run(specs, states, nsteps, record, entry="cass_gemc_run_device")

    def gcmc_run(self, specs, states, nsteps, record=True, entry="cass_gcmc_run_device"):
        """cass_gcmc_run_device: nsteps GCMC insertion / deletion moves in every
        box of specs (dicts: box, species, first_slot, max_mols, prob_insert, mu,
        de_broglie), one workgroup per box in one launch.  states (dicts: rng
        CassRng, energy dict, locate, reservoir) are updated in place; returns
        the per-move records (arrays [nboxes, nsteps])."""
        nb = len(specs)
        bx = (abi.CassGcmcBox * nb)()
        st = (abi.CassGcmcState * nb)()
        ens = _energies_in([s["energy"] for s in states])
        # one array for all boxes' locate and reservoir lists
        at = np.concatenate([[0], np.cumsum([2 * g["max_mols"] for g in specs])])
        slots = np.zeros(max(1, int(at[-1])), dtype=np.int32)
        keep = []
        i32p = C.POINTER(C.c_int32)
        for i, (g, s) in enumerate(zip(specs, states)):
            bx[i] = abi.CassGcmcBox(g["box"], g["species"], g["first_slot"], g["max_mols"], g["prob_insert"],
                                    g["mu"], g["de_broglie"])
            o, m = int(at[i]), g["max_mols"]
            loc, res = slots[o:o + m], slots[o + m:o + 2 * m]
            loc[:len(s["locate"])] = s["locate"]
            res[:len(s["reservoir"])] = s["reservoir"]
            keep += [loc, res]
            x = st[i]
            x.rng = s["rng"]
            x.energy = ens[i]
            x.nmols = len(s["locate"])
            x.nres = len(s["reservoir"])
            x.locate = C.cast(slots.ctypes.data + 4 * o, i32p)
            x.reservoir = C.cast(slots.ctypes.data + 4 * (o + m), i32p)
        rec = None
        if record:
            kind = np.zeros((nb, nsteps), dtype=np.uint8)
            acc = np.zeros((nb, nsteps), dtype=np.uint8)
            nm = np.zeros((nb, nsteps), dtype=np.int32)
            en = np.zeros((nb, nsteps))
            rr = np.zeros((nb, nsteps, 5), dtype=np.int64)
            rec = abi.CassGcmcRecord(_p(kind, C.c_uint8), _p(acc, C.c_uint8), _p(nm, C.c_int32), _p(en),
                                     _p(rr, C.c_int64))
        n_arg = nb // 2 if entry == "cass_gemc_run_device" else nb
        self._chk(getattr(self.lib, entry)(self.h, n_arg, bx, st, nsteps, C.byref(rec) if rec else None), entry)
        for i, s in enumerate(states):
            s["rng"] = st[i].rng
            s["energy"] = st[i].energy.as_dict()
            s["locate"] = keep[2 * i][:st[i].nmols].copy()
            s["reservoir"] = keep[2 * i + 1][:st[i].nres].copy()
        if not record:
            return None
        return dict(kind=kind, accepted=acc.astype(bool), nmols=nm, energy=en, rng=rr)

    def nvt_run_batch(self, boxes, rngs, nsteps, energies, species=0, record=True):
        """cass_nvt_run_device_batch: nsteps NVT moves in every box at once,
        one workgroup per box, each box on its own generator (rngs[i], updated
        in place) from its energy dict energies[i]; returns one record dict
        per box as Box.nvt_run does."""
        n = len(boxes)
        energies = list(energies)
        _at_least(n, rngs=rngs, energies=energies)
        ids = np.ascontiguousarray([b.id for b in boxes], dtype=np.int32)
        opts = (abi.CassNvtOptions * n)()
        rng_arr = (abi.CassRng * n)()
        ens = _energies_in(energies)
        recs = _NvtRecords(n, nsteps)
        linear = {}     # per species object: boxes of one system share theirs
        for k, (b, r) in enumerate(zip(boxes, rngs)):
            sp = b.system.species[species]
            if id(sp) not in linear:
                linear[id(sp)] = int(sp.linear)
            opts[k] = abi.CassNvtOptions(b.params_prob_translate(), b.system.max_disp, b.system.max_rot_radians(),
                                         linear[id(sp)], species)
            rng_arr[k] = r
        self._chk(self.lib.cass_nvt_run_device_batch(self.h, n, _p(ids, C.c_int32), rng_arr, opts, nsteps, ens,
                                                     recs.table if record else None), "cass_nvt_run_device_batch")
        finals = _energies_out(ens)
        for k in range(n):
            C.memmove(C.addressof(rngs[k]), C.addressof(rng_arr[k]), C.sizeof(abi.CassRng))
        return [recs.result(k, finals[k]) for k in range(n)]

    def regrow_run(self, boxes, species, locates, rngs, nsteps, energies, first_slot=0, record=True):
        """cass_regrow_run_device: nsteps Cut_N_Grow regrowth moves of
        `species` in every box at once, one workgroup per box, box i's
        molecules first_slot + locates[i][im], on its own generator (rngs[i],
        updated in place) from its energy dict energies[i]; returns one
        record dict per box as nvt_run_batch does."""
        n = len(boxes)
        locates, energies = list(locates), list(energies)
        _at_least(n, locates=locates, rngs=rngs, energies=energies)
        bx = (abi.CassRegrowBox * n)()
        rng_arr = (abi.CassRng * n)()
        ens = _energies_in(energies)
        recs = _NvtRecords(n, nsteps)
        keep = []
        for k, (b, loc, r) in enumerate(zip(boxes, locates, rngs)):
            loc = np.ascontiguousarray(loc, dtype=np.int32)
            keep.append(loc)
            bx[k] = abi.CassRegrowBox(b.id, species, first_slot, len(loc), _p(loc, C.c_int32))
            rng_arr[k] = r
        self._chk(self.lib.cass_regrow_run_device(self.h, n, bx, rng_arr, nsteps, ens, recs.table if record else None),
                  "cass_regrow_run_device")
        finals = _energies_out(ens)
        for k in range(n):
            C.memmove(C.addressof(rngs[k]), C.addressof(rng_arr[k]), C.sizeof(abi.CassRng))
        return [recs.result(k, finals[k]) for k in range(n)]

    def total_energy_batch(self, boxes, intra=True):
        """cass_total_energy_batch: total energies of several boxes in one set
        of launches; a list of energy dicts (None for a box with an overlap)."""
        ids = np.ascontiguousarray([b.id if hasattr(b, "id") else int(b) for b in boxes], dtype=np.int32)
        n = len(ids)
        out = (abi.CassEnergy * max(1, n))()
        ov = np.zeros(max(1, n), dtype=np.int32)
        self._chk(self.lib.cass_total_energy_batch(self.h, n, _p(ids, C.c_int32), int(intra), out,
                                                   _p(ov, C.c_int32)), "cass_total_energy_batch")
        return [None if ov[k] else out[k].as_dict() for k in range(n)]

    def add_box(self, system: S.System, max_mols=None, fold=True, live=None):
        """cass_box_create + cass_box_upload of a System (coordinates folded
        into the central box as the reference's start-up does, main.f90:367-376);
        live overrides the live flags of the molecule slots (dead slots hold
        molecules a GCMC move or a Widom insertion may fill)."""
        p = derive(system)
        spec, live0, xyz = abi.box_arrays(system)
        live = live0 if live is None else np.ascontiguousarray(live, dtype=np.int32)
        # the start-up charge-neutrality check (main.f90:300-330)
        q = C.c_double()
        rc = self.lib.cass_net_charge(C.byref(p), C.byref(self.topo.c), len(spec), _p(spec, C.c_int32),
                                      _p(live, C.c_int32), C.byref(q))
        if rc:
            raise CassError(rc, f"box carries a net charge of {q.value!r} e with Ewald/DSF sums")
        cap = max(int(max_mols or 0), len(spec), 1)
        bid = C.c_int32()
        self._chk(self.lib.cass_box_create(self.h, C.byref(p), cap, C.byref(bid)), "cass_box_create")
        box = Box(self, bid.value, system, p)
        self.boxes.append(box)
        if fold:
            xyz = box.fold(spec, xyz)
        box.upload(spec, live, xyz)
        return box


class Box:
    def __init__(self, eng: Engine, bid, system, params):
        self.eng, self.id, self.system, self.params = eng, bid, system, params
        self.lib = eng.lib

    # ---------------------------------------------------------------- state
    def fold(self, spec, xyz):
        """Fold_Molecule for every molecule of a cubic box (COM into the box)."""
        if self.system.box_shape != "cubic":
            return xyz
        xyz = xyz.copy()
        L = np.array(self.system.box)
        k = 0
        for s in spec:
            sp = self.system.species[s]
            n = sp.natoms
            sites = xyz[3 * k:3 * (k + n)].reshape(n, 3)
            com = S.com_of(sp, sites)
            for d in range(3):
                if com[d] > 0.5 * L[d]:
                    sites[:, d] -= L[d]
                elif com[d] < -0.5 * L[d]:
                    sites[:, d] += L[d]
            xyz[3 * k:3 * (k + n)] = sites.ravel()
            k += n
        return xyz

    def upload(self, spec, live, xyz, com=None, max_dcom=None):
        self.spec = np.ascontiguousarray(spec, dtype=np.int32)
        self.live = np.ascontiguousarray(live, dtype=np.int32)
        self.nmols = len(spec)
        xyz = np.ascontiguousarray(xyz, dtype=np.float64)
        self.nsites = xyz.size // 3
        self.eng._chk(self.lib.cass_box_upload(self.eng.h, self.id, self.nmols, _p(self.spec, C.c_int32),
                                               _p(self.live, C.c_int32), _p(xyz), _p(com), _p(max_dcom)),
                      "cass_box_upload")

    def set_geometry(self, system: S.System):
        """cass_box_set_params from a System of the new cell (a volume move's
        rescaled box), then the upload of its folded coordinates; Ewald boxes
        regenerate their k vectors.  Returns the new k-vector count or None."""
        p = derive(system)
        self.eng._chk(self.lib.cass_box_set_params(self.eng.h, self.id, C.byref(p)), "cass_box_set_params")
        self.system, self.params = system, p
        spec, live, xyz = abi.box_arrays(system)
        self.upload(spec, live, self.fold(spec, xyz))
        return self.ewald_setup() if system.charge_style == "ewald" else None

    def load_frame(self, cell, nmols, coords):
        """One frame of a pregenerated trajectory (Read_H_frame and
        Set_Frame_Coords, load_next_frame.f90:170-330) into this box: the
        cell from the frame's H matrix (cubic or orthogonal), the molecules
        folded into it, k vectors regenerated for Ewald."""
        import dataclasses
        cell = np.asarray(cell, dtype=np.float64)
        if np.any(np.abs(cell - np.diag(np.diag(cell))) > 0.0):
            raise ValueError("frames with a non-orthogonal cell are not supported")
        L = np.diag(cell).copy()
        shape = "cubic" if L[0] == L[1] == L[2] else "orthogonal"
        s2 = dataclasses.replace(self.system, box=L, box_shape=shape, nmols=list(nmols),
                                 coords=[np.asarray(c, dtype=np.float64) for c in coords])
        return self.set_geometry(s2)

    def download(self):
        out = np.zeros(3 * self.nsites)
        self.eng._chk(self.lib.cass_box_download(self.eng.h, self.id, _p(out)), "cass_box_download")
        return out

    def mol_update(self, mol, xyz, live=True, com=None, max_dcom=None):
        xyz = np.ascontiguousarray(xyz, dtype=np.float64)
        c = None if com is None else np.ascontiguousarray(com, dtype=np.float64)
        d = None if max_dcom is None else np.array([max_dcom], dtype=np.float64)
        self.eng._chk(self.lib.cass_mol_update(self.eng.h, self.id, mol, int(live), _p(xyz), _p(c), _p(d)),
                      "cass_mol_update")

    # ------------------------------------------------------------- energies
    def compute_molecule_nonbond_inter_energy(self, mol, cbmc=False, xyz=None):
        ev, eq, ov = C.c_double(), C.c_double(), C.c_int32()
        x = None if xyz is None else np.ascontiguousarray(xyz, dtype=np.float64)
        self.eng._chk(self.lib.cass_mol_inter_energy(self.eng.h, self.id, mol, int(cbmc), _p(x), None, None,
                                                     C.byref(ev), C.byref(eq), C.byref(ov)),
                      "cass_mol_inter_energy")
        return ev.value, eq.value, bool(ov.value)

    def compute_molecule_nonbond_intra_energy(self, species, xyz, cbmc=False):
        a, b, c, ov = C.c_double(), C.c_double(), C.c_double(), C.c_int32()
        x = np.ascontiguousarray(xyz, dtype=np.float64)
        self.eng._chk(self.lib.cass_mol_intra_energy(self.eng.h, self.id, species, int(cbmc), _p(x), C.byref(a),
                                                     C.byref(b), C.byref(c), C.byref(ov)),
                      "cass_mol_intra_energy")
        return a.value, b.value, c.value, bool(ov.value)

    def set_energy_table(self, res=1000, rcut_cbmcsq_max=0.0):
        """The `energy_table` keyword: CBMC trials score molecule pairs from a
        table of res bins (Create_Atompair_Nrg_table,
        atompair_nrg_table_routines.f90:149-261); res=0 removes it."""
        self.eng._chk(self.lib.cass_set_energy_table(self.eng.h, self.id, int(res), float(rcut_cbmcsq_max)),
                      "cass_set_energy_table")

    def rminsq_table(self, u_max_base):
        """Type-pair core radii^2 of calc_rmin (create_nonbond_table.f90:285-301,
        398-417), ntypes x ntypes."""
        nt = self.eng.topo.ntypes
        out = np.zeros(nt * nt)
        self.eng._chk(self.lib.cass_rminsq_table(self.eng.h, self.id, float(u_max_base), _p(out)),
                      "cass_rminsq_table")
        return out.reshape(nt, nt)

    def widom_set_rminsq(self, rminsq):
        """The type-pair overlap pre-screen of the Widom batch (check_overlap,
        sector_routines.f90:160-233); None turns it off."""
        if rminsq is None:
            ptr = None
        else:
            self._rminsq = np.ascontiguousarray(rminsq, dtype=np.float64).ravel()
            ptr = _p(self._rminsq)
        self.eng._chk(self.lib.cass_widom_set_rminsq(self.eng.h, self.id, ptr), "cass_widom_set_rminsq")

    def trial_energies(self, species, trial_xyz, cbmc=False, exclude=-1):
        t = np.ascontiguousarray(trial_xyz, dtype=np.float64)
        n = t.shape[0]
        nrg = np.zeros(n)
        ov = np.zeros(n, dtype=np.int32)
        self.eng._chk(self.lib.cass_trial_energies(self.eng.h, self.id, species, n, _p(t), int(cbmc), exclude,
                                                   _p(nrg), _p(ov, C.c_int32)), "cass_trial_energies")
        return nrg, ov.astype(bool)

    def compute_system_total_energy(self, intra=True):
        e = abi.CassEnergy()
        ov = C.c_int32()
        self.eng._chk(self.lib.cass_total_energy(self.eng.h, self.id, int(intra), C.byref(e), C.byref(ov)),
                      "cass_total_energy")
        if ov.value:
            raise CassError(6, "overlap in the configuration")
        return e.as_dict()

    def lrc(self, nbeads):
        nb = np.ascontiguousarray(nbeads, dtype=np.float64)
        out = C.c_double()
        self.eng._chk(self.lib.cass_lrc(self.eng.h, self.id, _p(nb), C.byref(out)), "cass_lrc")
        return out.value

    def molecule_self_energy(self, species):
        out = C.c_double()
        self.eng._chk(self.lib.cass_mol_self_energy(self.eng.h, self.id, species, C.byref(out)),
                      "cass_mol_self_energy")
        return out.value

    # ----------------------------------------------------------------- Ewald
    def ewald_setup(self):
        n = C.c_int32()
        self.eng._chk(self.lib.cass_ewald_setup(self.eng.h, self.id, C.byref(n)), "cass_ewald_setup")
        return n.value

    def ewald_full(self):
        e = C.c_double()
        self.eng._chk(self.lib.cass_ewald_full(self.eng.h, self.id, C.byref(e)), "cass_ewald_full")
        return e.value

    def ewald_move(self, mol, flag, xyz=None):
        e, de = C.c_double(), C.c_double()
        x = None if xyz is None else np.ascontiguousarray(xyz, dtype=np.float64)
        self.eng._chk(self.lib.cass_ewald_move(self.eng.h, self.id, mol, flag, _p(x), C.byref(e), C.byref(de)),
                      "cass_ewald_move")
        return e.value, de.value

    def ewald_commit(self):
        self.eng._chk(self.lib.cass_ewald_commit(self.eng.h, self.id), "cass_ewald_commit")

    def ewald_revert(self):
        self.eng._chk(self.lib.cass_ewald_revert(self.eng.h, self.id), "cass_ewald_revert")

    def ewald_widom(self, species, trial_xyz):
        t = np.ascontiguousarray(trial_xyz, dtype=np.float64)
        out = np.zeros(t.shape[0])
        self.eng._chk(self.lib.cass_ewald_widom(self.eng.h, self.id, species, t.shape[0], _p(t), _p(out)),
                      "cass_ewald_widom")
        return out

    # ----------------------------------------------------------------- Widom
    def widom_set_template(self, species, xyz):
        x = np.ascontiguousarray(xyz, dtype=np.float64)
        e = C.c_double()
        self.eng._chk(self.lib.cass_widom_set_template(self.eng.h, self.id, species, _p(x), C.byref(e)),
                      "cass_widom_set_template")
        return e.value

    def widom_batch(self, species, n_ins, seed, keep=False):
        r = abi.CassWidomResult()
        wv = np.zeros(n_ins) if keep else None
        self.eng._chk(self.lib.cass_widom_batch(self.eng.h, self.id, species, n_ins, seed, _p(wv), C.byref(r)),
                      "cass_widom_batch")
        return r, wv

    def widom_emax(self, species, n=None, seed=0, xyz=None, rsq_min=False):
        """cass_widom_emax: a rigid Widom batch (n insertions from seed, or the
        placements xyz) with est_emax's per-insertion outputs.  Returns
        (widom_var, eij_max, overlap, result[, rsq_min (n, sites, natoms)])."""
        x = None if xyz is None else np.ascontiguousarray(xyz, dtype=np.float64)
        n = x.shape[0] if x is not None else n
        res = abi.CassWidomResult()
        wv, em = np.zeros(n), np.zeros(n)
        ov = np.zeros(n, dtype=np.uint8)
        rsq = None
        if rsq_min:
            rsq = np.zeros((n, len(self.eng.topo.atom_charge), self.system.species[species].natoms))
        self.eng._chk(self.lib.cass_widom_emax(self.eng.h, self.id, species, n, seed, _p(x), _p(wv), _p(em),
                                               ov.ctypes.data_as(C.POINTER(C.c_uint8)), _p(rsq), C.byref(res)),
                      "cass_widom_emax")
        out = (wv, em, ov.astype(bool), res)
        return out + (rsq,) if rsq_min else out

    def widom_placements(self, species, xyz):
        x = np.ascontiguousarray(xyz, dtype=np.float64)
        n = x.shape[0]
        wv = np.zeros(n)
        eo = np.zeros((n, 4))
        r = abi.CassWidomResult()
        self.eng._chk(self.lib.cass_widom_placements(self.eng.h, self.id, species, n, _p(x), _p(wv), _p(eo),
                                                     C.byref(r)), "cass_widom_placements")
        return r, wv, eo

    # ------------------------------------------------------------------- NVT
    def nvt_run(self, rng: abi.CassRng, nsteps, energy: dict, species=0, record=True, device=False):
        """nsteps NVT moves.  device=False: the host-driven loop (one set of
        energy launches per move); device=True: the device-resident chain
        (cass_nvt_run_device), the same draws and arithmetic in one workgroup."""
        sp = self.system.species[species]
        opt = abi.CassNvtOptions(self.params_prob_translate(), self.system.max_disp, self.system.max_rot_radians(),
                                 int(sp.linear), species)
        e = abi.CassEnergy(**{k: energy.get(k, 0.0) for k in abi.ENERGY_FIELDS})
        kind = np.zeros(nsteps, dtype=np.uint8)
        acc = np.zeros(nsteps, dtype=np.uint8)
        et = np.zeros(nsteps)
        lp = np.zeros(nsteps)
        rs = np.zeros(5 * nsteps, dtype=np.int64)
        rec = abi.CassNvtRecord(_p(kind, C.c_uint8), _p(acc, C.c_uint8), _p(et), _p(rs, C.c_int64), _p(lp))
        fn = self.lib.cass_nvt_run_device if device else self.lib.cass_nvt_run
        self.eng._chk(fn(self.eng.h, self.id, C.byref(rng), C.byref(opt), nsteps, C.byref(e),
                         C.byref(rec) if record else None), "cass_nvt_run_device" if device else "cass_nvt_run")
        return dict(kind=kind, accepted=acc.astype(bool), energy=et, ln_pacc=lp, rng=rs.reshape(-1, 5),
                    final=e.as_dict())

    def widom_cbmc(self, species, n_ins, rng: abi.CassRng = None, seed=0, n_sub=0, per_insertion=False):
        """cass_widom_cbmc_batch: n_ins CBMC insertions of a grown species.
        rng (a CassRng, advanced in place): the reference's single stream,
        insertions in sequence; None: per-insertion streams from seed, all in
        parallel.  Returns (widom_sum, n_overlaps, sub-interval sums,
        per-insertion widom_var or None)."""
        res = abi.CassWidomResult()
        sub = np.zeros(max(n_sub, 1))
        wv = np.zeros(n_ins) if per_insertion else None
        self.eng._chk(self.lib.cass_widom_cbmc_batch(self.eng.h, self.id, species, n_ins,
                                                     C.byref(rng) if rng is not None else None, seed, n_sub,
                                                     _p(sub), _p(wv), C.byref(res)), "cass_widom_cbmc_batch")
        return res.widom_sum, res.n_overlaps, sub[:n_sub], wv

    def widom_cbmc_emax(self, species, n_ins, rng=None, seed=0, rsq_min=False):
        """cass_widom_cbmc_emax: the insertions of widom_cbmc with est_emax's
        per-insertion outputs.  Returns (widom_var, eij_max, overlap) arrays
        and the CassWidomResult; with rsq_min also the closest r^2 per
        (species site, inserted atom), shape (n_ins, sites, natoms)."""
        res = abi.CassWidomResult()
        wv = np.zeros(n_ins)
        em = np.zeros(n_ins)
        ov = np.zeros(n_ins, dtype=np.uint8)
        rsq = None
        if rsq_min:
            rsq = np.zeros((n_ins, len(self.eng.topo.atom_charge), self.system.species[species].natoms))
        self.eng._chk(self.lib.cass_widom_cbmc_emax(self.eng.h, self.id, species, n_ins,
                                                    C.byref(rng) if rng is not None else None, seed, _p(wv),
                                                    _p(em), ov.ctypes.data_as(C.POINTER(C.c_uint8)),
                                                    _p(rsq) if rsq is not None else None, C.byref(res)),
                      "cass_widom_cbmc_emax")
        if rsq_min:
            return wv, em, ov.astype(bool), res, rsq
        return wv, em, ov.astype(bool), res

    def params_prob_translate(self):
        return self.system.prob_translate

    # --------------------------------------------------------------- adjoint
    def adjoint(self):
        """cass_adjoint: (E_nonbonded, dE/d eps_t, dE/d sigma_t, dE/d q_kind, forces[nsites,3])."""
        nt = self.eng.topo.ntypes
        nk = len(self.eng.topo.atom_charge)
        e = C.c_double()
        de = np.zeros(nt)
        ds = np.zeros(nt)
        dq = np.zeros(nk)
        f = np.zeros(3 * self.nsites)
        self.eng._chk(self.lib.cass_adjoint(self.eng.h, self.id, C.byref(e), _p(de), _p(ds), _p(dq), _p(f)),
                      "cass_adjoint")
        return e.value, de, ds, dq, f.reshape(-1, 3)

    def adjoint_set_frames(self, frames):
        """cass_adjoint_set_frames: frames (nframes, nsites, 3) or
        (nframes, 3 * nsites) stored in device memory."""
        x = np.ascontiguousarray(frames, dtype=np.float64).reshape(-1, 3 * self.nsites)
        self.eng._chk(self.lib.cass_adjoint_set_frames(self.eng.h, self.id, x.shape[0], _p(x)),
                      "cass_adjoint_set_frames")
        self._nframes = x.shape[0]

    def adjoint_frames(self, first=0, count=None, forces=False):
        """cass_adjoint_frames: per frame (energy[F], dE/d eps [F, nt],
        dE/d sigma [F, nt], dE/d q [F, nk], forces [F, nsites, 3] or None)."""
        if count is None:
            count = self._nframes - first
        nt = self.eng.topo.ntypes
        nk = len(self.eng.topo.atom_charge)
        e = np.zeros(count)
        de = np.zeros((count, nt))
        ds = np.zeros((count, nt))
        dq = np.zeros((count, nk))
        f = np.zeros((count, self.nsites, 3)) if forces else None
        self.eng._chk(self.lib.cass_adjoint_frames(self.eng.h, self.id, first, count, _p(e), _p(de), _p(ds), _p(dq),
                                                   _p(f) if forces else None), "cass_adjoint_frames")
        return e, de, ds, dq, f


class TrialPlan:
    """cass_trial_plan: trial sets of several boxes in one launch, optionally
    replayed from a captured hipGraph."""

    def __init__(self, eng: Engine, boxes, species, ntrial, exclude=None, cbmc=True):
        self.eng = eng
        n = len(boxes)
        self.boxes = np.ascontiguousarray([b.id if isinstance(b, Box) else b for b in boxes], dtype=np.int32)
        self.species = np.ascontiguousarray(species, dtype=np.int32)
        self.ntrial = np.ascontiguousarray(ntrial, dtype=np.int32)
        self.exclude = np.ascontiguousarray(exclude if exclude is not None else [-1] * n, dtype=np.int32)
        h = C.c_void_p()
        eng._chk(eng.lib.cass_trial_plan_create(eng.h, n, _p(self.boxes, C.c_int32), _p(self.species, C.c_int32),
                                                _p(self.ntrial, C.c_int32), _p(self.exclude, C.c_int32), int(cbmc),
                                                C.byref(h)), "cass_trial_plan_create")
        self.h = h
        self.total = int(self.ntrial.sum())

    def run(self, xyz, graph=True):
        x = np.ascontiguousarray(xyz, dtype=np.float64)
        nrg = np.zeros(self.total)
        ov = np.zeros(self.total, dtype=np.int32)
        self.eng._chk(self.eng.lib.cass_trial_plan_run(self.h, _p(x), int(graph), _p(nrg), _p(ov, C.c_int32)),
                      "cass_trial_plan_run")
        return nrg, ov.astype(bool)

    def update(self, species=None, exclude=None):
        s = None if species is None else np.ascontiguousarray(species, dtype=np.int32)
        x = None if exclude is None else np.ascontiguousarray(exclude, dtype=np.int32)
        self.eng._chk(self.eng.lib.cass_trial_plan_update(self.h, _p(s, C.c_int32), _p(x, C.c_int32)),
                      "cass_trial_plan_update")

    def autotune(self, xyz):
        x = np.ascontiguousarray(xyz, dtype=np.float64)
        blk = C.c_int32()
        self.eng._chk(self.eng.lib.cass_trial_plan_autotune(self.h, _p(x), C.byref(blk)), "cass_trial_plan_autotune")
        return blk.value

    def close(self):
        if getattr(self, "h", None):
            if getattr(self.eng, "h", None):
                self.eng.lib.cass_trial_plan_destroy(self.h)
            self.h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


def rng(i1, i3) -> abi.CassRng:
    """init_seeds (random_generators.f90:51-90) with one thread."""
    r = abi.CassRng()
    load_library().cass_rng_init(C.byref(r), i1, i3)
    return r


def startup_draws(species) -> int:
    """The rranf() draws the reference makes while it reads the MCF files,
    before init_seeds: for every fragment bond, Fragment_Order grows the
    fragments on each side of the bond (input_routines.f90:3040-3070), one
    draw per fragment added (fragment_growth.f90:1413)."""
    n = 0
    for sp in species:
        fb = list(sp.fragment_bonds or [])
        for f1, f2 in fb:
            for start, blocked in ((f1, f2), (f2, f1)):
                seen, stack = {start, blocked}, [start]
                while stack:
                    f = stack.pop()
                    for a, b in fb:
                        for x, y in ((a, b), (b, a)):
                            if x == f and y not in seen:
                                seen.add(y)
                                stack.append(y)
                                n += 1
    return n


def startup_rng(i1, i3, species) -> abi.CassRng:
    """The generator state the reference holds when its first move starts:
    the module defaults advanced by the start-up draws of startup_draws(),
    then init_seeds, which replaces only s1 and s3 (random_generators.f90:42-90)."""
    lib = load_library()
    r = abi.CassRng()
    lib.cass_rng_init(C.byref(r), 153587801, 1288503317)   # the module's default state
    for _ in range(startup_draws(species)):
        lib.cass_rng_int(C.byref(r))
    seeded = rng(i1, i3)
    r.s[0], r.s[2] = seeded.s[0], seeded.s[2]
    return r


class EmaxHistogram:
    """est_emax's running totals of one species in one box (the reference's
    w_max, Eij_w_sum, Eij_freq_total and Eij_factor, widom_insert.f90), fed
    one frame of insertions at a time through cass_emax_frame; estimate()
    is Estimate_Pair_Emax (pair_emax_estimation.f90:41-77)."""

    def __init__(self, beta, ub=2047):
        self.lib = load_library()
        self.ub = ub
        self.beta = beta
        self.factor = C.c_double(2.0 * beta)     # 0.5 kT bins (input_routines.f90:5683)
        self.w_max = np.zeros(ub + 1)
        self.w_sum = np.zeros(ub + 1)
        self.freq = np.zeros(ub + 1, dtype=np.int64)

    def add_frame(self, widom_var, eij_max, overlap, prefactor):
        wv = np.ascontiguousarray(widom_var, dtype=np.float64)
        em = np.ascontiguousarray(eij_max, dtype=np.float64)
        ov = np.ascontiguousarray(overlap, dtype=np.uint8)
        rc = self.lib.cass_emax_frame(self.ub, C.byref(self.factor), _p(self.w_max), _p(self.w_sum),
                                      self.freq.ctypes.data_as(C.POINTER(C.c_int64)), len(wv), _p(wv), _p(em),
                                      ov.ctypes.data_as(C.POINTER(C.c_uint8)), prefactor)
        if rc:
            raise RuntimeError(f"cass_emax_frame: status {rc}")

    def estimate(self, widom_sum):
        """(U*_max in kT, skipped insertions, weight fraction per bin)."""
        em = C.c_double()
        ns = C.c_int64()
        wf = np.zeros(self.ub + 1)
        rc = self.lib.cass_emax_estimate(self.ub, self.factor.value, _p(self.w_sum),
                                         self.freq.ctypes.data_as(C.POINTER(C.c_int64)), widom_sum, self.beta,
                                         C.byref(em), C.byref(ns), _p(wf))
        if rc:
            raise RuntimeError(f"cass_emax_estimate: status {rc}")
        return em.value, ns.value, wf


class RminsqHistogram:
    """est_atompair_rminsq's running totals of one species in one box (the
    reference's rsqmin_atompair_w_max / _w_sum / _freq, [solvent site]
    [inserted atom][bin]), fed one frame at a time through
    cass_rminsq_frame; estimate() is Estimate_Pair_rminsq
    (pair_emax_estimation.f90:79-168) at one tolerance."""

    def __init__(self, rows, nsolute, res, step, rcut_lowsq):
        self.lib = load_library()
        self.rows = np.ascontiguousarray(rows, dtype=np.int32)
        self.nsolv, self.nsolute, self.res = len(self.rows), nsolute, res
        self.step, self.rcut_lowsq = step, rcut_lowsq
        shape = (self.nsolv, nsolute, res)
        self.w_max = np.zeros(shape)
        self.w_sum = np.zeros(shape)
        self.freq = np.zeros(shape, dtype=np.int64)

    def add_frame(self, widom_var, rsq_min, overlap, prefactor):
        wv = np.ascontiguousarray(widom_var, dtype=np.float64)
        rm = np.ascontiguousarray(rsq_min, dtype=np.float64)
        ov = np.ascontiguousarray(overlap, dtype=np.uint8)
        rc = self.lib.cass_rminsq_frame(self.nsolv, _p(self.rows, C.c_int32), self.nsolute, rm.shape[1], self.res,
                                        self.step, self.rcut_lowsq, _p(self.w_max), _p(self.w_sum),
                                        self.freq.ctypes.data_as(C.POINTER(C.c_int64)), len(wv), _p(wv), _p(rm),
                                        ov.ctypes.data_as(C.POINTER(C.c_uint8)), prefactor)
        if rc:
            raise RuntimeError(f"cass_rminsq_frame: status {rc}")

    def estimate(self, widom_sum, tol):
        """(index table [solvent site][inserted atom], skips, widom_var bound)."""
        ind = np.zeros((self.nsolv, self.nsolute), dtype=np.int32)
        ns = C.c_int64()
        wm = C.c_double()
        rc = self.lib.cass_rminsq_estimate(self.nsolv, self.nsolute, self.res, _p(self.w_max), _p(self.w_sum),
                                           self.freq.ctypes.data_as(C.POINTER(C.c_int64)), widom_sum, tol,
                                           _p(ind, C.c_int32), C.byref(ns), C.byref(wm))
        if rc:
            raise RuntimeError(f"cass_rminsq_estimate: status {rc}")
        return ind, ns.value, wm.value
