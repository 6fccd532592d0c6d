"""A batch of NVT chains over boxes of different sizes, styles and species:
each box equal bit for bit to its own run, its host mirrors equal to the
device's coordinates, one launch and several.  A batch whose staging cannot be
had leaves its boxes as they were; records of any length need no more than the
bounded staging."""
import ctypes as C

import numpy as np
import pytest

from cassandra_amd import cbmc
from cassandra_amd import engine as E
from cassandra_amd import systems as S


def _systems():
    out = []
    for k, (n, L) in enumerate(((3, 20.0), (64, 22.0), (65, 23.0))):
        sp = S.species_spce()
        coords = S.place_random([(sp, n)], [L] * 3, 40 + k, 1.2, 2.6)
        out.append(S.System([sp], [n], coords, np.array([L] * 3), 300.0, "lj", "cut_tail", 9.0,
                            charge_style="ewald" if k != 1 else "cut", rcut_coul=9.0, rcut_low=0.85,
                            prob_translate=0.5, max_disp=0.3, seed=(11 + k, 23 + k), name=f"w{n}").parsed())
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("steps", [1, 37, 4099])   # 4096 moves a launch
def test_nvt_batch_of_unlike_boxes(steps):
    print(f"[gpu] nvt batch of unlike boxes, {steps} steps", flush=True)
    systems = _systems()

    def run(batch):
        eng = E.Engine(systems[0], max_boxes=len(systems), precision=E.FP64)
        boxes = [eng.add_box(s) for s in systems]
        for b, s in zip(boxes, systems):
            if s.charge_style == "ewald":
                b.ewald_setup()
        e0 = [b.compute_system_total_energy() for b in boxes]
        rngs = [E.rng(*s.seed) for s in systems]
        if batch:
            out = eng.nvt_run_batch(boxes, rngs, steps, e0)
        else:
            out = [b.nvt_run(r, steps, e, device=True) for b, r, e in zip(boxes, rngs, e0)]
        for b, s in zip(boxes, systems):
            xyz = b.download().reshape(-1, 3, 3)
            for m in (0, b.nmols - 1):   # the stored molecule against the device's own coordinates
                assert b.compute_molecule_nonbond_inter_energy(m) == \
                    b.compute_molecule_nonbond_inter_energy(m, xyz=xyz[m])
        got = [(o, b.download(), list(r.s)) for o, b, r in zip(out, boxes, rngs)]
        eng.close()
        return got

    for (a, xa, ra), (b, xb, rb) in zip(run(True), run(False)):
        for k in ("kind", "accepted", "energy", "rng"):
            assert np.array_equal(a[k], b[k]), k
        assert np.array_equal(xa, xb) and ra == rb and a["final"] == b["final"]
    eng = E.Engine(systems[0])
    assert eng.nvt_run_batch([], [], 5, []) == []
    eng.close()


def _pinned_limit():
    lim = E.load_library().cass_test_pinned_limit
    lim.argtypes, lim.restype = [C.c_void_p, C.c_size_t], None
    return lim


def _pentanes(n, cap):
    sp = cbmc.pentane_frag_species(S.species_pentane())
    coords = np.zeros((cap, sp.natoms, 3))
    coords[:n] = S.place_random_grid([(sp, n)], [30.0] * 3, 5, 2.2, 3.0)[0]
    system = S.System([sp], [cap], [coords], np.array([30.0] * 3), 420.0, "lj", "cut_tail", 13.0, rcut_low=1.0,
                      rcut_cbmc=6.5, seed=(3, 8), name="staging")
    return sp, system, (np.arange(cap) < n).astype(np.int32)


@pytest.mark.gpu
@pytest.mark.parametrize("entry", ["nvt", "gcmc", "regrow"])
def test_no_staging_leaves_boxes_untouched(entry):
    print(f"[gpu] no staging, {entry}", flush=True)
    n, cap, steps = 20, 30, 25
    sp, system, live = _pentanes(n, cap)
    if entry == "nvt":
        system, live = _systems()[0], None
    lim = _pinned_limit()

    def run(fail):
        eng = E.Engine(system, precision=E.FP64)
        box = eng.add_box(system, live=live)
        if entry != "nvt":
            eng.set_cbmc_species(0, cbmc.pentane_growth(420.0, 12, 24, seed=1)[1])
        elif system.charge_style == "ewald":
            box.ewald_setup()
        e0 = box.compute_system_total_energy()
        rng = E.startup_rng(3, 8, [sp]) if entry != "nvt" else E.rng(*system.seed)
        state = dict(rng=rng, energy=e0, locate=np.arange(n), reservoir=np.arange(cap - 1, n - 1, -1))

        def call():
            if entry == "nvt":
                return eng.nvt_run_batch([box], [rng], steps, [e0])[0]
            if entry == "regrow":
                return eng.regrow_run([box], 0, [np.arange(n)], [rng], steps, [e0])[0]
            lam = cbmc.de_broglie(sp, 420.0)
            return eng.gcmc_run([dict(box=box.id, species=0, first_slot=0, max_mols=cap, prob_insert=0.5, mu=-6000.0,
                                      de_broglie=lam)], [state], steps)

        if fail:
            before, words = box.download(), list(rng.s)
            lim(eng.h, 1)
            with pytest.raises(E.CassError) as ex:
                call()
            assert ex.value.code == 3
            lim(eng.h, 1 << 40)
            assert np.array_equal(box.download(), before) and list(rng.s) == words
            assert box.compute_system_total_energy() == e0
        out = call()
        got = out["energy"], box.download(), box.compute_system_total_energy()
        eng.close()
        return got

    (ea, xa, ta), (eb, xb, tb) = run(True), run(False)
    assert np.array_equal(ea, eb) and np.array_equal(xa, xb) and ta == tb
    assert len(np.unique(ea)) > 1   # moves were accepted


@pytest.mark.gpu
@pytest.mark.parametrize("entry", ["nvt", "gcmc", "regrow"])
def test_long_records_within_bounded_staging(entry):
    """54 to 58 bytes a move and box: 18 to 19 MB in one call, past the 16 MiB that
    go through the staging; the same moves in two calls, which do."""
    print(f"[gpu] long records, {entry}", flush=True)
    nb, steps = {"nvt": (16, 20000), "gcmc": (48, 7000), "regrow": (48, 6800)}[entry]
    n, cap = 6, 12
    sp, system, live = _pentanes(n, cap)
    if entry == "nvt":
        ar = S.species_lj()
        system, live = S.System([ar], [2], S.place_random([(ar, 2)], [20.0] * 3, 3, 1.2, 2.6), np.array([20.0] * 3),
                                300.0, "lj", "cut", 9.0, rcut_low=0.85, max_disp=1.0, name="two").parsed(), None

    def run(calls):
        eng = E.Engine(system, max_boxes=nb, precision=E.FP64)
        boxes = [eng.add_box(system, live=live) for _ in range(nb)]
        if entry != "nvt":
            eng.set_cbmc_species(0, cbmc.pentane_growth(420.0, 4, 4, seed=1)[1])
        e0 = eng.total_energy_batch(boxes)
        rngs = [E.startup_rng(3 + k, 8, [sp]) if entry != "nvt" else E.rng(3 + k, 8) for k in range(nb)]
        lam = cbmc.de_broglie(sp, 420.0)
        mu = S.KBOLTZ * 420.0 * (np.log(n / 30.0 ** 3 * lam ** 3) - 1.0)
        specs = [dict(box=b.id, species=0, first_slot=0, max_mols=cap, prob_insert=0.45, mu=mu, de_broglie=lam)
                 for b in boxes]
        states = [dict(rng=r, energy=e, locate=np.arange(n), reservoir=np.arange(cap - 1, n - 1, -1))
                  for r, e in zip(rngs, e0)]
        _pinned_limit()(eng.h, 17 << 20)
        out = []
        for _ in range(calls):
            if entry == "gcmc":
                out.append(eng.gcmc_run(specs, states, steps // calls))
                continue
            r = (eng.nvt_run_batch(boxes, rngs, steps // calls, e0) if entry == "nvt" else
                 eng.regrow_run(boxes, 0, [np.arange(n)] * nb, rngs, steps // calls, e0))
            e0 = [x["final"] for x in r]
            out.append({k: np.array([x[k] for x in r]) for k in ("kind", "accepted", "energy", "ln_pacc", "rng")})
        eng.close()
        return {k: np.concatenate([o[k] for o in out], axis=1) for k in out[0]}

    one, two = run(1), run(2)
    for k in one:
        assert np.array_equal(one[k], two[k], equal_nan=one[k].dtype == np.float64), k
    assert one["rng"][:, -1].all() and 0 < one["accepted"][:, -100:].sum()


@pytest.mark.gpu
@pytest.mark.parametrize("long", [False, True])
def test_records_after_a_stop_are_zero(long):
    """A GCMC chain that runs out of free slots reports it; what it recorded
    before stands in the caller's arrays, the rest is zero, through the staging
    and past it."""
    print(f"[gpu] records after a stop, long={long}", flush=True)
    from cassandra_amd import abi
    n, cap = 6, 8
    steps = 320000 if long else 200
    sp, system, live = _pentanes(n, cap)
    eng = E.Engine(system, precision=E.FP64)
    eng.set_cbmc_species(0, cbmc.pentane_growth(420.0, 4, 4, seed=1)[1])
    box = eng.add_box(system, live=live)
    lam = cbmc.de_broglie(sp, 420.0)
    mu = S.KBOLTZ * 420.0 * (np.log(40 / 30.0 ** 3 * lam ** 3) + 2.0)   # insertions win: the slots fill
    slots = np.zeros(2 * cap, dtype=np.int32)
    slots[:n], slots[cap:cap + 2] = np.arange(n), [7, 6]
    at = slots.ctypes.data
    p32 = C.POINTER(C.c_int32)
    gb = abi.CassGcmcBox(box.id, 0, 0, cap, 0.9, mu, lam)
    st = abi.CassGcmcState()
    st.rng = E.startup_rng(3, 8, [sp])
    st.energy = abi.CassEnergy(**box.compute_system_total_energy())
    st.nmols, st.nres, st.locate, st.reservoir = n, 2, C.cast(at, p32), C.cast(at + 4 * cap, p32)
    kind, acc = np.full(steps, 9, np.uint8), np.full(steps, 9, np.uint8)
    nm, en, rr = np.full(steps, 9, np.int32), np.full(steps, 9.0), np.full(5 * steps, 9, np.int64)
    rec = abi.CassGcmcRecord(*[a.ctypes.data_as(t) for a, t in zip((kind, acc, nm, en, rr), (
        C.POINTER(C.c_uint8), C.POINTER(C.c_uint8), p32, C.POINTER(C.c_double), C.POINTER(C.c_int64)))])
    rc = eng.lib.cass_gcmc_run_device(eng.h, 1, C.byref(gb), C.byref(st), steps, C.byref(rec))
    assert rc == 6   # max_molecules reached
    done = np.flatnonzero(nm)[-1] + 1
    assert 0 < done < 200 and nm[done - 1] == cap
    assert all(np.all(a[done * k:] == 0) for a, k in ((kind, 1), (acc, 1), (nm, 1), (en, 1), (rr, 5)))
    assert np.all(rr[:5 * done].reshape(-1, 5) != 9) and np.all(nm[:done] >= n)
    eng.close()
