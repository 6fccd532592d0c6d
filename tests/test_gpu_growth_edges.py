"""The growth kernels at the edges of their ranges, against the oracle: one
and the most trials a stage takes, live lists about a wave's 64 lanes and
beyond the LDS, pair styles off the LJ kernels, and molecules many images away."""
import dataclasses

import numpy as np
import pytest

from cassandra_amd import abi, cbmc
from cassandra_amd import engine as E
from cassandra_amd import systems as S

# FP64: the same pairs summed in another order, some 1e4 terms of alternating
# sign (1e4 * 2^-53 = 1e-12 of the largest) in energies that add up over moves
REL = 1e-10

CASES = [
    # molecules, slots, kappa_ins, kappa_dih, vdW sum style
    (2, 8, 1, 1, "cut_tail"),
    (63, 70, 12, 24, "cut_tail"),
    (65, 130, 32, 32, "cut_shift"),
    (64, 2100, 3, 5, "cut"),          # the live list in device memory
    (40, 60, 32, 31, "cut_switch"),   # not an LJ-kernel style
    (30, 50, 7, 9, "charmm"),
]


def _box(n, cap, style, seed):
    sp = cbmc.pentane_frag_species(S.species_pentane())
    L = 30.0
    coords = np.zeros((cap, sp.natoms, 3))
    coords[:n] = S.place_random_grid([(sp, n)], [L] * 3, seed, 2.2, 3.0)[0]
    system = S.System([sp], [cap], [coords], np.array([L] * 3), 420.0, "lj", style, 13.0, charge_style="none",
                      rcut_low=1.0, rcut_cbmc=6.5, ron_switch=11.0, roff_switch=13.0, seed=(seed, 2 * seed + 1),
                      name="edge")
    return sp, system, (np.arange(cap) < n).astype(np.int32)


def _rel(a, b):
    return float(np.max(np.abs(a - b) / np.maximum(np.abs(b), 1.0)))


@pytest.mark.gpu
@pytest.mark.parametrize("n,cap,ki,kd,style", CASES)
def test_growth_chains_at_edges(n, cap, ki, kd, style, oracle_mod):
    print(f"[gpu] growth edges n={n} cap={cap} kappa={ki}/{kd} {style}", flush=True)
    sp, system, live = _box(n, cap, style, 1000 + n)
    _, growth = cbmc.pentane_growth(420.0, ki, kd, seed=n)
    nsteps = 25
    lam = cbmc.de_broglie(sp, 420.0)
    mu = S.KBOLTZ * 420.0 * (np.log(n / 30.0 ** 3 * lam ** 3) - 1.0)

    def start():
        eng = E.Engine(system, precision=E.FP64)
        eng.set_cbmc_species(0, growth)
        box = eng.add_box(system, live=live)
        oc = oracle_mod.OracleCbmc(oracle_mod.OracleBox(system, live=live), 0, growth)
        return eng, box, oc, box.compute_system_total_energy(), E.startup_rng(*system.seed, [sp])

    # insertions and deletions
    eng, box, oc, e0, r = start()
    loc, res = np.arange(n), np.arange(cap - 1, n - 1, -1)
    ref = oc.gcmc(np.array(list(r.s), dtype=np.int64), nsteps, 0, cap, 0.5, mu, lam, n, loc.copy(), res.copy(),
                  dict(e0))
    state = dict(rng=r, energy=e0, locate=loc, reservoir=res)
    out = eng.gcmc_run([dict(box=box.id, species=0, first_slot=0, max_mols=cap, prob_insert=0.5, mu=mu,
                             de_broglie=lam)], [state], nsteps)
    for k in ("kind", "accepted", "nmols", "rng"):
        assert np.array_equal(out[k][0], ref[k]), k
    assert _rel(out["energy"][0], ref["energy"]) < REL
    eng.close()
    # regrowth
    eng, box, oc, e0, r = start()
    s = np.array(list(r.s), dtype=np.int64)
    ref = oc.regrow(s, nsteps, 0, np.arange(n), dict(e0))
    out = eng.regrow_run([box], 0, [np.arange(n)], [r], nsteps, [e0])[0]
    assert np.array_equal(out["accepted"], ref["accepted"])
    assert np.array_equal(out["rng"], ref["rng"])
    assert _rel(out["energy"], ref["energy"]) < REL
    # parallel Widom insertions into the box as the chain left it
    wv = box.widom_cbmc(0, 300, seed=9, per_insertion=True)[3]
    system2 = dataclasses.replace(system, coords=[box.download().reshape(cap, sp.natoms, 3)])
    oc2 = oracle_mod.OracleCbmc(oracle_mod.OracleBox(system2, live=live), 0, growth)
    ref, _ = oc2.widom_streams(9, 300)
    ok = ref > 0
    assert np.array_equal(wv > 0, ok)
    assert np.all(np.abs(wv[ok] - ref[ok]) <= REL * 10 * ref[ok])  # a weight is exp(-beta dE): |beta dE| to some tens
    eng.close()


@pytest.mark.gpu
def test_growth_many_images_away(oracle_mod):
    """One-site molecules whose coordinates stand 8000 box lengths off (those of a
    non-cubic box are never folded): each pair within the cutoff counts, also
    the last hundredth of an angstrom, which single precision cannot tell there."""
    print("[gpu] growth many images away", flush=True)
    ch4 = S.species_methane()
    ch4.fragments = [[0]]
    box, n = np.array([24.0, 27.0, 25.0]), 400
    rng = np.random.default_rng(4)
    cell = np.stack(np.meshgrid(*[np.arange(8)] * 3, indexing="ij"), -1).reshape(-1, 3)[rng.permutation(512)[:n]]
    xyz = (cell + 0.5 + rng.uniform(-0.1, 0.1, (n, 3))) / 8 * box - box / 2 + box * [8000.0, -9000.0, 7000.0]
    system = S.System([ch4], [n + 1], [np.concatenate([xyz, np.zeros((1, 3))])[:, None, :]], box, 300.0, "lj", "cut",
                      9.0, rcut_low=1.0, rcut_cbmc=6.5, box_shape="orthogonal", seed=(3, 5), name="far")
    live = (np.arange(n + 1) < n).astype(np.int32)
    growth = abi.CbmcSpecies(ch4, [np.zeros((1, 1, 3))], kappa_ins=8)
    eng = E.Engine(system, precision=E.FP64)
    eng.set_cbmc_species(0, growth)
    b = eng.add_box(system, live=live)
    wv = b.widom_cbmc(0, 1500, seed=11, per_insertion=True)[3]
    ref, _ = oracle_mod.OracleCbmc(oracle_mod.OracleBox(system, live=live), 0, growth).widom_streams(11, 1500)
    ok = ref > 0
    assert ok.sum() > 500 and np.array_equal(wv > 0, ok)
    # the separations carry the rounding of coordinates of 2e5 (2e5 * 2^-53 = 2e-11),
    # r^-12 of them 1e-10 of a term, exp(-beta dE) at |beta dE| of some tens 1e-8
    assert np.all(np.abs(wv[ok] - ref[ok]) <= 1e-7 * ref[ok])
    eng.close()
