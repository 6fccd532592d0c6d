"""Device GEMC particle transfers (cbmc_grow.h::k_gemc_chain) against the
reference's own run and the oracle.

* The reference's 2000-transfer pentane GEMC run between a 28 A box of 60
  molecules and a 40 A box of 20 (tests/golden/pentane_gemc_gemc.npz,
  written by the reference's GEMC_Particle_Transfer through oracle/ref_probe
  in gemc mode): every decision, both boxes' molecule counts and the
  generator state bit for bit, both running total energies within 1e-10, in
  two launches whose state carries over; then each box's energy against a
  fresh recompute and against the reference's recomputed end energies.
* The mixed mode along the same run: the same decisions up to a first one
  near its threshold, energies within 1e-8.
* Four pairs of uneven boxes in one launch against the oracle, pair by
  pair."""
import numpy as np
import pytest

from cassandra_amd import engine as E
from tests import pentane_cases as P

REL = 1e-10


def _setup(prec, boxes, cb, st, fx):
    system0 = boxes[0][0]
    eng = E.Engine(system0, max_boxes=2, precision=prec)
    bx = [eng.add_box(system, live=live) for system, live in boxes]
    eng.set_cbmc_species(0, cb)
    sp = system0.species[0]
    rng = E.startup_rng(int(fx["seed"][0]), int(fx["seed"][1]), [sp])
    specs = [dict(box=b.id, species=0, first_slot=0, max_mols=st["cap"], prob_insert=0.0, mu=0.0, de_broglie=1.0)
             for b in bx]
    states = [dict(rng=rng if k == 0 else E.startup_rng(1, 2, [sp]), energy=dict(st["energies"][k]),
                   locate=st["locate"][k].copy(), reservoir=st["reservoir"][k].copy()) for k in range(2)]
    return eng, bx, specs, states


@pytest.mark.gpu
def test_gemc_device_chain_replays_reference():
    print("[gpu] device GEMC chain vs the reference, FP64", flush=True)
    fx, boxes, cb, st = P.gemc_case()
    eng, bx, specs, states = _setup(E.FP64, boxes, cb, st, fx)
    n = int(fx["nsteps"])
    o1 = eng.gemc_run(specs, states, n // 2)
    assert np.array_equal(list(states[1]["rng"].s), list(states[0]["rng"].s))
    o2 = eng.gemc_run(specs, states, n - n // 2)
    acc = np.concatenate([o1["accepted"][0], o2["accepted"][0]])
    assert np.array_equal(acc, fx["accept"])
    for b in range(2):
        assert np.array_equal(np.concatenate([o1["accepted"][b], o2["accepted"][b]]), fx["accept"])
        nm = np.concatenate([o1["nmols"][b], o2["nmols"][b]])
        assert np.array_equal(nm, fx["nmols"][:, b])
        en = np.concatenate([o1["energy"][b], o2["energy"][b]])
        assert np.max(np.abs(en - fx["energy"][:, b]) / np.abs(fx["energy"][:, b])) < REL
        rr = np.concatenate([o1["rng"][b], o2["rng"][b]])
        assert np.array_equal(rr, fx["rng"])
    for b in range(2):
        e = bx[b].compute_system_total_energy()
        for k in ("total", "inter_vdw", "lrc", "angle", "dihedral", "intra_vdw"):
            assert abs(e[k] - states[b]["energy"][k]) <= 1e-9 * max(1.0, abs(e[k])), (b, k)
        ref = fx["energy_recomputed_end"][b]
        assert abs(e["total"] - ref[0]) <= 1e-10 * abs(ref[0])
        assert abs(e["inter_vdw"] - ref[3]) <= 1e-10 * abs(ref[3])
        assert len(states[b]["locate"]) == fx["nmols"][-1, b]
    eng.close()


@pytest.mark.gpu
def test_gemc_device_chain_mixed():
    """Mixed-mode pair arithmetic: the reference's decisions until a first one
    that the rounding of the pair sums can flip (reported), energies within
    1e-8 up to there."""
    print("[gpu] device GEMC chain vs the reference, mixed", flush=True)
    fx, boxes, cb, st = P.gemc_case()
    eng, bx, specs, states = _setup(E.MIXED, boxes, cb, st, fx)
    n = int(fx["nsteps"])
    out = eng.gemc_run(specs, states, n)
    diff = np.nonzero(out["accepted"][0] != fx["accept"])[0]
    m = n if not diff.size else int(diff[0])
    if m < n:
        import warnings
        warnings.warn(f"mixed GEMC chain parts from the reference at move {m}")
        assert m > 100
    for b in range(2):
        assert np.max(np.abs(out["energy"][b][:m] - fx["energy"][:m, b]) / np.abs(fx["energy"][:m, b])) < 1e-8
    eng.close()


@pytest.mark.gpu
def test_gemc_pairs_against_oracle(oracle_mod):
    """Four pairs in one launch, each pair two boxes of the fixture's set-up
    with other densities and its own generator: every pair against the
    oracle's restatement from the same start (FP64: the same decisions,
    counts and generator states, energies within 1e-10)."""
    print("[gpu] device GEMC, 4 pairs vs the oracle", flush=True)
    from cassandra_amd import systems as S
    fx, boxes, cb, st = P.gemc_case()
    sp = boxes[0][0].species[0]
    geo = S.species_pentane()  # all-trans geometry for the start configurations
    cap = st["cap"]
    pairs = []
    rs = np.random.default_rng(3)
    for p in range(4):
        L = (27.0 + 2 * p, 36.0 + 3 * p)
        nm = (50 + 5 * p, 30 - 5 * p)
        pair = []
        for b in range(2):
            c = np.zeros((cap, sp.natoms, 3))
            c[:nm[b]] = S.place_random([(geo, nm[b])], [L[b]] * 3, int(rs.integers(1 << 30)), 2.2, 3.2)[0]
            system = S.System([sp], [cap], [c], np.array([L[b]] * 3), 380.0 + 10 * p, "lj", "cut_tail", 12.0,
                              rcut_low=1.0, rcut_cbmc=6.5, name=f"gemc_pair{p}_{b}")
            live = np.zeros(cap, dtype=np.int32)
            live[:nm[b]] = 1
            pair.append((system, live, nm[b]))
        pairs.append(pair)
    eng = E.Engine(pairs[0][0][0], max_boxes=8, precision=E.FP64)
    eng.set_cbmc_species(0, cb)
    specs, states, refs = [], [], []
    nsteps = 300
    for p, pair in enumerate(pairs):
        obs, ocs, energies = [], [], []
        for system, live, nm in pair:
            box = eng.add_box(system, live=live)
            e = box.compute_system_total_energy()
            energies.append(e)
            specs.append(dict(box=box.id, species=0, first_slot=0, max_mols=cap, prob_insert=0.0, mu=0.0,
                              de_broglie=1.0))
            ob = oracle_mod.OracleBox(system, live=live)
            obs.append(ob)
            ocs.append(oracle_mod.OracleCbmc(ob, 0, cb))
        seed = E.startup_rng(1000 + p, 77 + p, [sp])
        s = np.array(list(seed.s), dtype=np.int64)
        loc = [np.arange(nm) for _, _, nm in pair]
        res = [np.arange(cap - 1, nm - 1, -1) for _, _, nm in pair]
        for k in range(2):
            states.append(dict(rng=E.startup_rng(1000 + p, 77 + p, [sp]), energy=dict(energies[k]),
                               locate=loc[k].copy(), reservoir=res[k].copy()))
        refs.append(oracle_mod.gemc(ocs, s, nsteps, [0, 0], [len(x) for x in loc], loc, res, energies))
    out = eng.gemc_run(specs, states, nsteps)
    for p, ref in enumerate(refs):
        for b in range(2):
            i = 2 * p + b
            assert np.array_equal(out["kind"][i], ref["box_out"]), (p, b)
            assert np.array_equal(out["accepted"][i], ref["accepted"]), (p, b)
            assert np.array_equal(out["nmols"][i], ref["nmols"][:, b])
            assert np.array_equal(out["rng"][i], ref["rng"])
            assert np.max(np.abs(out["energy"][i] - ref["energy"][:, b]) / np.abs(ref["energy"][:, b])) < REL
    assert sum(int(out["accepted"][2 * p].sum()) for p in range(4)) > 0
    eng.close()
