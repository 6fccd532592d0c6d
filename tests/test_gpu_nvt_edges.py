"""The device NVT chain against the host-driven loop where its parts change:
one and two molecules (the next move takes the molecule just moved), molecule
pairs of more than 64 site pairs, species of unlike site counts, k vectors
beyond the lanes' registers, phases without tables, orthogonal boxes, a style
without its own pair arithmetic, boxes beyond the LDS copy."""
import ctypes as C

import numpy as np
import pytest

from cassandra_amd import engine as E
from cassandra_amd import systems as S

REL = 1e-10   # the energies' tolerance against the reference


def _chain(n, q):
    """n sites on a zigzag, charges alternating (the first of an odd count 0)"""
    xyz = np.array([[1.1 * i, 0.3 * (i % 2), 0.0] for i in range(n)])
    charge = [0.0] * (n % 2) + [q if i % 2 else -q for i in range(n - n % 2)]
    atoms = [S.Atom(f"A{i % 3}", "C", 12.0 + i % 3, charge[i], 40.0 + 10.0 * (i % 3), 2.6 + 0.1 * (i % 3))
             for i in range(n)]
    return S.Species("chain", atoms, xyz)


def _lattice(sp, n, box):
    """n molecules, each along x, in cells as long as a molecule and 2.6 A"""
    x = sp.ref_coords - sp.ref_coords.mean(0)
    nx = max(1, min(int(np.ceil(n ** (1 / 3))), int(box[0] // (np.ptp(x[:, 0]) + 2.6))))
    m = int(np.ceil(np.sqrt(n / nx)))
    cell = np.stack(np.meshgrid(np.arange(nx), np.arange(m), np.arange(m), indexing="ij"), -1).reshape(-1, 3)[:n]
    box = np.array(box)
    return ((cell + 0.5) / [nx, m, m] * box - 0.5 * box)[:, None, :] + x


def _system(case):
    w = S.species_spce()
    if case == "lj2000":
        return S.config_lj2000().parsed()
    species, counts, box, rc, style = {
        "one": ([w], [1], [20.0] * 3, 9.0, "cut"),   # (Ewald: its energy changes are rounding alone)
        "two": ([w], [2], [20.0] * 3, 9.0, "ewald"),
        "dsf": ([w], [40], [20.0] * 3, 9.0, "dsf"),
        "orthogonal": ([w], [70], [19.0, 24.0, 21.5], 9.0, "ewald"),
        "many_k": ([w], [30], [44.0] * 3, 9.0, "ewald"),
        "mixture": ([w, S.species_methane(), _chain(11, 0.2)], [33, 20, 4], [24.0] * 3, 9.0, "ewald"),
        "sites9": ([_chain(9, 0.15)], [25], [30.0] * 3, 10.0, "ewald"),
        "sites64": ([_chain(64, 0.1)], [2], [76.0] * 3, 9.0, "ewald"),
        # the copy and the waves' buffers take 156.6 kB of the 159.7 for 2000
        # one-site molecules and 161.7 for 2080; 164.9 for 1130 waters with the
        # phase powers, 156.0 without; 180.9 for 80 of 64 sites; the phase
        # powers alone 140 for 40 sites
        "memory": ([S.species_lj()], [2080], [46.0] * 3, 9.0, "none"),
        "memory_k": ([w], [1130], [32.3] * 3, 9.0, "ewald"),
        "memory_dsf": ([w], [1400], [36.0] * 3, 9.0, "dsf"),
        "memory_orthogonal": ([w], [1130], [30.0, 34.0, 33.0], 9.0, "ewald"),
        "memory_sites64": ([_chain(64, 0.1)], [80], [110.0] * 3, 10.0, "cut"),
        "memory_sites40": ([_chain(40, 0.1)], [150], [90.0] * 3, 20.0, "ewald"),
    }[case]
    coords = ([_lattice(species[0], counts[0], box)] if case.startswith("memory") else
              S.place_random(list(zip(species, counts)), box, 5, 1.2, 2.6))
    return S.System(species, counts, coords, np.array(box), 350.0, "lj", "cut_tail", rc, charge_style=style,
                    rcut_coul=rc, alpha_dsf=0.2 if style == "dsf" else None, rcut_low=0.85,
                    box_shape="orthogonal" if case.endswith("orthogonal") else "cubic", max_disp=0.4,
                    # (a site's own rotation changes its energy by rounding alone)
                    prob_translate=1.0 if species[0].natoms == 1 else 0.5, max_rot=25.0, seed=(101, 203), name=case).parsed()


@pytest.mark.gpu
@pytest.mark.parametrize("prec", [E.FP64, E.MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("case", ["one", "two", "dsf", "orthogonal", "many_k", "mixture", "sites9", "sites64", "lj2000",
                                  "memory", "memory_k", "memory_dsf", "memory_orthogonal", "memory_sites64",
                                  "memory_sites40"])
def test_nvt_chain_equals_host_loop(case, prec):
    print(f"[gpu] nvt chain edges {case} {prec}", flush=True)
    system, steps = _system(case), 120
    got = []
    for device in (True, False):
        eng = E.Engine(system, precision=E.FP64 if not device else prec)
        box = eng.add_box(system)
        if system.charge_style == "ewald":
            box.ewald_setup()
        e0 = box.compute_system_total_energy()
        rng = E.rng(*system.seed)
        out = box.nvt_run(rng, steps, e0, device=device)
        got.append((out, list(rng.s), box.download(), box.compute_system_total_energy()))
        eng.close()
    (a, ra, xa, ta), (b, rb, xb, _) = got
    tol = REL if prec == E.FP64 else 1e-8   # the mixed chain's tolerance in the replay of the reference
    for k in ("kind", "accepted", "rng"):
        assert np.array_equal(a[k], b[k]), k
    assert ra == rb
    assert np.max(np.abs(a["energy"] - b["energy"]) / np.maximum(np.abs(b["energy"]), 1.0)) < tol
    assert np.array_equal(np.isnan(a["ln_pacc"]), np.isnan(b["ln_pacc"]))
    assert np.max(np.abs(xa - xb)) < 1e-9
    # the running sums of the chain against a fresh evaluation of its end state
    assert abs(a["final"]["total"] - ta["total"]) <= tol * max(1.0, abs(ta["total"]))


@pytest.mark.gpu
def test_nvt_batch_over_all_paths():
    """a box copied to LDS, one in device memory and one for the host loop in
    one batch, each as in a run of its own"""
    print("[gpu] nvt batch over all paths", flush=True)
    sp, steps = S.species_lj(), 40
    systems = [S.System([sp], [n], [_lattice(sp, n, [L] * 3)], np.array([L] * 3), 150.0, "lj", "cut_tail", 9.0,
                        rcut_low=0.85, prob_translate=1.0, max_disp=0.4, seed=(7, 9 + n), name="lj").parsed()
               for n, L in ((100, 22.0), (40000, 130.0), (2400, 50.0))]

    def run(batch):
        eng = E.Engine(systems[0], max_boxes=3, precision=E.FP64)
        boxes = [eng.add_box(s) for s in systems]
        e0 = eng.total_energy_batch(boxes)
        rngs = [E.rng(*s.seed) for s in systems]
        if batch:
            out = eng.nvt_run_batch(boxes, rngs, steps, e0)
        else:
            out = [b.nvt_run(r, steps, e, device=True) for b, r, e in zip(boxes, rngs, e0)]
        got = [(o, b.download(), list(r.s)) for o, b, r in zip(out, boxes, rngs)]
        eng.close()
        return got

    for (a, xa, ra), (b, xb, rb) in zip(run(True), run(False)):
        for k in ("kind", "accepted", "energy", "rng"):
            assert np.array_equal(a[k], b[k]), k
        assert np.array_equal(xa, xb) and ra == rb and a["final"] == b["final"]
        assert 0 < a["accepted"].sum()


@pytest.mark.gpu
@pytest.mark.parametrize("device", [True, False])
def test_nvt_draw_of_one(device):
    """rranf rounds its largest words to 1.0 (random_generators.f90:118): a first
    word for which the third draw, the molecule's, does takes the last molecule"""
    print(f"[gpu] nvt draw of one, device={device}", flush=True)
    sp, n = S.species_lj(), 5
    system = S.System([sp], [n], [_lattice(sp, n, [22.0] * 3)], np.array([22.0] * 3), 150.0, "lj", "cut_tail", 9.0,
                      rcut_low=0.85, prob_translate=1.0, max_disp=0.4, name="lj").parsed()
    eng = E.Engine(system, precision=E.FP64)
    box = eng.add_box(system)
    rng = E.rng(101, 203)
    rng.s[0] = 4707937272820449914
    probe = E.rng(101, 203)
    probe.s[0] = rng.s[0]
    assert [eng.lib.cass_rng_uniform(C.byref(probe)) for _ in range(3)][2] == 1.0
    before = box.download().reshape(n, 3)
    out = box.nvt_run(rng, 1, box.compute_system_total_energy(), device=device)
    assert out["accepted"][0]
    moved = np.any(box.download().reshape(n, 3) != before, axis=1)
    assert list(np.flatnonzero(moved)) == [n - 1]
    eng.close()
