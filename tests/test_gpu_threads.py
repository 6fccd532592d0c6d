"""Two engines on two threads whose chains share a kernel at unlike LDS sizes:
each gives what it gives alone."""
import threading

import numpy as np
import pytest

from cassandra_amd import cbmc
from cassandra_amd import engine as E
from cassandra_amd import systems as S


def _lattice(sp, n, L):
    m = int(np.ceil(n ** (1 / 3)))
    cell = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    return ((cell + 0.5) * (L / m) - 0.5 * L)[:, None, :] + sp.ref_coords - sp.ref_coords.mean(0)


def _nvt(n, calls):
    w, L = S.species_spce(), (n / 512) ** (1 / 3) * 24.83
    L = max(L, 19.0)
    system = S.System([w], [n], [_lattice(w, n, L)], np.array([L] * 3), 300.0, "lj", "cut_tail", 9.0, charge_style="cut",
                      rcut_coul=9.0, rcut_low=0.5, prob_translate=0.5, max_disp=0.2, seed=(n, n + 1), name="t").parsed()
    eng = E.Engine(system, precision=E.FP64)
    box = eng.add_box(system)
    state = [box.compute_system_total_energy()]
    rng = E.rng(*system.seed)

    def run():
        out = []
        for _ in range(calls):
            r = box.nvt_run(rng, 10, state[0], device=True)
            state[0] = r["final"]
            out.append(r["energy"])
        eng.close()
        return np.concatenate(out)
    return run


def _gcmc(cap, calls):
    sp, n, L = cbmc.pentane_frag_species(S.species_pentane()), 20, 30.0
    coords = np.zeros((cap, sp.natoms, 3))
    coords[:n] = S.place_random_grid([(sp, n)], [L] * 3, 5, 2.2, 3.0)[0]
    system = S.System([sp], [cap], [coords], np.array([L] * 3), 420.0, "lj", "cut_tail", 13.0, rcut_low=1.0,
                      rcut_cbmc=6.5, seed=(cap, 8), name="t")
    eng = E.Engine(system, precision=E.FP64)
    eng.set_cbmc_species(0, cbmc.pentane_growth(420.0, 4, 4, seed=1)[1])
    box = eng.add_box(system, live=(np.arange(cap) < n).astype(np.int32))
    lam = cbmc.de_broglie(sp, 420.0)
    mu = S.KBOLTZ * 420.0 * (np.log(n / L ** 3 * lam ** 3) - 1.0)
    spec = dict(box=box.id, species=0, first_slot=0, max_mols=cap, prob_insert=0.5, mu=mu, de_broglie=lam)
    state = dict(rng=E.startup_rng(cap, 8, [sp]), energy=box.compute_system_total_energy(), locate=np.arange(n),
                 reservoir=np.arange(cap - 1, n - 1, -1))
    eng.gcmc_run([spec], [state], 1)

    def run():
        out = [eng.gcmc_run([spec], [state], 5)["energy"][0] for _ in range(calls)]
        eng.close()
        return np.concatenate(out)
    return run


@pytest.mark.gpu
@pytest.mark.parametrize("make,small,large,calls", [(_nvt, 30, 1100, 60), (_gcmc, 60, 1900, 60)], ids=["nvt", "gcmc"])
def test_two_engines_on_two_threads(make, small, large, calls):
    print(f"[gpu] two threads {make.__name__}", flush=True)
    alone = [make(k, calls)() for k in (small, large)]
    runs, got = [make(k, calls) for k in (small, large)], [None, None]

    def work(k):
        got[k] = runs[k]()

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for a, b in zip(alone, got):
        assert b is not None and np.array_equal(a, b)
