"""A batch of NVT chains over boxes of different sizes, styles and species:
each box equal bit for bit to its own run, its host mirrors equal to the
device's coordinates, one launch and several."""
import numpy as np
import pytest

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
