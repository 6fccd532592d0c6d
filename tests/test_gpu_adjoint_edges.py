"""The adjoint's reciprocal and pair kernels at their edges: n_y ranges of two,
three and four register steps and beyond, boxes of unlike edges, molecules of
one to eight sites (site groups of three), site counts around a tile, one and
many frames, molecules more than an image away.  Against the total energy and
its central differences in the coordinates, the types' parameters and the
charges."""
import numpy as np
import pytest

from cassandra_amd import engine as E
from cassandra_amd import systems as S


def _species(n):
    xyz = np.array([[1.0 * i, 0.4 * (i % 2), 0.2 * (i % 3)] for i in range(n)])
    q = [0.0] if n == 1 else [(-0.3 if i % 2 else 0.3) if i < n - n % 2 else 0.0 for i in range(n)]
    return S.Species(f"s{n}", [S.Atom(f"T{i % 2}", "C", 12.0 + i % 2, q[i], 50.0 + 20.0 * (i % 2), 2.7 + 0.2 * (i % 2))
                               for i in range(n)], xyz)


CASES = {
    # name: (sites, molecules, box, cutoff) -- n_y up to 4, 9, 13, 17
    "two_steps": (3, 21, [16.0] * 3, 7.5),
    "three_steps": (4, 16, [27.0] * 3, 11.0),
    "four_steps": (8, 8, [28.0] * 3, 8.0),
    "beyond": (2, 33, [30.0] * 3, 6.5),
    "unlike_edges": (5, 13, [18.0, 31.0, 23.0], 8.5),
    "tile": (1, 64, [24.0] * 3, 8.0),
}


@pytest.mark.gpu
@pytest.mark.parametrize("case", list(CASES))
def test_adjoint_edges(case):
    print(f"[gpu] adjoint edges {case}", flush=True)
    n, count, box, rc = CASES[case]
    sp = _species(n)
    coords = S.place_random([(sp, count)], box, 9, 1.2, 2.6)
    system = S.System([sp], [count], coords, np.array(box), 300.0, "lj", "cut_tail", rc, charge_style="ewald",
                      rcut_coul=rc, rcut_low=0.85, box_shape="cubic" if len(set(box)) == 1 else "orthogonal",
                      name=case).parsed()
    eng = E.Engine(system, precision=E.FP64)
    b = eng.add_box(system)
    b.ewald_setup()
    e0 = b.compute_system_total_energy()["total"]
    energy, deps, dsig, dq, forces = b.adjoint()
    assert abs(energy - e0) <= 1e-10 * max(1.0, abs(e0))
    # frames: the box's own coordinates and shifted ones; each equal to one alone
    xyz = b.download().reshape(-1, 3)
    rng = np.random.default_rng(3)
    h = 1e-4
    site = int(rng.integers(n * count))
    frames = [xyz]
    for d in range(3):
        for sgn in (1.0, -1.0):
            f = xyz.copy()
            f[site, d] += sgn * h
            frames.append(f)
    b.adjoint_set_frames(np.array(frames))
    ef, _, _, dqf, ff = b.adjoint_frames(0, len(frames), forces=True)
    assert ef[0] == pytest.approx(energy, rel=1e-12, abs=1e-9)
    fmax = np.max(np.abs(forces))
    assert np.max(np.abs(ff[0] - forces)) <= 1e-11 * max(1.0, fmax)
    assert np.max(np.abs(dqf[0] - dq)) <= 1e-11 * max(1.0, np.max(np.abs(dq)))
    # central differences of step h: truncation h^2 |U'''| / 6 (two powers of a
    # site distance below the force) and rounding eps |U| / h
    fd = [-(ef[1 + 2 * d] - ef[2 + 2 * d]) / (2 * h) for d in range(3)]
    tol = 50.0 * h * h * max(1.0, fmax) + 1e-15 * max(1.0, abs(e0)) * count / h
    assert np.max(np.abs(np.array(fd) - forces.reshape(-1, 3)[site])) <= tol
    # the derivatives by the parameters, as the total energy has them
    eps, sig, _, _ = system.type_tables()
    charge = np.array([a.charge for a in sp.atoms])

    def total(eps_t=None, sig_t=None, q=None):
        e = None if eps_t is None else np.sqrt(np.outer(eps_t, eps_t))
        g = None if sig_t is None else 0.5 * (sig_t[:, None] + sig_t[None, :])
        eng.set_nonbond_params(eps if e is None else e, sig if g is None else g, charge if q is None else q)
        return b.compute_system_total_energy()["total"]

    # four-point differences of relative step 1e-3.  A term of order sigma^12 is off
    # by h^4 / 30 of its fifth derivative, 12 * 11 * 10 * 9 * 8 / 30 * 1e-12 = 3e-9
    # of itself over x, one of order sqrt(eps) or q^2 by less; rounding adds eps |U|
    # / (x h), 1e-13 of it.  The derivative and U are differences of sums of such
    # terms, taken to be within 30 of |grad| + |U| / x.
    for name, grad, x in (("eps_t", deps, np.diag(eps)), ("sig_t", dsig, np.diag(sig)), ("q", dq, charge)):
        for k in range(len(x)):
            scale = max(abs(x[k]), 0.1)

            def at(steps):
                y = x.copy()
                y[k] += steps * 1e-3 * scale
                return total(**{name: y})

            fd = (8 * (at(1) - at(-1)) - (at(2) - at(-2))) / (12e-3 * scale)
            assert abs(fd - grad[k]) <= 1e-7 * (np.max(np.abs(grad)) + abs(e0) / scale), (name, k)
    eng.close()


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 3])
def test_adjoint_of_molecules_images_away(n):
    """Frames are not folded: a molecule three box lengths off is beyond the one
    image shift that the energy takes (minimum_image_separation.f90:35-112), so
    it has no neighbours there, and none in the derivatives."""
    print(f"[gpu] adjoint images away {n}", flush=True)
    sp, L = _species(n), 20.0
    coords = S.place_random([(sp, 40)], [L] * 3, 13, 1.2, 2.6)
    system = S.System([sp], [40], coords, np.array([L] * 3), 300.0, "lj", "cut", 8.0, charge_style="cut", rcut_coul=8.0,
                      rcut_low=0.85, name="away").parsed()
    eng = E.Engine(system, precision=E.FP64)
    b = eng.add_box(system)
    xyz = b.download().reshape(-1, 3)
    far = xyz.copy()
    far[5 * n:6 * n] += [3 * L, 0.0, 0.0]
    far[9 * n:10 * n] += [0.0, -3 * L, 3 * L]
    b.adjoint_set_frames(np.array([xyz, far]))
    energy, _, _, _, forces = b.adjoint_frames(0, 2, forces=True)
    for k, x in enumerate((xyz, far)):
        b.upload(b.spec, b.live, x.ravel())
        total = b.compute_system_total_energy()["total"]
        assert abs(energy[k] - total) <= 1e-10 * max(1.0, abs(total))
    assert abs(energy[0] - energy[1]) > 1.0
    intra = forces[1].reshape(40, n, 3)[[5, 9]].sum(1)   # no net force from others
    assert np.max(np.abs(intra)) <= 1e-9 * np.max(np.abs(forces[1]))
    eng.close()
