"""GPU test of the external potential's site sums (Lennard-Jones and minimum-image Coulomb) and
of the two-orientations-per-transform Poisson path against the host restatements, for solvents
whose sites stand at the origin, on the molecule's axis and off it, for bricks of points that
the grid does not fill, and for boxes smaller than the cutoff.

Tolerance: rounding of sums of a few hundred terms, 1e-11 of the largest unclipped value (the
Poisson path's transforms: the 1e-9 of its own test)."""
import numpy as np
import pytest

from mdft import workloads
from mdft.constants import QFACT, Site, Solvent
from oracle import poisson_oracle as P

pytestmark = pytest.mark.gpu

SOLVENTS = {
    "one site at the origin": [(-0.5, 3.1, 0.65, (0.0, 0.0, 0.0))],
    "charges off axis": [(-0.8476, 3.166, 0.65, (0.0, 0.0, 0.0)), (0.4238, 0.0, 0.0, (0.8165, 0.0, 0.5774)),
                         (0.4238, 0.0, 0.0, (-0.8165, 0.0, 0.5774))],
    "sites on the axis": [(0.4, 2.6, 0.3, (0.0, 0.0, -0.6)), (-0.4, 3.0, 0.5, (0.0, 0.0, 0.7))],
    "all sites off axis": [(0.3, 2.4, 0.2, (0.5, 0.3, -0.4)), (-0.5, 2.9, 0.6, (-0.4, 0.6, 0.2)),
                           (0.2, 2.1, 0.1, (0.1, -0.7, 0.5)), (0.1, 0.0, 0.0, (0.6, 0.1, 0.1)),
                           (-0.1, 2.0, 0.1, (-0.6, -0.1, 0.3))],
}


@pytest.mark.parametrize("solvent", list(SOLVENTS))
@pytest.mark.parametrize("n,length,mmax", [((9, 5, 10), (7.0, 4.0, 8.0), 3), ((16, 8, 4), (12.0, 6.0, 24.0), 1),
                                           ((3, 1, 2), (5.0, 2.0, 3.0), 0), ((8, 9, 5), (26.0, 27.0, 25.0), 2)])
def test_vext_of_every_kind_of_site(solvent, n, length, mmax):
    from mdft.gpu import Engine
    w = workloads.Workload("vext", 3, n, length, mmax, 256)
    solv = Solvent("test", 2, 0.0333, [Site(*s) for s in SOLVENTS[solvent]])
    rng = np.random.default_rng(sum(n))
    for natom in (1, 5, 300):
        q = rng.normal(0, 0.4, natom)
        q[natom // 2] = 0.0
        q -= 0.3 if natom == 1 else 0.0
        eps = rng.uniform(0.2, 0.9, natom)
        eps[natom // 3] = 0.0 if natom > 1 else 0.5
        sol = workloads.Solute(rng.uniform(0, 1, (natom, 3)) * length, q, rng.uniform(2.0, 3.5, natom), eps)
        eng = Engine(n, length, mmax, 2, w.kT, w.n0, "fp64")

        class W:  # the workload with this solvent
            mmax, mrso, n, length, solvent = w.mmax, w.mrso, w.n, w.length, solv

        lj = workloads.vext_numpy(W, sol, rcut=7.0, clip=np.inf, coulomb=False)
        full = workloads.vext_numpy(W, sol, rcut=7.0, clip=np.inf, coulomb=True)
        offs = workloads.orientation_site_offsets(mmax, 2, solv)
        vq = P.vextq(n, length, sol.xyz, sol.q, offs, np.array([s.q for s in solv.sites]), QFACT)
        for kind, ref, bar in (("none", lj, 1e-11), ("direct", full, 1e-11), ("poisson", lj + vq, 1e-9)):
            print(f"[vext] {solvent}, {n} mmax={mmax}, {natom} atoms, {kind}", flush=True)
            eng.compute_vext(sol, solv, rcut=7.0, electrostatics=kind)
            got = eng.get_vext().reshape(ref.shape)
            ref = np.minimum(ref, QFACT / 2.0)
            below = ref < QFACT / 2.0
            scale = np.abs(ref[below]).max() if below.any() else 1.0
            # (next to the clip a rounding of the unclipped sum may clip it)
            err = np.where(below | (got < QFACT / 2.0), np.abs(got - ref), 0.0).max()
            assert err <= bar * max(scale, 1.0), (natom, kind, err, scale)
        eng.close()


@pytest.mark.parametrize("solvent", list(SOLVENTS))
@pytest.mark.parametrize("n,length,mmax", [((9, 5, 4), (7.0, 4.0, 3.0), 4), ((3, 9, 5), (26.0, 27.0, 25.0), 5),
                                           ((4, 3, 5), (9.0, 8.0, 7.0), 6)])
def test_vext_of_sites_at_few_places(solvent, n, length, mmax):
    """Orders at which a site on the axis has five and more orientations per place: solutes of fewer atoms than the
    table of places is made for, of as many, and of more."""
    from mdft.gpu import Engine
    w = workloads.Workload("vext", 3, n, length, mmax, 256)
    solv = Solvent("test", 2, 0.0333, [Site(*s) for s in SOLVENTS[solvent]])
    rng = np.random.default_rng(sum(n))
    eng = Engine(n, length, mmax, 2, w.kT, w.n0, "fp64")

    class W:  # the workload with this solvent
        mmax, mrso, n, length, solvent = w.mmax, w.mrso, w.n, w.length, solv

    for natom in (1, 3, 4, 20):
        sol = workloads.Solute(rng.uniform(0, 1, (natom, 3)) * length, rng.normal(0, 0.4, natom),
                               rng.uniform(2.0, 3.5, natom), rng.uniform(0.2, 0.9, natom))
        lj = workloads.vext_numpy(W, sol, rcut=7.0, clip=np.inf, coulomb=False)
        full = workloads.vext_numpy(W, sol, rcut=7.0, clip=np.inf, coulomb=True)
        offs = workloads.orientation_site_offsets(mmax, 2, solv)
        vq = P.vextq(n, length, sol.xyz, sol.q, offs, np.array([s.q for s in solv.sites]), QFACT)
        for kind, ref, bar in (("none", lj, 1e-11), ("direct", full, 1e-11), ("poisson", lj + vq, 1e-9)):
            print(f"[vext] {solvent}, {n} mmax={mmax}, {natom} atoms, {kind}", flush=True)
            eng.compute_vext(sol, solv, rcut=7.0, electrostatics=kind)
            got = eng.get_vext().reshape(ref.shape)
            ref = np.minimum(ref, QFACT / 2.0)
            below = ref < QFACT / 2.0
            scale = np.abs(ref[below]).max() if below.any() else 1.0
            err = np.where(below | (got < QFACT / 2.0), np.abs(got - ref), 0.0).max()
            assert err <= bar * max(scale, 1.0), (natom, kind, err, scale)
    eng.close()
