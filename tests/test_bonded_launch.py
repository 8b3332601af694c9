"""The one-launch bonded terms (k_bonded): blocks and waves that hold the terms of one replica, of several, and
partial blocks of every kind, against the oracle replica by replica."""
import numpy as np
import pytest

from oracle import pyoracle as po

from readdy_amd import workloads as W

pytestmark = pytest.mark.gpu

L = pytest.importorskip("readdy_amd._lib")
from readdy_amd import Engine  # noqa: E402


@pytest.mark.parametrize("chain_counts", [(1,), (5, 1, 3), (1,) * 40, (52, 1, 53), (7, 0, 260)])
def test_bonded_forces_and_energies_per_replica(chain_counts):
    """Chains of 6 beads: 5 bonds, 4 angles, 3 dihedrals each, so the replicas' terms meet inside waves (many
    small replicas), at their edges and at block edges (52 chains: 260 bonds).  FP64 terms in 2^-32 / 2^-24 fixed
    point: forces within 1e-9 of the oracle's, the energy within 2^-24 per term."""
    beads, box = 6, 30.0
    rng = np.random.default_rng(len(chain_counts))
    e = Engine(1, [1.0], potentials=[(L.POT_HARMONIC_REPULSION, 0, 0, [0.0, 0.5])], topology_flavor=[1],
               max_replicas=len(chain_counts))
    refs = []
    for n in chain_counts:
        r = e.add_replica([box] * 3, (1, 1, 1), seed=3, max_particles=4000)
        pos = W.chains(n, beads, box, rng) if n else np.zeros((0, 3))
        e.set_particles(r, pos, np.zeros(len(pos), np.uint32))
        o = po.System(1, [box] * 3, [1, 1, 1], diffusion=[1.0])
        o.add_particles(pos, np.zeros(len(pos), np.int32), ids=np.arange(len(pos)))
        terms = 0
        if n:
            idx = np.arange(n * beads).reshape(n, beads)
            bonds = np.stack([idx[:, :-1], idx[:, 1:]], axis=2).reshape(-1, 2)
            angles = np.stack([idx[:, :-2], idx[:, 1:-1], idx[:, 2:]], axis=2).reshape(-1, 3)
            dihedrals = np.stack([idx[:, :-3], idx[:, 1:-2], idx[:, 2:-1], idx[:, 3:]], axis=2).reshape(-1, 4)
            e.set_bonds(r, bonds, 7.0, 0.9)
            e.set_angles(r, angles, 3.0, 2.0)
            e.set_dihedrals(r, dihedrals, 1.5, 2, 0.3)
            for b in bonds:
                o.add_bond(int(b[0]), int(b[1]), 7.0, 0.9)
            for a in angles:
                o.add_angle(int(a[0]), int(a[1]), int(a[2]), 3.0, 2.0)
            for d in dihedrals:
                o.add_dihedral(int(d[0]), int(d[1]), int(d[2]), int(d[3]), 1.5, 2, 0.3)
            terms = len(bonds) + len(angles) + len(dihedrals)
        o.nl_setup(0.5)
        refs.append((r, o, o.calculate_forces(), terms))
    e.calculate_forces()
    for r, o, energy, terms in refs:
        f, h = e.get_forces(r)
        x = o.particles()
        f_ref = x[3][np.argsort(x[2])] if terms else np.zeros((0, 3))
        assert f.shape == f_ref.shape
        if terms:
            assert np.linalg.norm(f - f_ref) <= 1e-9 * np.linalg.norm(f_ref)
        assert abs(e.energy(r) - energy) <= terms * 2.0 ** -24 + 1e-12 * abs(energy)
    e.close()
