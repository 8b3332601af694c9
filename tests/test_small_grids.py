"""Bricks on short axes: periodic axes of 1 to 2r cells (whole-axis bricks), of 2r + 1 and more (halo bricks whose
halo repeats their own cells), open axes of any length, one and several bricks an axis."""
import numpy as np
import pytest

from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

L = pytest.importorskip("readdy_amd._lib")
from readdy_amd import Engine  # noqa: E402

POTS = [(L.POT_HARMONIC_REPULSION, a, b, [10.0, 1.0]) for a in range(3) for b in range(a, 3)]
RXS = [dict(kind=L.RX_FUSION, educts=[0, 1], products=[2], rate=9.0, educt_distance=0.9),
       dict(kind=L.RX_FISSION, educts=[2], products=[0, 1], rate=2.0, product_distance=0.8)]


def _engine(dims, pbc, radius, brick, seed=4):
    box = [d / radius * 1.0 * (1.0 + 1e-9) for d in dims]  # cells as narrow as they can be
    rng = np.random.default_rng([*dims, radius])
    n = max(20, min(600, int(3 * np.prod(box))))
    pos = (rng.random((n, 3)) - 0.5) * box
    pos[:4] = np.array(box) * [[-0.5, -0.5, -0.5], [0.4999999, 0.4999999, 0.4999999], [-0.5, 0.4999999, 0.0],
                               [0.0, -0.5, 0.4999999]]  # corners: neighbours through every boundary
    types = rng.integers(0, 3, n).astype(np.uint32)
    e = Engine(3, [1.0, 1.0, 0.5], potentials=POTS, reactions=RXS, cell_radius=radius, brick=brick, nl_cutoff=1.0)
    r = e.add_replica(box, pbc, seed=seed, max_particles=2 * n)
    e.set_particles(r, pos, types)
    return e, r, box, pos, types


@pytest.mark.parametrize("radius,dims", [(1, (1, 2, 3)), (1, (3, 3, 3)), (1, (4, 3, 5)), (1, (2, 2, 2)), (1, (5, 7, 6)),
                                         (2, (5, 5, 5)), (2, (4, 6, 5)), (3, (7, 6, 8))])
@pytest.mark.parametrize("pbc", [(1, 1, 1), (0, 1, 0)])
@pytest.mark.parametrize("brick", [(0, 0, 0), (2, 3, 2), (16, 16, 16)])
def test_forces_and_steps_on_short_axes(radius, dims, pbc, brick):
    # the reference's axes have at least one cell per cutoff; an axis shorter than that stays one cell
    if any(d < radius for d in dims):
        pytest.skip("box shorter than the cutoff")
    e, r, box, pos, types = _engine(dims, pbc, radius, brick)
    e.calculate_forces()
    f, _ = e.get_forces(r)
    o = po.System(3, box, list(pbc), diffusion=[1.0, 1.0, 0.5])
    for _, a, b, p in POTS:
        o.add_pair_potential(po.POT_HARMONIC_REPULSION, a, b, p)
    o.add_particles(pos, types.astype(np.int32), ids=np.arange(len(types)))
    o.nl_setup(1.0)
    energy = o.calculate_forces()
    f_ref = o.particles()[3][np.argsort(o.particles()[2])]
    assert np.linalg.norm(f - f_ref) <= 1e-5 * np.linalg.norm(f_ref)
    assert abs(e.energy(r) - energy) <= 1e-5 * abs(energy)
    # three fused steps against the same steps as separate actions, bit for bit
    e2, r2, *_ = _engine(dims, pbc, radius, brick)
    e.run(L.HANDLER_UA, 1e-3, 3)
    e2.calculate_forces()
    for _ in range(3):
        e2.integrate(1e-3)
        e2.update_neighbor_list()
        e2.react(L.HANDLER_UA, 1e-3)
        e2.update_neighbor_list()
        e2.calculate_forces()
    for a, b in zip(e.get_particles(r), e2.get_particles(r2)):
        assert np.array_equal(a, b)
    assert e.energy(r) == e2.energy(r2)
    assert np.array_equal(e.reaction_totals(r), e2.reaction_totals(r2))
    e.close()
    e2.close()


def _walled(n_types, radius, seed=8, **kw):
    """two cells on the periodic axis (the general walk), open axes with a fifth of the particles beyond their walls"""
    box = [6.0, 2.0 / radius * (1.0 + 1e-9), 5.0]
    rng = np.random.default_rng(seed)
    n = 240
    pos = (rng.random((n, 3)) - 0.5) * box
    out = rng.random(n) < 0.2
    axis = rng.choice([0, 2], n)
    beyond = np.where(rng.random(n) < 0.5, -1.0, 1.0) * (0.5 * np.array(box)[axis] + 0.4 * rng.random(n))
    pos[out, axis[out]] = beyond[out]
    types = rng.integers(0, n_types, n).astype(np.uint32)
    pots = [(L.POT_HARMONIC_REPULSION, a, b, [10.0, 1.0]) for a in range(n_types) for b in range(a, n_types)]
    rxs = [dict(kind=L.RX_FUSION, educts=[a, (a + 1) % n_types], products=[(a + 2) % n_types], rate=60.0,
                educt_distance=0.9) for a in range(n_types)]
    rxs += [dict(kind=L.RX_FISSION, educts=[a], products=[a, (a + 1) % n_types], rate=20.0, product_distance=0.8)
            for a in range(n_types)]
    e = Engine(n_types, np.ones(n_types), potentials=pots, reactions=rxs, cell_radius=radius, nl_cutoff=1.0, **kw)
    r = e.add_replica(box, (0, 1, 0), seed=3, max_particles=8 * n)
    e.set_particles(r, pos, types)
    return e, r, box, pos, types, pots


@pytest.mark.parametrize("n_types", [2, 4, 5, 8, 16])
@pytest.mark.parametrize("radius", [1, 2])
def test_outside_and_dead_records_are_no_neighbours_in_the_general_walk(n_types, radius):
    """The staged species of such a record carries a flag beyond every table of the species: it is refused by that
    flag.  Forces against the oracle; separate actions and fused runs, and separate reactions right after a fused run
    (whose buffer holds the withdrawn copies), against the bin-reading path."""
    e, r, box, pos, types, pots = _walled(n_types, radius)
    s, q, *_ = _walled(n_types, radius, lds_states=1)
    o = po.System(n_types, box, [0, 1, 0], diffusion=[1.0] * n_types)
    for _, a, b, p in pots:
        o.add_pair_potential(po.POT_HARMONIC_REPULSION, a, b, p)
    o.add_particles(pos, types.astype(np.int32), ids=np.arange(len(types)))
    o.nl_setup(1.0)
    energy = o.calculate_forces()
    f_ref = o.particles()[3][np.argsort(o.particles()[2])]
    for x, i in ((e, r), (s, q)):
        x.calculate_forces()
        f = x.get_forces(i)[0]
        assert np.linalg.norm(f - f_ref) <= 1e-5 * np.linalg.norm(f_ref)
        assert abs(x.energy(i) - energy) <= 1e-5 * abs(energy)

    def same():
        for a, b in zip((*e.get_particles(r), e.energy(r)), (*s.get_particles(q), s.energy(q))):
            assert np.array_equal(a, b)
        assert np.array_equal(e.get_forces(r)[0], s.get_forces(q)[0])
        assert np.array_equal(e.reaction_totals(r), s.reaction_totals(q))

    for rounds in range(3):
        for x in (e, s):
            x.run(L.HANDLER_UA, 2e-3, 2 + rounds)
            x.react(L.HANDLER_UA, 2e-3)
            x.update_neighbor_list()
            x.calculate_forces()
        same()
        for x in (e, s):
            x.integrate(1e-3)
            x.update_neighbor_list()
            x.react(L.HANDLER_GILLESPIE, 2e-3)
            x.calculate_forces()
        same()
    assert e.reaction_totals(r).sum() > 0
    e.close()
    s.close()
