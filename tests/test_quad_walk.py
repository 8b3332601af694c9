"""The walk of quads on the matrix cores against the bin-reading path (every brick outgrows a staging of one record)
and the oracle: rows of cells of 0 to 9 records, rows longer than a wave, more quads than one round of a block,
halos of more than 1024 cells, overflowed bins, stencils of radius 2 and 3, draw lists that fill up, particles at and
beyond the boundary of an open box, a cutoff whose pairs lie within rounding of it."""
import numpy as np
import pytest

from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

L = pytest.importorskip("readdy_amd._lib")
from readdy_amd import Engine  # noqa: E402

POTS = [(L.POT_HARMONIC_REPULSION, a, b, [10.0, 1.0]) for a in range(3) for b in range(a, 3)]


def _rows(rng):
    """z-rows of 0 to 9 records in one cell's width, side by side"""
    return np.concatenate([np.stack([np.full(k, i % 7 - 3.0), np.full(k, i // 7 - 3.0), rng.uniform(-1.4, 1.4, k)], 1)
                           for i, k in enumerate(rng.integers(0, 10, 49))]), 8.0


def _long_rows(rng):
    """two rows of 150 and 90 records, the quads of the first more than a wave's sixteen"""
    z = np.linspace(-3.9, 3.9, 150)
    return np.concatenate([np.stack([0.1 + 0 * z, 0 * z, z], 1), np.stack([0 * z[:90], 0.6 + 0 * z[:90], z[:90]], 1)]), 8.0


def _clump(rng):
    """900 records in a few cells (rounds of 64 quads), a thin gas around them"""
    return np.concatenate([rng.uniform(-1.6, 1.6, (900, 3)), rng.uniform(-3.9, 3.9, (60, 3))]), 8.0


def _lattice(rng):
    """pairs at the cutoff to within a few units in the last place"""
    g = np.stack(np.meshgrid(*[np.arange(-4, 4) * 1.0] * 3, indexing="ij"), -1).reshape(-1, 3)
    return g + rng.integers(-2, 3, g.shape) * 2.0 ** -52, 8.0


def _gas(rng):
    return rng.uniform(-7.0, 7.0, (1500, 3)), 14.0


FILLS = dict(rows=_rows, long_rows=_long_rows, clump=_clump, lattice=_lattice, gas=_gas)


def _engine(fill, pbc, rate, **kw):
    rng = np.random.default_rng(11)
    pos, box = FILLS[fill](rng)
    types = rng.integers(0, 3, len(pos)).astype(np.uint32)
    rxs = [dict(kind=L.RX_FUSION, educts=[0, 1], products=[2], rate=rate, educt_distance=0.9),
           dict(kind=L.RX_ENZYMATIC, educts=[2, 0], products=[2, 1], rate=rate, educt_distance=1.0),
           dict(kind=L.RX_CONVERSION, educts=[1], products=[0], rate=rate),
           dict(kind=L.RX_FISSION, educts=[2], products=[0, 1], rate=rate, product_distance=0.8)]
    e = Engine(3, [1.0, 1.0, 0.5], potentials=POTS, reactions=rxs, nl_cutoff=1.0, events_per_replica=200000, **kw)
    r = e.add_replica([box] * 3, pbc, seed=6, max_particles=4 * len(pos))
    e.set_particles(r, pos, types)
    return e, r, box, pos, types


@pytest.mark.parametrize("fill", FILLS)
@pytest.mark.parametrize("kw", [dict(), dict(bin_capacity=2), dict(brick=(8, 8, 8)), dict(brick=(1, 1, 2)),
                                dict(cell_radius=2), dict(cell_radius=3, brick=(6, 6, 7))],
                         ids=lambda k: "-".join(map(str, k)) or "default")
@pytest.mark.parametrize("pbc,rate", [((1, 1, 1), 40.0), ((0, 1, 0), 0.5)])
def test_quads_equal_the_bin_reading_path(fill, kw, pbc, rate):
    e, r, box, pos, types = _engine(fill, pbc, rate, **kw)
    s, rs, *_ = _engine(fill, pbc, rate, **dict(kw, lds_states=1))
    for x in (e, s):
        x.calculate_forces()
    f, _ = e.get_forces(r)
    assert np.array_equal(f, s.get_forces(rs)[0])
    o = po.System(3, [box] * 3, list(pbc), diffusion=[1.0, 1.0, 0.5])
    for _, a, b, p in POTS:
        o.add_pair_potential(po.POT_HARMONIC_REPULSION, a, b, p)
    o.add_particles(pos, types.astype(np.int32), ids=np.arange(len(types)))
    o.nl_setup(1.0)
    energy = o.calculate_forces()
    f_ref = o.particles()[3][np.argsort(o.particles()[2])]
    # FP32 pair terms: at most 4 units of 2^-24 of |k| (sigma - d) <= 10 a term, up to 100 terms a particle
    assert np.abs(f - f_ref).max() <= 100 * 10 * 4 * 2.0 ** -24
    assert abs(e.energy(r) - energy) <= 1e-5 * abs(energy) + 1e-5
    for n in (1, 3):
        for x in (e, s):
            x.run(L.HANDLER_UA, 2e-3, n)
        for a, b in zip(e.get_particles(r), s.get_particles(rs)):
            assert np.array_equal(a, b)
        assert e.energy(r) == s.energy(rs)
        assert np.array_equal(e.reaction_totals(r), s.reaction_totals(rs))
    assert e.reaction_totals(r).sum() > 0
    e.close()
    s.close()


def test_the_brick_shape_follows_the_particles():
    """The same replica filled with 40 and with 4000 particles in turn: each as in an engine of its own."""
    rng = np.random.default_rng(3)
    e, r, box, _, _ = _engine("gas", (1, 1, 1), 5.0)
    for n in (40, 4000, 600):
        pos, types = rng.uniform(-7.0, 7.0, (n, 3)), rng.integers(0, 3, n).astype(np.uint32)
        alone, ra, *_ = _engine("gas", (1, 1, 1), 5.0, brick=(3, 3, 3))
        for x, i in ((e, r), (alone, ra)):
            x.set_particles(i, pos, types)
            x.calculate_forces()
        assert np.array_equal(e.get_forces(r)[0], alone.get_forces(ra)[0])
        assert e.energy(r) == alone.energy(ra)
        alone.close()
    e.close()


@pytest.mark.parametrize("steps", [300, 600])
@pytest.mark.parametrize("graph", [False, True])
def test_the_brick_shape_follows_growth_within_a_run(steps, graph):
    """125 particles that multiply to thousands in one run: the bricks are fitted on the way (after 256 steps or 512),
    and the run goes on in them as in bricks of a given shape."""
    out = []
    for kw in (dict(), dict(brick=(3, 3, 3))):
        rxs = [dict(kind=L.RX_FISSION, educts=[0], products=[0, 0], rate=5.5, product_distance=0.5)]
        e = Engine(1, [0.5], potentials=[(L.POT_HARMONIC_REPULSION, 0, 0, [0.1, 1.0])], reactions=rxs, nl_cutoff=1.0,
                   bin_capacity=64, **kw)
        r = e.add_replica([5.0] * 3, (1, 1, 1), seed=2, max_particles=20000)
        pos = np.random.default_rng(1).uniform(-2.5, 2.5, (125, 3))
        e.set_particles(r, pos, np.zeros(125, np.uint32))
        e.calculate_forces()
        before = e.brick_shape()
        e.run(L.HANDLER_UA, 2e-3 * 300 / steps, steps, graph=graph)
        assert kw or e.brick_shape() != before  # (a fit that is due at the end of a run waits for the next launch)
        out.append((*e.get_particles(r), e.energy(r), e.reaction_totals(r)))
        e.close()
    assert len(out[0][0]) > 2000
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("kw", [dict(), dict(lds_states=1), dict(n_types=20)],
                         ids=["staged", "bin-reading", "more types than are staged"])
@pytest.mark.parametrize("graph", [False, True])
def test_a_replica_without_a_handler_reacts_in_no_launch(kw, graph):
    """Its own handler NONE holds in a launch with reactions, on the bin-reading path too: no reactions, and the
    trajectory of a launch without any; its neighbour in the launch reacts."""
    rng = np.random.default_rng(5)
    rxs = [dict(kind=L.RX_FUSION, educts=[0, 1], products=[2], rate=40.0, educt_distance=0.9),
           dict(kind=L.RX_CONVERSION, educts=[1], products=[0], rate=40.0)]
    nt = kw.get("n_types", 3)
    kw = {k: v for k, v in kw.items() if k != "n_types"}
    n, steps = 400, 41
    e, quiet = (Engine(nt, np.ones(nt), potentials=POTS, reactions=rxs, nl_cutoff=1.0, max_replicas=2, **kw)
                for _ in range(2))
    ids = []
    for k in range(2):
        pos, types = rng.uniform(-4.0, 4.0, (n, 3)), rng.integers(0, 3, n).astype(np.uint32)
        for x in (e, quiet):
            r = x.add_replica([8.0] * 3, seed=k, max_particles=2 * n)
            x.set_particles(r, pos, types)
        ids.append(r)
    e.set_handler(ids[0], L.HANDLER_NONE)
    e.run(L.HANDLER_UA, 1e-3, steps, graph=graph)
    quiet.run(L.HANDLER_NONE, 1e-3, steps)
    assert e.reaction_totals(ids[0]).sum() == 0 and e.reaction_totals(ids[1]).sum() > 0
    for a, b in zip(e.get_particles(ids[0]), quiet.get_particles(ids[0])):
        assert np.array_equal(a, b)
    for x in (e, quiet):
        x.close()


@pytest.mark.parametrize("cutoff", [1e9, 3e18, 1e20])
def test_a_cutoff_far_beyond_the_box(cutoff):
    """Every pair of an open box interacts; records outside it, and the padding of a quad's last step, stay out."""
    rng = np.random.default_rng(2)
    box = 9.0
    g = np.stack(np.meshgrid(*[np.arange(-3, 3) * 1.4 + 0.7] * 3, indexing="ij"), -1).reshape(-1, 3)
    pos = g + rng.uniform(-0.15, 0.15, g.shape)
    pos[::17, 0] += box  # beyond the wall
    lj = [12, 6, cutoff, 0.0, 1.0, 1.0]
    e = Engine(1, [1.0], potentials=[(L.POT_LENNARD_JONES, 0, 0, lj)])
    r = e.add_replica([box] * 3, (0, 0, 0), max_particles=len(pos))
    e.set_particles(r, pos, np.zeros(len(pos), np.uint32))
    e.calculate_forces()
    f, _ = e.get_forces(r)
    o = po.System(1, [box] * 3, [0, 0, 0], diffusion=[1.0])
    o.add_pair_potential(po.POT_LENNARD_JONES, 0, 0, lj)
    o.add_particles(pos, np.zeros(len(pos), np.int32), ids=np.arange(len(pos)))
    o.nl_setup(cutoff)
    energy = o.calculate_forces()
    f_ref = o.particles()[3][np.argsort(o.particles()[2])]
    assert np.linalg.norm(f - f_ref) <= 1e-5 * np.linalg.norm(f_ref)
    assert abs(e.energy(r) - energy) <= 1e-5 * abs(energy)
    assert not f[::17].any()
    for _ in range(2):
        e.run(L.HANDLER_NONE, 1e-5, 3)
    assert np.isfinite(e.get_particles(r)[0]).all()
    e.close()


def _gas_engine(replicas=1):
    e = Engine(1, [0.5], potentials=POTS[:1], nl_cutoff=1.0, max_replicas=replicas)
    return e, [e.add_replica([20.0] * 3, seed=k, max_particles=4000) for k in range(replicas)]


def _fill(e, r, clump):
    rng = np.random.default_rng(7)
    pos = rng.uniform(-9.9, 9.9, (2000, 3))
    if clump:
        pos[:1500] = rng.normal(scale=1.2, size=(1500, 3))
    e.set_particles(r, pos, np.zeros(2000, np.uint32))
    e.calculate_forces()


def test_the_brick_shape_does_not_depend_on_what_the_engine_held():
    """A clump raises the occupancy that the bricks are made for; a gas uploaded over it, or left alone with the
    engine, has the bricks of an engine that never held a clump."""
    e, (r,) = _gas_engine()
    _fill(e, r, False)
    gas = e.brick_shape()
    _fill(e, r, True)
    clump = e.brick_shape()
    assert clump != gas
    _fill(e, r, False)
    assert e.brick_shape() == gas
    e.close()

    e, (a, b) = _gas_engine(2)
    _fill(e, a, False)
    one = e.brick_shape()
    _fill(e, b, True)
    both = e.brick_shape()
    assert both != one
    _fill(e, a, False)  # the clump stays, and so do its bricks
    assert e.brick_shape() == both
    e.remove_replica(b)
    e.calculate_forces()
    assert e.brick_shape() == one
    e.close()


def test_records_that_no_bricks_stage_do_not_shrink_the_others():
    """8000 of 24000 particles in 27 cells, more than a block's LDS holds around any of them: the rest keeps the bricks
    of a gas of as many particles, in every later call too."""
    rng = np.random.default_rng(4)
    shapes = []
    for clump in (0, 8000):
        e = Engine(1, [0.0], potentials=[(L.POT_HARMONIC_REPULSION, 0, 0, [1e-3, 1.0])], nl_cutoff=1.0, bin_capacity=480)
        r = e.add_replica([40.0] * 3, max_particles=24000)
        pos = rng.uniform(-20.0, 20.0, (24000, 3))
        pos[:clump] = rng.uniform(0.0, 3.0, (clump, 3))
        e.set_particles(r, pos, np.zeros(24000, np.uint32))
        for _ in range(3):
            e.calculate_forces()
            shapes.append(e.brick_shape())
        e.close()
    assert len(set(shapes)) == 1
