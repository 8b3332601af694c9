"""Radial distribution by bricks against the oracle, to the count: uneven, repeated, many and few borders, distances on
the borders, bricks that outgrow their staging, short bricks, walls with particles beyond them, overflowed bins, boxes
at the line to the general kernel (2 rad + 2 cells an axis)."""
import numpy as np
import pytest

from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

L = pytest.importorskip("readdy_amd._lib")
from readdy_amd import Engine  # noqa: E402

BORDERS = dict(even=np.linspace(0.0, 2.5, 26), log=np.concatenate([[0.0], np.geomspace(1e-4, 2.5, 300)]),
               shell=[0.75, 1.0, 1.0, 1.0, 1.25], one=[0.5, 2.9], most=np.linspace(0.0, 2.0, 4097),
               negative=[-1.0, 0.0, 0.5, 2.0])


def _fill(name, rng, box):
    n = int(2.0 * np.prod(box))
    pos = (rng.random((n, 3)) - 0.5) * box
    if name == "lattice":  # distances of exactly 0.25 k along the axes
        pos = np.round(pos * 4.0) / 4.0
        pos = np.unique(np.where(pos >= np.array(box) / 2, -np.array(box) / 2, pos), axis=0)
    if name == "clump":
        pos[: n // 2] *= 0.12
    if name == "walls":
        k = n // 40
        pos[:k, 1] = np.where(rng.random(k) < 0.5, -1, 1) * (box[1] / 2 + rng.random(k))
    return pos


@pytest.mark.parametrize("fill,box,pbc,kw", [
    ("gas", (10.0, 11.0, 13.0), (1, 1, 1), {}), ("lattice", (8.0, 8.0, 9.0), (1, 1, 1), {}),
    ("clump", (12.0, 12.0, 12.0), (1, 1, 1), {}), ("clump", (12.0, 12.0, 12.0), (1, 0, 1), dict(bin_capacity=3)),
    ("walls", (9.0, 10.0, 9.0), (1, 0, 1), {}), ("gas", (9.0, 9.0, 9.0), (0, 0, 0), dict(cell_radius=2)),
    ("gas", (8.0, 8.0, 8.0), (1, 1, 1), {}), ("gas", (7.0, 8.0, 8.0), (1, 1, 1), {}),
    ("gas", (5.0, 5.0, 5.0), (1, 1, 1), {})], ids=lambda v: v if isinstance(v, str) else None)
@pytest.mark.parametrize("borders", BORDERS)
def test_counts_equal_the_oracle(fill, box, pbc, kw, borders):
    rng = np.random.default_rng(17)
    pos = _fill(fill, rng, np.array(box))
    types = rng.integers(0, 3, len(pos)).astype(np.uint32)
    pots = [(L.POT_HARMONIC_REPULSION, a, b, [10.0, 1.0]) for a in range(3) for b in range(a, 3)]
    e = Engine(3, [1.0] * 3, potentials=pots, nl_cutoff=1.0, max_replicas=2, max_cells=8000, max_particles=20000, **kw)
    other = e.add_replica([6.0] * 3, (1, 1, 1), seed=2, max_particles=100)
    e.set_particles(other, rng.uniform(-3, 3, (50, 3)), np.zeros(50, np.uint32))
    r = e.add_replica(box, pbc, seed=1, max_particles=len(pos))
    e.set_particles(r, pos, types)
    o = po.System(3, list(box), list(pbc))
    o.add_particles(pos, types.astype(np.int32), ids=np.arange(len(types)))
    for frm, to in [([0, 1, 2], [0, 1, 2]), ([0], [1, 2]), ([1], [])]:
        got, n = e.rdf_counts(r, BORDERS[borders], frm, to)
        want, wn = o.rdf_counts(BORDERS[borders], frm, to)
        assert n == wn
        assert np.array_equal(got, want)
    e.close()
