"""Counts and particles read back from the device: cells that overflow their bins, blocks of cells that hold one
replica or many, empty replicas, removed replicas, and many types."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

L = pytest.importorskip("readdy_amd._lib")
from readdy_amd import Engine  # noqa: E402


def _engine(sizes, n_types=3, box=12.0, **kw):
    rng = np.random.default_rng(len(sizes))
    e = Engine(n_types, np.ones(n_types), potentials=[(L.POT_HARMONIC_REPULSION, 0, 1, [10.0, 1.0])],
               max_replicas=len(sizes), **kw)
    data = []
    for k, n in enumerate(sizes):
        r = e.add_replica([box] * 3, seed=k, max_particles=max(sizes) + 16)
        pos = (rng.random((n, 3)) - 0.5) * box
        types = rng.integers(0, n_types, n).astype(np.uint32)
        e.set_particles(r, pos, types)
        data.append((r, pos, types))
    return e, data


@pytest.mark.parametrize("sizes,kw", [
    ((1,), {}), ((63,), {}), ((5000,), {}),
    ((400, 0, 1, 700, 64), {}),                      # several replicas, one empty, share blocks of cells
    ((300,) * 9, dict(nl_cutoff=4.0)),               # 27 cells a replica: many replicas in one block
    ((3000, 2000), dict(bin_capacity=2)),            # most records in the overflow region
    ((900,), dict(n_types=700)),                     # more types than a block has threads
])
def test_counts_per_replica_and_type(sizes, kw):
    e, data = _engine(sizes, **kw)
    nt = e.n_types
    got = e.count_types(len(sizes))
    for r, _, types in data:
        assert np.array_equal(got[r], np.bincount(types, minlength=nt))
    if len(sizes) > 1:  # a removed replica's records are not counted, and a shorter table is respected
        e.remove_replica(data[0][0])
        got = e.count_types(len(sizes))
        assert got[0].sum() == 0
        assert np.array_equal(e.count_types(2), got[:2])
    e.close()
