"""Counts and particles read back from the device: cells that overflow their bins, blocks of cells that hold one
replica or many, empty replicas, removed replicas, and many types."""
import ctypes

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


@pytest.mark.parametrize("n,kw", [(0, {}), (1, {}), (255, {}), (256, {}), (5000, {}), (3000, dict(bin_capacity=2)),
                                  (40000, {}),      # larger than the area a small answer comes back through
                                  (400001, {})])    # several halves of the streamed area, a remainder in each
def test_particles_come_back_in_handle_order(n, kw):
    """Handles are the upload order, so the arrays come back as they went up; a second replica's stay apart."""
    box = 12.0 if n < 6000 else 60.0
    e, data = _engine((n, 77), box=box, **kw)
    for r, pos, types in data:
        p, t, h = e.get_particles(r)
        assert np.array_equal(h, np.arange(len(types)))
        assert np.array_equal(t, types)
        assert np.array_equal(p, pos)
        assert e.n_particles(r) == len(types)
    e.close()


def test_handles_past_the_expected_range_and_forces_in_step():
    """Decays and conversions leave gaps and reach handles beyond the last read (a conversion renames: 900 x 40 steps
    pass the first estimate): the particles still come back ordered, and the forces in the same order."""
    rng = np.random.default_rng(5)
    e = Engine(2, [1.0, 1.0], potentials=[(L.POT_HARMONIC_REPULSION, a, b, [10.0, 1.0]) for a, b in ((0, 0), (0, 1), (1, 1))],
               reactions=[dict(kind=L.RX_CONVERSION, educts=[0], products=[1], rate=80.0),
                          dict(kind=L.RX_CONVERSION, educts=[1], products=[0], rate=80.0),
                          dict(kind=L.RX_DECAY, educts=[0], products=[], rate=0.5)])
    r = e.add_replica([10.0] * 3, seed=9, max_particles=1000)
    e.set_particles(r, (rng.random((900, 3)) - 0.5) * 10.0, np.zeros(900, np.uint32))
    e.run(L.HANDLER_UA, 0.01, 40)
    p, t, h = e.get_particles(r)
    assert h.max() > 4096 + 1350 and len(h) == e.n_particles(r) < 900
    assert np.all(np.diff(h.astype(np.int64)) > 0)
    assert np.array_equal(e.count_types(1)[0], np.bincount(t, minlength=2))
    f, hf = e.get_forces(r)
    assert np.array_equal(hf, h)
    d = p[None] - p[:, None]  # neighbour - particle
    d -= 10.0 * np.round(d / 10.0)
    dist = np.sqrt((d * d).sum(2)) + 10.0 * np.eye(len(p))
    ref = (np.where(dist < 1.0, 10.0 * (dist - 1.0) / dist, 0.0)[:, :, None] * d).sum(1)
    assert np.linalg.norm(f - ref) < 1e-5 * np.linalg.norm(ref)
    e.close()


def _converting(n, inert, box, seed=3):
    """the first `inert` particles stay (type 2), the others change their handle with every reaction (0 <-> 1)"""
    rng = np.random.default_rng(seed)
    e = Engine(3, [1.0] * 3, potentials=[(L.POT_HARMONIC_REPULSION, a, b, [10.0, 1.0]) for a in range(3) for b in range(a, 3)],
               reactions=[dict(kind=L.RX_CONVERSION, educts=[a], products=[1 - a], rate=1e4) for a in (0, 1)],
               events_per_replica=1024)
    r = e.add_replica([box] * 3, seed=9, max_particles=n + 16)
    pos = (rng.random((n, 3)) - 0.5) * box
    e.set_particles(r, pos, np.where(np.arange(n) < inert, 2, 0).astype(np.uint32))
    return e, r, pos


@pytest.mark.parametrize("inert,shared", [(0, 0), (30, 15)])
def test_readback_across_the_end_of_the_handle_counter(inert, shared):
    """60 - inert particles take the last 2^32 handles and the first ones after the counter has wrapped; with inert
    particles these are still in use, and every particle comes back all the same."""
    e, r, pos = _converting(60, inert, 8.0)
    new = 60 - inert
    e.set_next_handle(r, 2 ** 32 - new // 2)
    e.react(L.HANDLER_UA, 1.0)
    want = sorted([*range(inert), *((2 ** 32 - new // 2 + k) % 2 ** 32 for k in range(new))])
    assert len(want) - len(set(want)) == shared
    for _ in range(2):
        p, t, h = e.get_particles(r)
        assert h.tolist() == want
        assert np.array_equal(p[np.lexsort(p.T)], pos[np.lexsort(pos.T)])
        assert np.bincount(t, minlength=3).tolist() == [0, new, inert]
        e.calculate_forces()
        f, hf = e.get_forces(r)
        assert np.array_equal(hf, h) and np.abs(f).sum(1).astype(bool).any()
    with pytest.raises(L.EngineError):
        e.set_next_handle(r, 0)
    e.close()


@pytest.mark.parametrize("n,inert,start", [(500, 0, 2 ** 31), (500, 200, 87 * 10 ** 6), (500, 200, 88 * 10 ** 6),
                                           (20, 0, 2 ** 22), (20, 0, 2 ** 23), (10000, 9500, 2 ** 32 - 10 ** 6),
                                           (40000, 39500, 10 ** 8), (40000, 39500, 2 ** 32 - 10 ** 6)])
def test_readback_of_handles_far_apart(n, inert, start):
    """Both sides of the line between the bitmap and the sorted list, small answers and streamed ones; a shorter
    array takes the first rows."""
    e, r, pos = _converting(n, inert, 8.0 if n < 1000 else 40.0)
    twin, q, _ = _converting(n, inert, 8.0 if n < 1000 else 40.0)  # the same system with its handles close together
    e.set_next_handle(r, start)
    for k in range(3):
        for x in (e, twin):
            x.react(L.HANDLER_UA, 1.0)
            x.calculate_forces()
        p, t, h = e.get_particles(r)
        assert np.all(np.diff(h.astype(np.int64)) > 0)
        assert h[inert:].tolist() == [start + k * (n - inert) + j for j in range(n - inert)]
        # who takes which of the new handles depends on the draws, which follow the handles: compare by position
        tp, tt, _ = twin.get_particles(q)
        o, to = np.lexsort(p.T), np.lexsort(tp.T)
        assert np.array_equal(p[o], tp[to]) and np.array_equal(t[o], tt[to])
        f, hf = e.get_forces(r)
        assert np.array_equal(hf, h) and np.array_equal(f[o], twin.get_forces(q)[0][to])
    cap = min(33, n // 2)
    some, m = np.zeros(cap, np.uint32), ctypes.c_uint64()
    L.check(e._lib.rdy_get_particles(e._h, r, cap, None, None, some.ctypes.data_as(ctypes.POINTER(ctypes.c_uint32)),
                                     ctypes.byref(m)))
    assert m.value == n and np.array_equal(some, h[:cap])
    e.close()
    twin.close()


def test_readback_of_a_replica_that_never_held_particles():
    """with room for particles in the caller's arrays; the calls that follow are not affected"""
    e, ((r, pos, _),) = _engine((50,))
    e.remove_replica(r)
    q = e.add_replica([12.0] * 3, seed=1, max_particles=50)
    h, m = np.zeros(8, np.uint32), ctypes.c_uint64(7)
    hp = h.ctypes.data_as(ctypes.POINTER(ctypes.c_uint32))
    for _ in range(2):
        L.check(e._lib.rdy_get_particles(e._h, q, 8, None, None, hp, ctypes.byref(m)))
        assert m.value == 0
        e.calculate_forces()
        m.value = 7
        L.check(e._lib.rdy_get_forces(e._h, q, 8, None, hp, ctypes.byref(m)))
        assert m.value == 0
        e.run(L.HANDLER_UA, 0.01, 2)
    e.set_particles(q, pos, np.zeros(50, np.uint32))
    assert np.array_equal(e.get_particles(q)[0], pos)
    e.close()


@pytest.mark.parametrize("kw", [{}, dict(bin_capacity=2)])
def test_an_upload_takes_the_room_of_the_one_it_replaces(kw):
    """Uploads one after another without a step between them, more than the engine holds at once: each is as the first
    one of an engine of its own, and the other replica is untouched."""
    rng = np.random.default_rng(8)
    e, data = _engine((700, 700), **kw)
    (r, _, _), (other, opos, _) = data
    for k in range(16):
        n = 700 if k % 2 else 100 + k
        pos, types = (rng.random((n, 3)) - 0.5) * 12.0, rng.integers(0, 3, n).astype(np.uint32)
        e.set_particles(r, pos, types)
        p, t, h = e.get_particles(r)
        assert np.array_equal(p, pos) and np.array_equal(t, types) and np.array_equal(h, np.arange(n))
        assert np.array_equal(e.count_types(2)[r], np.bincount(types, minlength=3))
        assert np.array_equal(e.get_particles(other)[0], opos)
        one, ((q, _, _),) = _engine((700,), **kw)
        one.set_particles(q, pos, types)
        for x, i in ((e, r), (one, q)):
            x.calculate_forces()
        assert np.array_equal(e.get_forces(r)[0], one.get_forces(q)[0]) and e.energy(r) == one.energy(q)
        one.close()
    e.close()
