"""The four buffer states of the fused step: runs that start in each of them, graph-replayed and launched, with
replicas admitted, removed and re-binned in between."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

L = pytest.importorskip("readdy_amd._lib")
from readdy_amd import Engine  # noqa: E402
from readdy_amd import ensemble as E  # noqa: E402


def _engine(sizes, **kw):
    pots, rxs = E.chemistry()
    rxs = [dict(rx, rate=rx["rate"] * 20) for rx in rxs]
    e = Engine(3, E.DIFFUSION, potentials=pots, reactions=rxs, max_replicas=8, max_cells=8 * 1000, max_particles=40000, **kw)
    return e, [_admit(e, n, k) for k, n in enumerate(sizes)]


def _admit(e, n, seed):
    box = (n / 0.5) ** (1.0 / 3.0)
    r = e.add_replica([box] * 3, seed=seed, max_particles=2 * n)
    e.set_particles(r, *E.initial_state(n, box, seed))
    return r


def _same(e1, e2, ids):
    for r in ids:
        for a, b in zip(e1.get_particles(r), e2.get_particles(r)):
            assert np.array_equal(a, b)
        assert np.array_equal(e1.reaction_totals(r), e2.reaction_totals(r))
    assert np.array_equal(e1.count_types(8), e2.count_types(8))


@pytest.mark.parametrize("steps", [(1, 2, 3, 4, 5, 6), (33, 34, 35, 36), (2, 70, 1, 41, 3, 129)])
@pytest.mark.parametrize("handler", [L.HANDLER_UA, L.HANDLER_NONE])
def test_graph_replay_equals_launches_from_every_state(steps, handler):
    """Runs of n steps advance the state by n + 1 (the first walk), so the sequences start in every state; from 33
    steps on a run replays the graph of four steps, captured for the state it starts in."""
    e1, ids = _engine((500, 900, 40))
    e2, _ = _engine((500, 900, 40))
    for n in steps:
        e1.run(handler, 0.005, n, graph=True)
        e2.run(handler, 0.005, n, graph=False)
        _same(e1, e2, ids)
    for e in (e1, e2):
        e.close()


def test_admission_and_removal_between_runs():
    """A replica's cells are clear in every state's counters when the next replica takes them."""
    e, ids = _engine((600, 300), bin_capacity=4)  # crowded cells overflow
    alone = {}
    for k in range(6):
        e.run(L.HANDLER_UA, 0.005, 1 + k, graph=True)
        e.remove_replica(ids.pop(0))
        e.update_neighbor_list()
        ids.append(_admit(e, 200 + 150 * k, 50 + k))
        alone[ids[-1]] = (200 + 150 * k, 50 + k, k)
    e.run(L.HANDLER_UA, 0.005, 37, graph=True)
    for r in ids:
        n, seed, k = alone[r]
        one, _ = _engine((), bin_capacity=4)
        q = _admit(one, n, seed)
        for j in range(k + 1, 6):  # its neighbour's runs since its admission, with their own first walks
            one.run(L.HANDLER_UA, 0.005, 1 + j)
            one.update_neighbor_list()
        one.run(L.HANDLER_UA, 0.005, 37)
        for a, b in zip(e.get_particles(r), one.get_particles(q)):
            assert np.array_equal(a, b)
        one.close()
    e.close()


def test_no_replicas_left():
    e, (r,) = _engine((100,))
    e.run(L.HANDLER_UA, 0.005, 3)
    e.remove_replica(r)
    e.run(L.HANDLER_UA, 0.005, 3, graph=True)
    e.run(L.HANDLER_UA, 0.005, 3)
    e.update_neighbor_list()
    assert e.count_types(8).sum() == 0
    q = _admit(e, 150, 3)
    e.run(L.HANDLER_UA, 0.005, 40, graph=True)
    assert 75 <= e.n_particles(q) <= 300
    e.close()


@pytest.mark.parametrize("steps", [1, 2, 3])
def test_an_open_run_without_replicas(steps):
    """It steps nothing and leaves every state's counters as they are: the replica admitted next, under the removed
    one's id and with crowded cells, is as in an engine of its own."""
    e, (r,) = _engine((700,), bin_capacity=1)
    e.run(L.HANDLER_UA, 0.005, 5)  # overflow records in both buffers
    e.remove_replica(r)
    e.run_begin(L.HANDLER_UA, 0.005, steps)
    e.run_enqueue(steps)
    e.run_end()
    one, _ = _engine((), bin_capacity=1)
    for x in (e, one):
        assert _admit(x, 400, 7) == r
    _same(e, one, [r])
    for n in (1, 2, 3, 4):
        for x in (e, one):
            x.run(L.HANDLER_UA, 0.005, n)
        _same(e, one, [r])
    for x in (e, one):
        x.close()


def test_a_replicas_footprint_counts_every_state():
    """A cell takes its records in two buffers and a counter in each of the four states."""
    e, _ = _engine((100,), bin_capacity=8)
    assert e.footprint([20.0] * 3, 50) - e.footprint([10.0] * 3, 50) == (8000 - 1000) * (2 * 8 * 32 + 4 * 4)
    e.close()
