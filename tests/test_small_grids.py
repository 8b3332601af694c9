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
