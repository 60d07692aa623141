"""Constructions off the usual path on the GPU: phases of a unit repeated, room that runs out at each
stage, and states that are refused."""
import numpy as np
import pytest

from mdacp_amd import mdgpu
from mdacp_amd.lattice import fcc, initial_velocity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid", [(2, 2, 2), (1, 1, 1), (3, 1, 2)])
def test_a_units_ghosts_placed_again(grid):
    """FindBorderParticles of a unit several times in a row, the first of them making room (more
    ghosts than a unit made for one particle holds), with nothing that waits in between: the ghosts,
    pairs and observers of a group whose phases ran once each."""
    print("case: ghosts placed again", grid, flush=True)
    L = 21.0 if max(grid) > 2 else 14.0
    q = fcc(L, 0.9)
    q = np.mod(q + np.random.default_rng(5).uniform(-0.1, 0.1, q.shape), L)
    p = initial_velocity(len(q), 1.0, seed=2)
    sides = []
    for times in (3, 1):
        us = mdgpu.unit_grid(L, grid, dt=0.005, rc=2.5, margin=0.5, capacity=1)
        for u in us:
            u.add_particles(q, p)
            u.adjust_periodic_boundary()
        for u in us:
            for _ in range(times):
                u.find_border_particles()
        assert max(u.counts()[1] - u.counts()[0] for u in us) > 1024
        for u in us:
            u.make_pair_list()
        for u in us:
            u.send_border_particles()
        sides.append(us)
    for u, v in zip(*sides):
        assert u.counts() == v.counts()
        for x, y in zip(u.particles() + u.ghosts(), v.particles() + v.ghosts()):
            assert np.array_equal(x, y)
        assert np.array_equal(u.pairs(), v.pairs())
        assert u.observe_raw() == v.observe_raw()
