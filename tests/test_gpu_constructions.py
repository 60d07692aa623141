"""Constructions off the usual path on the GPU: phases of a unit repeated, room that runs out at each
stage, and states that are refused."""
import ctypes

import numpy as np
import pytest

from mdacp_amd import mdgpu
from mdacp_amd.lattice import fcc, initial_velocity
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def free_bytes():
    """Free device memory (the HIP runtime that the library has loaded)."""
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert mdgpu.load().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


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


@pytest.mark.parametrize("state", ["even", "cluster"])
def test_a_neighbourhood_beyond_16_bits_is_refused_before_the_search(state):
    """More particles around a brick than 16-bit indices reach: the capacity error, without the masks
    and lists that a search of them would need (2 GB and more), and a domain that still works."""
    print("case: refused neighbourhood", state, flush=True)
    rng = np.random.default_rng(3)
    if state == "even":
        L, q = 12.0, rng.uniform(0.0, 12.0, (165000, 3))  # 69,600 in 27 of 64 cells
    else:
        L, q = 20.0, np.concatenate([fcc(20.0, 0.5), rng.uniform(7.5, 8.5, (66000, 3))])
    d = mdgpu.Domain(L, dt=0.005, rc=2.5, margin=0.5, capacity=len(q))
    d.add_particles(q)
    before = free_bytes()
    with pytest.raises(mdgpu.MDGPUError, match="16-bit") as e:
        d.make_pair_list()
    assert e.value.code == mdgpu.ERR_CAPACITY
    assert before - free_bytes() < 1 << 29
    assert np.array_equal(np.sort(d.particles()[2]), np.arange(len(q)))
    d.clear_particles()
    x = fcc(L, 0.6)
    fresh = mdgpu.Domain(L, dt=0.005, rc=2.5, margin=0.5, capacity=len(x))
    for f in (d, fresh):
        f.add_particles(x, initial_velocity(len(x), 1.0, seed=1))
        f.make_pair_list()
    assert np.array_equal(O.canonical_pairs(d.pairs()), O.canonical_pairs(fresh.pairs()))
    d.calculate(20)
    for f in (d, fresh):
        f.close()
