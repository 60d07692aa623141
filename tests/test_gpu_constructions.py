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


def left(d):
    """What a construction leaves behind."""
    return d.particles() + d.ghosts() + (d.pairs(), d.kick(), np.array(d.observe_raw()))


def same(a, b):
    return all(np.array_equal(x, y, equal_nan=True) for x, y in zip(a, b))


# what is added to a box of a few hundred particles whose list is built: more than its ghosts', its
# gather lists', its candidate masks' and its list's room (a corner's particles have seven images),
# or more than its masks' and its list's (no images; over 1,024 candidates in 27 cells)
CROWDS = {"corner": (1500, 0.0, 2.9), "middle": (1100, 5.0, 7.0)}


@pytest.mark.parametrize("sort,cells", [(8, 1), (0, 1), (8, 0)])
@pytest.mark.parametrize("crowd", list(CROWDS))
def test_a_construction_that_runs_out_of_room(crowd, sort, cells):
    """A construction that lacks room stops, undoes the row order it had not made, gets its room and
    goes on from that stage: the oracle's pairs, and bit for bit what the next construction, which has
    all its room, makes of the same particles."""
    print("case: room", crowd, sort, cells, flush=True)
    n, lo, hi = CROWDS[crowd]
    L = 12.0
    rng = np.random.default_rng(11)
    x = fcc(L, 0.2)
    q = np.concatenate([x, rng.uniform(lo, hi, (n, 3))])
    p = rng.normal(size=q.shape)
    ids = rng.permutation(len(q)).astype(np.int32)
    d = mdgpu.Domain(L, dt=0.001, rc=2.5, margin=0.5, capacity=len(x))
    d.set_option(mdgpu.OPT_ROW_SORT, sort)
    d.set_option(mdgpu.OPT_SEARCH_CELLS, cells)
    d.add_particles(x, p[:len(x)], ids[:len(x)])
    d.make_pair_list()
    few = d.list_stats()
    d.add_particles(q[len(x):], p[len(x):], ids[len(x):])
    d.make_pair_list()
    st = d.list_stats()
    assert st["slots"] > 4 * few["slots"] and (crowd == "middle" or st["ghosts"] > 4 * few["ghosts"] + 4096), (few, st)
    first = left(d)
    order = np.argsort(first[2])
    by = np.argsort(ids)
    assert np.array_equal(first[2][order], ids[by])
    assert np.array_equal(first[0][order], q[by]) and np.array_equal(first[1][order], p[by])
    o = O.OracleSystem(L, 0.001, 2.5, 0.5)
    o.add(q, p, ids)
    o.make_pair_list()
    assert np.array_equal(O.canonical_pairs(d.pairs()), O.canonical_pairs(o.pairs()))
    d.make_pair_list()
    assert same(first, left(d))
    d.close()


@pytest.mark.parametrize("sort", [8, 0])
@pytest.mark.parametrize("crowd", list(CROWDS))
def test_a_groups_construction_that_runs_out_of_room(crowd, sort):
    """The same for one unit of a group, whose list the others' ghosts index."""
    print("case: room of a unit", crowd, sort, flush=True)
    n, lo, hi = CROWDS[crowd]
    L = 14.0
    rng = np.random.default_rng(12)
    x = fcc(L, 0.2)
    c = rng.uniform(lo, hi, (n, 3))
    us = mdgpu.unit_grid(L, (2, 1, 2), dt=0.001, rc=2.5, margin=0.5, capacity=len(x))
    for u in us:
        u.set_option(mdgpu.OPT_ROW_SORT, sort)
        u.add_particles(x, None, np.arange(len(x), dtype=np.int32))
    us[0].group_make_pair_list()
    for u in us:
        u.add_particles(c, None, np.arange(len(x), len(x) + n, dtype=np.int32))
    us[0].group_make_pair_list()
    for u in us:
        u.send_border_particles()
    first = [left(u) for u in us]
    assert sorted(np.concatenate([f[2] for f in first])) == list(range(len(x) + n))
    us[0].group_make_pair_list()
    for u in us:
        u.send_border_particles()
    for f, u in zip(first, us):
        assert same(f, left(u))


@pytest.mark.parametrize("sort", [8, 0])
@pytest.mark.parametrize("built", [True, False])
def test_particles_after_an_invalid_position(built, sort):
    """A construction refused for a particle that a wrap cannot bring back leaves every particle, its
    momentum and its id where they were; with a position inside again the list is the oracle's."""
    print("case: invalid position", built, sort, flush=True)
    L = 12.0
    rng = np.random.default_rng(13)
    q = np.mod(fcc(L, 0.5) + rng.uniform(-0.2, 0.2, (len(fcc(L, 0.5)), 3)), L)
    p = rng.normal(size=q.shape)
    ids = rng.permutation(len(q)).astype(np.int32)
    d = mdgpu.Domain(L, dt=0.001, rc=2.5, margin=0.5, capacity=len(q))
    d.set_option(mdgpu.OPT_ROW_SORT, sort)
    d.add_particles(q, p, ids)
    if built:
        d.make_pair_list()
    q0, p0, t0 = d.particles()
    bad = q0.copy()
    bad[len(q) // 3] += 5.0 * L
    d.set_positions(bad)
    for _ in range(2):  # refused as often as it is asked for
        with pytest.raises(mdgpu.MDGPUError) as e:
            d.make_pair_list()
        assert e.value.code == mdgpu.ERR_INVALID_POSITION
        _, p1, t1 = d.particles()
        assert np.array_equal(p1, p0) and np.array_equal(t1, t0)
    d.set_positions(q0)
    d.make_pair_list()
    o = O.OracleSystem(L, 0.001, 2.5, 0.5)
    o.add(q0, p0, t0)
    o.make_pair_list()
    assert np.array_equal(O.canonical_pairs(d.pairs()), O.canonical_pairs(o.pairs()))
    q2, p2, t2 = d.particles()
    i, k = np.argsort(t2), np.argsort(t0)
    assert np.array_equal(p2[i], p0[k]) and np.array_equal(q2[i], q0[k])
    d.close()


def test_units_after_an_invalid_position():
    """The same for one unit of a group: each unit keeps its particles."""
    print("case: invalid position of a unit", flush=True)
    L = 14.0
    rng = np.random.default_rng(14)
    q = fcc(L, 0.5)
    p = rng.normal(size=q.shape)
    us = mdgpu.unit_grid(L, (2, 1, 2), dt=0.001, rc=2.5, margin=0.5, capacity=len(q))
    for u in us:
        u.add_particles(q, p)
    us[0].group_make_pair_list()
    state = [u.particles() for u in us]
    bad = state[1][0].copy()
    bad[7, 1] += 5.0 * L  # along the axis of one unit, where it does not migrate
    us[1].set_positions(bad)
    with pytest.raises(mdgpu.MDGPUError) as e:
        us[0].group_make_pair_list()
    assert e.value.code == mdgpu.ERR_INVALID_POSITION
    after = [u.particles() for u in us]
    t, k = np.concatenate([a[2] for a in after]), np.concatenate([a[2] for a in state])
    assert np.array_equal(np.sort(t), np.arange(len(q)))
    pa, ps = np.concatenate([a[1] for a in after]), np.concatenate([a[1] for a in state])
    assert np.array_equal(pa[np.argsort(t)], ps[np.argsort(k)])
    want = np.concatenate([a[0] for a in state])[np.argsort(k)]
    for u, a in zip(us, after):
        u.set_positions(want[a[2]])
    us[0].group_make_pair_list()
    for u in us:
        u.send_border_particles()
    assert sum(u.counts()[0] for u in us) == len(q)
    for u, s in zip(us, state):
        assert all(np.array_equal(x, y) for x, y in zip(u.particles(), s))
