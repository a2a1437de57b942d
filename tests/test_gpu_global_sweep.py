"""Circle-pair sweeps of the GLOBAL engine against the f32 oracle bit for bit:
components at the edges of the replays (4, 16 and 64 lanes, workgroups in LDS and
in memory), lists at the edges of what they hold, more list entries than there was
room for, circles that scan their cells alone, by 16 lanes and over every record."""
import numpy as np
import pytest

from helpers import bits_equal, first_diff, state, to_oracle
from bendy2d_amd import BD_ENGINE_GLOBAL, Solver

pytestmark = pytest.mark.gpu

DT = 1.0 / 60.0


def check(circles, updates, span):
    s = Solver()
    s.set_engine(BD_ENGINE_GLOBAL)
    s.gravity, s.bounds = (0.0, 0.0), ((-span, -span), (2 * span, 2 * span))
    s.set_sub_steps(2)
    s.add_circles(circles)
    o = to_oracle(s, 32, candidate_mode=len(circles) > 2000)
    for _ in range(updates):
        s.update(DT)
        assert o.update(DT) == 0
        assert s.engine_used == BD_ENGINE_GLOBAL
    assert bits_equal(state(s), state(o)), first_diff(state(s), state(o))


def at(xy, r):
    c = np.zeros((len(xy), 7), np.float32)
    c[:, 0:2] = c[:, 2:4] = xy
    c[:, 6] = r
    return c


@pytest.mark.parametrize("size", [2, 3, 4, 5, 15, 16, 17, 63, 64, 65, 200, 1024, 1025])
def test_chains(size):
    # rows of `size` circles, each overlapping the next, far apart, in an order
    # that is not the rows'
    rows = max(2, 130 // size)
    xy = np.array([(0.9 * k, 20.0 * r + 0.05 * (k % 3)) for r in range(rows) for k in range(size)], np.float32)
    rng = np.random.default_rng(size)
    check(at(xy[rng.permutation(len(xy))], 0.5), 2, 5000.0)


@pytest.mark.parametrize("n", [8, 9, 10, 33, 34, 64, 90, 92, 300])
def test_clumps(n):
    # everything touches everything: lists of n - 1 entries (kept by the counting
    # scan up to 8, by a lane up to 32, by a workgroup up to 8,192 in all), beside
    # a few loose pairs; 300: more entries than there was room for
    rng = np.random.default_rng(n)
    xy = np.concatenate([rng.uniform(-0.3, 0.3, (n, 2)), [(50.0, 0.0), (50.9, 0.0), (-40.0, 7.0), (-40.0, 7.5)]])
    check(at(xy.astype(np.float32), 1.0), 3, 1000.0)


@pytest.mark.parametrize("n", [4, 5, 6, 16, 17, 18, 65, 66, 130])
def test_kept_lists(n):
    # a few hundred circles in clumps of n: lists of n - 1 entries around what a
    # lane sorts (4, 8, 16) and what a wavefront ranks at once (64), many of them
    # in each wavefront
    rng = np.random.default_rng(100 + n)
    clumps = -(-400 // n)
    xy = rng.uniform(-0.25, 0.25, (clumps, n, 2)) + np.array([(12.0 * k, 5.0 * (k % 3)) for k in range(clumps)])[:, None]
    check(at(xy.reshape(-1, 2)[rng.permutation(clumps * n)].astype(np.float32), 1.0), 2, 9000.0)


@pytest.mark.parametrize("n", [2, 3, 7, 16, 17, 257, 4097])
@pytest.mark.parametrize("mixed", [False, True])
def test_levels(n, mixed):
    # a gas in which some circles are shot through the others (large pushes and
    # margins) and, mixed, radii from 0.02 to 8; one circle far away
    rng = np.random.default_rng(n)
    span = 2.0 * np.sqrt(n)
    r = np.where(rng.uniform(size=n) < 0.01, 8.0, rng.uniform(0.02, 0.6, n)) if mixed else np.full(n, 0.5)
    c = at(rng.uniform(0.0, span, (n, 2)).astype(np.float32), r)
    speed = np.where(rng.uniform(size=n) < 0.1, 60.0, 1.0)[:, None]
    c[:, 2:4] -= (speed * rng.standard_normal((n, 2)) * DT / 2).astype(np.float32)
    c[0, 0:4] += 3000.0
    check(c, 3, 5000.0)


@pytest.mark.parametrize("polygons", [0, 1, 2, 3])
def test_bodies_after_a_sweep_run_again(polygons):
    # fast circles bring sweeps that run again; the bodies move once, also where
    # they are queued with the sweep (no two polygons), with initial acc pending
    rng = np.random.default_rng(polygons)
    s = Solver()
    s.set_engine(BD_ENGINE_GLOBAL)
    s.gravity, s.bounds = (0.0, -9.0), ((-10.0, -10.0), (90.0, 90.0))
    s.set_sub_steps(3)
    c = at(rng.uniform(0.0, 60.0, (1500, 2)).astype(np.float32), rng.uniform(0.2, 0.9, 1500))
    c[:, 2:4] -= (25.0 * rng.standard_normal((1500, 2)) * DT / 3).astype(np.float32)
    c[:, 4:6] = rng.uniform(-5.0, 5.0, (1500, 2))
    s.add_circles(c)
    s.add_particle((5.0, 5.0))
    for k in range(polygons):
        s.add_polygon_circle(5.0, (20.0 + 8.0 * k, 70.0), 8, k == 2)
    o = to_oracle(s, 32)
    for _ in range(4):
        s.update(DT)
        assert o.update(DT) == 0
        assert bits_equal(state(s), state(o)), first_diff(state(s), state(o))
    assert s.stats()["cc_redos"] > 0


@pytest.mark.parametrize("size", [2, 4, 5, 16, 17, 64, 65, 1024, 1025])
@pytest.mark.parametrize("clump", [False, True])
def test_pairs_are_taken_by_circle_number(size, clump):
    # every circle at x = -0: a pair's push leaves +0 at its first circle (the one
    # with the smaller number) and -0 at its second, so the signs in the previous
    # positions after one substep tell which end a replay took first.  Columns of
    # `size` circles, each overlapping the next; with clump one more in each place,
    # numbered far from it.
    rows = max(2, 130 // size)
    y = np.array([1.05 * size * r + 0.9 * k for r in range(rows) for k in range(size)])
    if clump:
        y = np.concatenate([y, y + 0.3])
    xy = np.stack([np.full(len(y), -0.0), y], 1).astype(np.float32)
    rng = np.random.default_rng(size)
    s = Solver()
    s.set_engine(BD_ENGINE_GLOBAL)
    s.gravity, s.bounds = (0.0, 0.0), ((-9000.0, -9000.0), (18000.0, 18000.0))
    s.add_circles(at(xy[rng.permutation(len(xy))], 0.5))
    o = to_oracle(s, 32)
    s.update(DT)
    assert o.update(DT) == 0
    a, b = state(s), state(o)
    assert np.signbit(b[2::4]).any() and not np.signbit(b[2::4]).all()
    assert bits_equal(a, b), first_diff(a, b)


@pytest.mark.parametrize("n", [17, 18, 64, 65, 66, 72, 73, 256, 257, 258, 700])
def test_ranked_lists(n):
    # clumps with lists of n - 1 entries, numbered in no order of place: the first
    # lengths that are not kept (above 16), those ranked by one key or four to a lane
    # (64), by blocks of 8 and 64 keys, and in more than one go (256)
    rng = np.random.default_rng(200 + n)
    clumps = max(2, 150 // n)
    xy = rng.uniform(-0.2, 0.2, (clumps, n, 2)) + np.array([(9.0 * k, 4.0 * (k % 2)) for k in range(clumps)])[:, None]
    check(at(xy.reshape(-1, 2)[rng.permutation(clumps * n)].astype(np.float32), 1.0), 2, 9000.0)


@pytest.mark.parametrize("n", [300, 1500, 4000])
@pytest.mark.parametrize("big", [3.0, 15.0])
def test_overruns_in_crowded_cells(n, big):
    # a few large circles make the cells so large that many records share one; fast
    # circles leave their margins, so their cells are searched for pairs that no list
    # holds, in rows of far more records than lanes; the component is replayed in memory
    rng = np.random.default_rng(n + int(big))
    span = 1.6 * np.sqrt(n)
    r = np.where(np.arange(n) % 300 == 7, big, rng.uniform(0.1, 0.4, n))
    c = at(rng.uniform(0.0, span, (n, 2)).astype(np.float32), r)
    speed = np.where(rng.uniform(size=n) < 0.2, 60.0, 1.0)[:, None]
    c[:, 2:4] -= (speed * rng.standard_normal((n, 2)) * DT / 2).astype(np.float32)
    s = Solver()
    s.set_engine(BD_ENGINE_GLOBAL)
    s.gravity, s.bounds = (0.0, 0.0), ((-9000.0, -9000.0), (18000.0, 18000.0))
    s.set_sub_steps(2)
    s.add_circles(c)
    o = to_oracle(s, 32, candidate_mode=True)
    for _ in range(4):
        s.update(DT)
        assert o.update(DT) == 0
        assert bits_equal(state(s), state(o)), first_diff(state(s), state(o))
    assert s.stats()["cc_redos"] > 0
