"""Polygon pairs against the f32 oracle bit for bit: many edges hit in one step of
the pair loop, polygons of as many points as the lanes of a workgroup and more, more
polygons than a wavefront's lanes hold, positions in LDS and in memory."""
import numpy as np
import pytest

from helpers import bits_equal, first_diff, state, to_oracle
from bendy2d_amd import BD_ENGINE_GLOBAL, Batch, Solver
from bendy2d_amd.solver import polygon_circle

pytestmark = pytest.mark.gpu

DT = 1.0 / 60.0
CASES = [(2, [3]), (5, [12, 3, 4, 40]), (3, [63, 64, 65]), (3, [130, 7, 257]), (66, [3, 5])]


def scene(count, points, seed):
    rng = np.random.default_rng(seed)
    s = Solver()
    s.gravity, s.bounds = (0.0, 10.0), ((0.0, 0.0), (60.0, 60.0))
    s.set_sub_steps(2)
    for k in range(count):
        n = points[k % len(points)]
        at = (float(rng.uniform(20.0, 40.0)), float(rng.uniform(20.0, 40.0)))
        pts, links, c = polygon_circle(float(rng.uniform(3.0, 9.0)), at, n, False)
        s.add_polygon(pts, links, False, c, 1.0)
    s.add_polygon_new([(0.0, 45.0), (60.0, 45.0), (60.0, 55.0), (0.0, 55.0)], True)
    return s


def check(s, o, updates):
    for _ in range(updates):
        assert o.update(DT) == 0
    assert bits_equal(state(s), state(o)), first_diff(state(s), state(o))


@pytest.mark.parametrize("count,points", CASES)
def test_global(count, points):
    s = scene(count, points, count)
    s.set_engine(BD_ENGINE_GLOBAL)
    o = to_oracle(s, 32)
    for _ in range(4):
        s.update(DT)
    assert s.engine_used == BD_ENGINE_GLOBAL
    check(s, o, 4)


@pytest.mark.parametrize("lds", [0, 64 * 1024])
@pytest.mark.parametrize("wg", [64, 128, 256, 512, 1024])
@pytest.mark.parametrize("count,points", CASES)
def test_scene(count, points, wg, lds):
    s = scene(count, points, count)
    o = to_oracle(s, 32)
    b = Batch()
    b.add_scene(s)
    b.config = dict(wg_small=wg, wg_large=wg, split_points=16384, lds_small=lds, lds_large=lds, steps_per_launch=2,
                    use_graph=0, split_tiny=0)
    b.update(DT, 4)
    b.sync()
    b.read_scene(0, s)
    check(s, o, 4)
