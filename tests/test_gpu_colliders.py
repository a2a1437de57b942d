"""Static colliders on the GPU against the f32 oracle bit for bit: as many as the
batches in which their records are read, one less and one more, circles and
polygons in turn, bodies that hit several."""
import numpy as np
import pytest

from helpers import bits_equal, first_diff, state, to_oracle
from bendy2d_amd import BD_ENGINE_GLOBAL, BD_ENGINE_SCENE, BD_ENGINE_TILED, Solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("engine", [BD_ENGINE_SCENE, BD_ENGINE_GLOBAL, BD_ENGINE_TILED])
@pytest.mark.parametrize("count", [0, 1, 3, 4, 5, 7, 8, 9, 13])
def test_counts(count, engine):
    rng = np.random.default_rng(10 * count + engine)
    n = 17000 if engine == BD_ENGINE_TILED else 700
    span = 60.0
    s = Solver()
    s.set_engine(engine)
    s.gravity, s.bounds = (1.0, -30.0), ((0.0, 0.0), (span, span))
    s.set_sub_steps(2)
    p = rng.uniform(0.0, span, (n, 2)).astype(np.float32)
    s.add_particles(p, p)
    i = np.arange(0, n - 1, 2, dtype=np.uint32)
    s.add_particle_links(i, i + 1, np.full(len(i), 30.0, np.float32))
    if engine != BD_ENGINE_TILED:
        c = np.zeros((300, 7), np.float32)
        c[:, 0:2] = c[:, 2:4] = rng.uniform(0.0, span, (300, 2))
        c[:, 6] = rng.uniform(0.1, 0.8, 300)
        s.add_circles(c)
    for k in range(count):
        at = rng.uniform(0.2 * span, 0.8 * span, 2)
        if k % 3 == 1:
            m = 3 + k % 5
            a = 2 * np.pi * np.arange(m) / m
            s.add_static_polygon((at + 9.0 * np.stack([np.cos(a), np.sin(a)], -1)).astype(np.float32))
        else:
            s.add_static_circle(tuple(float(np.float32(x)) for x in at), 8.0)
    o = to_oracle(s, 32)
    for _ in range(3):
        s.update(1.0 / 60.0)
        assert o.update(1.0 / 60.0) == 0
    assert s.engine_used == engine
    assert bits_equal(state(s), state(o)), first_diff(state(s), state(o))
