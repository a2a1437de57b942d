"""The link solves' shared root and reciprocal and the layered link phase,
against the f32 oracle bit for bit: link lengths over the whole range of f32
(the plain operations take over outside a part of it), differences of zero of
either sign, coinciding ends, layer counts around the 64 bounds a wavefront
holds, and layers of one record more or less than a workgroup has lanes."""
import numpy as np
import pytest

from helpers import bits_equal, first_diff, state, to_oracle
from bendy2d_amd import BD_ENGINE_GLOBAL, BD_ENGINE_SCENE, BD_ENGINE_TILED, Solver

pytestmark = pytest.mark.gpu

FAR = ((-1.0e30, -1.0e30), (2.0e30, 2.0e30))


def run(s, updates, engine):
    s.set_engine(engine)
    o = to_oracle(s, 32)
    for _ in range(updates):
        s.update(1.0 / 60.0)
        assert o.update(1.0 / 60.0) == 0
    assert s.engine_used == engine
    a, b = state(s), state(o)
    assert bits_equal(a, b), f"first diff {first_diff(a, b)}"


@pytest.mark.parametrize("engine", [BD_ENGINE_SCENE, BD_ENGINE_GLOBAL, BD_ENGINE_TILED])
@pytest.mark.parametrize("scale", [1e-38, 1e-24, 3e-17, 1e-9, 1.0, 1e9, 1e18, 2e19, 1e30])
def test_link_lengths(engine, scale):
    n = 16386 if engine == BD_ENGINE_TILED else 600  # TILED takes more than 16,384 points
    rng = np.random.default_rng(int(np.log2(scale)) + 2000)
    p = (rng.uniform(-1, 1, (n, 2)) * scale).astype(np.float32)
    p[0:40:2] = p[1:41:2]                       # coinciding ends
    p[40:80:2, 0] = p[41:81:2, 0]               # axis-aligned
    p[80:120:2, 0], p[81:121:2, 0] = -0.0, 0.0  # a difference of -0
    p[120:160:2, 0] = p[121:161:2, 0] + np.float32(1e-30)
    s = Solver()
    s.gravity, s.bounds = (0.0, 0.0), FAR
    s.set_link_iterations(2)
    s.add_particles(p, p)
    a = np.arange(0, n - 1, 2)
    s.add_particle_links(a, a + 1, rng.uniform(0, 2, len(a)) * scale)
    s.set_pinned_range(0, (np.arange(n) % 7 == 3).astype(np.uint8))
    run(s, 2, engine)


@pytest.mark.parametrize("links", [1, 62, 63, 64, 65, 130])
def test_chain_depth(links):
    s = Solver()
    s.gravity, s.bounds = (0.0, -9.81), FAR
    s.set_link_iterations(3)
    s.add_particles(np.stack([np.arange(links + 1) * 0.9, np.zeros(links + 1)], -1))
    a = np.arange(links)
    s.add_particle_links(a, a + 1, np.full(links, 1.0))
    s.set_pinned(0)
    run(s, 3, BD_ENGINE_SCENE)


@pytest.mark.parametrize("circles", [False, True])
@pytest.mark.parametrize("pairs", [63, 64, 65, 255, 257, 1024, 1025, 3073])
def test_layer_sizes(pairs, circles):
    rng = np.random.default_rng(pairs)
    n = 2 * pairs + 1
    p = np.stack([np.arange(n) * 3.0, rng.uniform(-1, 1, n)], -1).astype(np.float32)
    s = Solver()
    s.gravity, s.bounds = (0.0, -9.81), FAR
    a, t = np.arange(0, n - 1, 2), rng.uniform(2.5, 3.5, pairs)
    if circles:
        c = np.zeros((n, 7), np.float32)
        c[:, 0:2] = c[:, 2:4] = p
        c[:, 6] = 0.5
        s.add_circles(c)
        s.add_circle_links(np.r_[a, a + 1], np.r_[a + 1, a + 2], np.r_[t, t])
    else:
        s.add_particles(p)
        s.add_particle_links(np.r_[a, a + 1], np.r_[a + 1, a + 2], np.r_[t, t])
    run(s, 2, BD_ENGINE_SCENE)
