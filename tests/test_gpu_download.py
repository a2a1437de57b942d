"""Reading a scene back on the GPU: the gather of its arrays at the sizes where
the launch's grid begins and ends, parameters that change between updates, and
solvers that share the page-locked buffers."""
import threading

import numpy as np
import pytest

from helpers import bits_equal, first_diff, state, to_oracle
from bendy2d_amd import BD_ENGINE_GLOBAL, BD_ENGINE_SCENE, BD_ENGINE_TILED, Solver, workloads

pytestmark = pytest.mark.gpu


def strip(n, engine):
    """A chain of n particles under gravity."""
    s = Solver()
    s.set_engine(engine)
    s.gravity, s.bounds = (0.0, -9.81), ((-1e6, -1e6), (2e6, 2e6))
    rng = np.random.default_rng(n)
    p = np.stack([np.arange(n), rng.uniform(-0.1, 0.1, n)], -1).astype(np.float32)
    s.add_particles(p, p)
    i = np.arange(n - 1, dtype=np.uint32)
    for part in (i[0::2], i[1::2]):
        if len(part):
            s.add_particle_links(part, part + 1, np.ones(len(part), np.float32))
    return s


@pytest.mark.parametrize("n,engine", [(1, BD_ENGINE_SCENE), (255, BD_ENGINE_SCENE), (257, BD_ENGINE_GLOBAL),
                                      (16385, BD_ENGINE_TILED), (524288 + 1, BD_ENGINE_TILED),
                                      (600001, BD_ENGINE_GLOBAL)])
def test_sizes(n, engine):
    s = strip(n, engine)
    o = to_oracle(s, 32)
    for _ in range(2):
        s.update(1.0 / 60.0)
        assert o.update(1.0 / 60.0) == 0
        a, w = state(s), state(o)
        assert bits_equal(a, w), first_diff(a, w)
    assert s.engine_used == engine


# 64 MiB of state, the most that goes through page-locked memory, and more, whole
# arrays or read by index
@pytest.mark.parametrize("n,engine", [(4194304, BD_ENGINE_GLOBAL), (4194305, BD_ENGINE_GLOBAL),
                                      (4194305, BD_ENGINE_TILED)])
def test_large_sizes(n, engine):
    s = Solver()
    s.set_engine(engine)
    s.gravity, s.bounds = (0.0, -9.81), ((-1e6, -1e6), (2e6, 2e6))
    i = np.arange(n)
    p = np.stack([i % 2048, i // 2048], -1).astype(np.float32)
    s.add_particles(p, p - np.float32(0.25))
    a = np.arange(0, 2000, 2, dtype=np.uint32)
    s.add_particle_links(a, a + 1, np.full(len(a), 0.75, np.float32))
    o = to_oracle(s, 32)
    for _ in range(2):
        s.update(1.0 / 60.0)
        assert o.update(1.0 / 60.0) == 0
        x, w = s.get_particles()[:, :4], o.get_particles()[:, :4]
        assert bits_equal(x, w), first_diff(x.ravel(), np.asarray(w).ravel())
    assert s.engine_used == engine


def test_parameters_change_between_updates():
    s = Solver()
    workloads.cloth_pinned(s, n=12, sub_steps=2, link_iters=2)
    o = to_oracle(s, 32)
    for dt, g, subs in ((0.01, -9.81, 2), (0.01, -9.81, 2), (0.02, -9.81, 2), (0.02, 3.0, 2), (0.02, 3.0, 5),
                        (0.01, -9.81, 2)):
        s.gravity = (0.5, g)
        o.set_gravity((0.5, g))
        s.set_sub_steps(subs)
        o.set_sub_steps(subs)
        s.update(dt)
        assert o.update(dt) == 0
        assert bits_equal(state(s), state(o))


def test_solvers_share_the_buffers():
    sizes = (300, 5000, 40000, 70, 20000, 900)
    failed = []

    def work(n):
        try:
            s = strip(n, BD_ENGINE_GLOBAL if n == 5000 else BD_ENGINE_TILED if n > 16384 else BD_ENGINE_SCENE)
            o = to_oracle(s, 32)
            for _ in range(5):
                s.update(0.01)
                assert o.update(0.01) == 0
                assert bits_equal(state(s), state(o))
        except BaseException as e:  # noqa: BLE001 -- reported by the main thread
            failed.append((n, e))

    threads = [threading.Thread(target=work, args=(n,)) for n in sizes]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed
