"""The TILED engine's own choice of tile size against the f32 oracle bit for bit:
both sides of the line to larger tiles, and a deep link graph."""
import numpy as np
import pytest

from helpers import bits_equal, first_diff, state, to_oracle
from bendy2d_amd import BD_ENGINE_TILED, BD_ORDER_PARTICLE, Solver, workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,kw", [(129, {}), (362, {}), (363, {}), (513, {}), (129, {"order": BD_ORDER_PARTICLE})])
def test_default_tiles(n, kw):
    s = Solver()
    s.set_engine(BD_ENGINE_TILED)
    dt, _ = workloads.cloth_pinned(s, n=n, sub_steps=2, link_iters=3, **kw)
    o = to_oracle(s, 32)
    for _ in range(2):
        s.update(dt)
        assert s.engine_used == BD_ENGINE_TILED
        assert o.update(dt) == 0
    assert bits_equal(state(s), state(o)), first_diff(state(s), state(o))


# the tiles behind the linked particles have no record of their own; 513 linked
# ones make 512 records, which fill a page
@pytest.mark.parametrize("n,linked,chain", [(20480, 513, 1), (20011, 65, 3), (16385, 2, 1)])
def test_tiles_without_links(n, linked, chain):
    s = Solver()
    s.set_engine(BD_ENGINE_TILED)
    s.set_tiling(512, 256)
    i = np.arange(n)
    s.add_particles(np.stack([i % 128, i // 128], 1).astype(np.float32))
    for d in range(1, chain + 1):
        a = np.arange(linked - d)
        s.add_particle_links(a, a + d, np.full(linked - d, 0.9 * d, np.float32))
    s.set_link_iterations(2)
    o = to_oracle(s, 32)
    for _ in range(2):
        s.update(1.0 / 60.0)
        assert s.engine_used == BD_ENGINE_TILED
        assert o.update(1.0 / 60.0) == 0
    assert bits_equal(state(s), state(o)), first_diff(state(s), state(o))
