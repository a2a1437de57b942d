"""The TILED engine's own choice of tile size against the f32 oracle bit for bit:
both sides of the line to larger tiles, and a deep link graph."""
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
