"""Circle-pair sweeps over active lists against the f32 oracle bit for bit:
piles whose round state and lists sit in LDS, in place of parked positions or
in the workspace, of one radius or several, slow and fast enough that circles
leave their margins (so sweeps are checked pair by pair, or run again wider)."""
import numpy as np
import pytest

from helpers import bits_equal, first_diff, state, to_oracle
from bendy2d_amd import Batch, Solver

pytestmark = pytest.mark.gpu

DT = 1.0 / 60.0
# bytes of LDS: none; a few circles' state; positions without previous ones;
# state in place of previous positions and lists in the workspace; all of it
BUDGETS = [0, 2048, 9 * 1024, 28 * 1024, 144 * 1024]


def pile(n, seed, mixed, speed):
    rng = np.random.default_rng(seed)
    cols = max(2, int(np.sqrt(n)))
    k = np.arange(n)
    c = np.zeros((n, 7), np.float32)
    c[:, 0] = 1.0 + 0.72 * (k % cols) + rng.uniform(-0.03, 0.03, n)
    c[:, 1] = 0.6 + 0.72 * (k // cols) + rng.uniform(-0.03, 0.03, n)
    c[:, 2:4] = c[:, 0:2] - speed * rng.standard_normal((n, 2)) * (DT / 4)
    c[:, 6] = rng.uniform(0.2, 0.5, n) if mixed else 0.35
    s = Solver()
    s.gravity, s.bounds = (0.0, -9.81), ((0.0, 0.0), (0.75 * cols + 2.0, 200.0))
    s.set_sub_steps(4)
    s.add_circles(c)
    return s


@pytest.mark.parametrize("lds", BUDGETS)
@pytest.mark.parametrize("mixed,speed", [(False, 0.5), (True, 2.0), (False, 60.0), (True, 200.0)])
def test_piles(lds, mixed, speed):
    scenes = [pile(n, 10 * n + int(speed), mixed, speed) for n in (2, 33, 65, 300, 1500)]
    oracles = [to_oracle(s, 32, candidate_mode=True) for s in scenes]
    b = Batch()
    for s in scenes:
        b.add_scene(s)
    b.config = dict(wg_small=128, wg_large=1024, split_points=1024, lds_small=lds, lds_large=lds,
                    steps_per_launch=2, use_graph=0, split_tiny=64, wg_tiny=64, lds_tiny=lds)
    b.update(DT, 4)
    b.sync()
    assert b.cc_stats()["err_scenes"] == 0
    for i, (s, o) in enumerate(zip(scenes, oracles)):
        for _ in range(4):
            assert o.update(DT) == 0
        b.read_scene(i, s)
        assert bits_equal(state(s), state(o)), f"scene {i}: {first_diff(state(s), state(o))}"


@pytest.mark.parametrize("n", [31, 32, 33, 34, 300])
def test_clump(n):
    # every circle touches every other: lists as long as the scene
    rng = np.random.default_rng(n)
    s = Solver()
    for _ in range(n):
        s.add_circle(rng.uniform(-0.3, 0.3, 2).astype(np.float32), 1.0)
    s.gravity, s.bounds = (0.0, 0.0), ((-1000.0, -1000.0), (2000.0, 2000.0))
    o = to_oracle(s, 32)
    for _ in range(3):
        s.update(DT)
        assert o.update(DT) == 0
    assert bits_equal(state(s), state(o)), first_diff(state(s), state(o))


@pytest.mark.parametrize("lds", [0, 144 * 1024])
@pytest.mark.parametrize("n,span", [(15, 3.0), (16, 3.0), (17, 40.0), (31, 6.0), (32, 1000.0), (700, 30.0), (2049, 90.0),
                                    (13312, 240.0), (13313, 240.0)])
def test_grid_edges(n, span, lds):
    # tables too small for separate rows of cells, the first that has them, and
    # the largest counters in LDS and the first of half as many; counters in LDS
    # and in memory; some circles fast enough to outlie (n = 2049: more than one
    # stage of a 128-lane workgroup holds) and one far away
    rng = np.random.default_rng(n)
    c = np.zeros((n, 7), np.float32)
    c[:, 0:2] = rng.uniform(0.0, span, (n, 2))
    speed = np.where(rng.uniform(size=n) < 0.1, 30.0, 2.0)[:, None]
    c[:, 2:4] = c[:, 0:2] - speed * rng.standard_normal((n, 2)) * (DT / 4)
    c[:, 6] = 0.35
    c[0, 0:4] += 5000.0
    s = Solver()
    s.gravity, s.bounds = (0.0, 0.0), ((-100.0, -100.0), (6000.0, 6000.0))
    s.set_sub_steps(4)
    s.add_circles(c)
    o = to_oracle(s, 32, candidate_mode=True)
    b = Batch()
    b.add_scene(s)
    b.config = dict(wg_small=128, wg_large=1024, split_points=4096, lds_small=lds, lds_large=lds, steps_per_launch=1,
                    use_graph=0, split_tiny=64, wg_tiny=64, lds_tiny=lds)
    b.update(DT, 2)
    b.sync()
    for _ in range(2):
        assert o.update(DT) == 0
    b.read_scene(0, s)
    assert bits_equal(state(s), state(o)), first_diff(state(s), state(o))


@pytest.mark.parametrize("n", [65, 300])
@pytest.mark.parametrize("speed", [20.0, 60.0])
def test_the_launches_do_not_change_the_schedule(n, speed):
    # what a scene has learnt (margins, and the sweeps since one was too small) is
    # kept between launches: the same rounds, sweeps run again and lists, a launch
    # for each update (4 sweeps) or for 16 of them
    def run(per_launch):
        b = Batch()
        s = pile(n, n, False, speed)
        b.add_scene(s)
        b.config = dict(steps_per_launch=per_launch)
        b.update(DT, 48)
        b.sync()
        st = b.scene_status(0)
        b.read_scene(0, s)
        assert b.cc_stats()["fallbacks"] == 0  # (a run of those ends with the launch)
        return state(s), st

    a, b = run(1), run(16)
    assert a[1]["redos"] > 0
    assert bits_equal(a[0], b[0]) and a[1] == b[1]


@pytest.mark.parametrize("n", [2, 100, 200, 400, 900, 2500])
def test_flight_that_outruns_its_lists(n):
    # circles far from each other, without a candidate pair, fast enough to leave
    # their skins every few sweeps: the sweep that has nothing to do and the one that
    # builds a new list follow each other, in workgroups of every size
    rng = np.random.default_rng(n)
    k = np.arange(n)
    c = np.zeros((n, 7), np.float32)
    c[:, 0:2] = 6.0 * np.stack([k % 50, k // 50], 1) + rng.uniform(-1.0, 1.0, (n, 2))
    c[:, 2:4] = c[:, 0:2] - 3.0 * rng.standard_normal((n, 2)) * (DT / 8)
    c[:, 6] = 0.35
    s = Solver()
    s.gravity, s.bounds = (0.0, 0.0), ((-50.0, -50.0), (500.0, 500.0))
    s.set_sub_steps(8)
    s.add_circles(c)
    o = to_oracle(s, 32, candidate_mode=True)
    for _ in range(12):
        s.update(DT)
        assert o.update(DT) == 0
    assert bits_equal(state(s), state(o)), first_diff(state(s), state(o))


@pytest.mark.parametrize("n", [1000, 4000])
def test_few_sweeps_run_twice(n):
    # a gas that falls into a heap, one update (4 sweeps) a launch: margins that are
    # too small again and again grow, and sweeps seldom have to run a second time
    rng = np.random.default_rng(n)
    box = np.sqrt(n * np.pi * 0.25 / 0.5)
    c = np.zeros((n, 7), np.float32)
    c[:, 0:2] = rng.uniform(0.5, box - 0.5, (n, 2))
    c[:, 2:4] = c[:, 0:2] - rng.standard_normal((n, 2)) * (DT / 4)
    c[:, 6] = 0.5
    s = Solver()
    s.gravity, s.bounds = (0.0, -20.0), ((0.0, 0.0), (box, box))
    s.set_sub_steps(4)
    s.add_circles(c)
    b = Batch()
    b.add_scene(s)
    for _ in range(60):
        b.update(DT, 1)
    b.sync()
    st = b.scene_status(0)
    assert st["err"] == 0 and st["redos"] <= 60 * 4 // 16
