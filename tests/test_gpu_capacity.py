"""What is left after an iteration whose agents are more than the capacity:
the run ends with PP_OUT_OF_RESOURCES at that iteration, which does not count,
and the state that can be read is the one before it, with the tiles laid out
and forced (PPHPC_TILE=shape,columns,rows)."""
import numpy as np
import pytest

from helpers import assert_state_equal, gpu_params, v2ref, v2s

pytestmark = pytest.mark.gpu

# 100, 141, 203, ... agents: 1558 after 9 iterations, 1854 after 10
GROWS = dict(v2ref(40, iters=500), init_sheep=100, init_wolves=0,
             sheep_reproduce_prob=40)
# 300 wolves who neither starve (but for one or two) nor reproduce
STAYS = dict(v2s(40, iters=500), init_sheep=0, init_wolves=300,
             wolves_gain_from_food=2000, wolves_reproduce_prob=0)
FAILS = 9

TILES = [None, "0,0,64", "0,0,3", "0,16,8"]
TILE_IDS = ["as laid out", "one tile", "tiles of three rows", "cut rows"]


def _states(d, seed, upto):
    """The oracle's states after 0 .. upto iterations, and their rows."""
    from oracle.pp_oracle import Oracle
    o = Oracle(d, seed=seed, capacity=1 << 22)
    states, rows = [o.state()], [o.stats()]
    for _ in range(upto):
        assert o.step() == 0
        states.append(o.state())
        rows.append(o.stats())
    o.close()
    return states, np.array(rows, np.uint64)


def _left(d, states, t):
    """The state that iteration t leaves when it fails: the one before it, in
    which the grass that it ate reads as alive (it is eaten in place; a cell
    so marked may have had a countdown of 1)."""
    cell, energy, typ, grass = states[t]
    ate = states[t + 1][3] == d["grass_restart"]
    assert (grass[ate] <= 1).all()
    return cell, energy, typ, np.where(ate, 0, grass).astype(np.uint32)


def _failing_batch():
    """A batch of two replicas whose agents exceed its capacity in iteration
    FAILS: reservations of what they hold before, which one outgrows by more
    than the other leaves."""
    from pphpc_amd import Batch
    ref = [_states(GROWS, 1, FAILS + 1), _states(STAYS, 2, FAILS + 1)]
    reserve = [len(r[0][FAILS][0]) for r in ref]
    assert sum(len(r[0][FAILS + 1][0]) for r in ref) > sum(reserve)
    b = Batch(sum(reserve), 3200, 2, 15, device=0)
    ids = [b.add(gpu_params(d), s, n) for d, s, n in
           ((GROWS, 1, reserve[0]), (STAYS, 2, reserve[1]))]
    return b, ids, ref


def _run_to_failure(run, pieces):
    from pphpc_amd import PP_OUT_OF_RESOURCES, PPError
    with pytest.raises(PPError) as e:
        for n in pieces:
            run(n)
    assert e.value.code == PP_OUT_OF_RESOURCES


@pytest.mark.parametrize("pieces", [[1] * 20, [60]], ids=["stepped", "one run"])
@pytest.mark.parametrize("tile", TILES, ids=TILE_IDS)
def test_a_failed_iteration_does_not_count(tile, pieces, monkeypatch):
    if tile:
        monkeypatch.setenv("PPHPC_TILE", tile)
    print(f"[case] failed iteration: {tile} {pieces[:2]}", flush=True)
    b, ids, ref = _failing_batch()
    with b:
        _run_to_failure(b.run, pieces)
        assert b.tick == FAILS
        _run_to_failure(b.run, [5])      # nothing runs any more
        assert b.tick == FAILS
        for rid, (_, rows) in zip(ids, ref):
            assert b.replica(rid)["steps"] == FAILS
            assert np.array_equal(b.rows_array(rid), rows[:FAILS + 1])


@pytest.mark.parametrize("pieces", [[1] * 20, [60]], ids=["stepped", "one run"])
@pytest.mark.parametrize("fails", [0, 2, 9])
@pytest.mark.parametrize("tile", TILES, ids=TILE_IDS)
def test_state_before_the_failed_iteration(tile, fails, pieces, monkeypatch):
    """fails 0: the staged iteration before the first of tiles; 2: a tile that
    is given no spare records in the iteration that fails. Changing the sort
    brings the agents into other forms; init starts anew."""
    from pphpc_amd import Simulation
    if tile:
        monkeypatch.setenv("PPHPC_TILE", tile)
    print(f"[case] state after failure: {tile} {fails} {pieces[:2]}", flush=True)
    states, rows = _states(GROWS, 1, fails + 1)
    cap = len(states[fails][0])
    assert len(states[fails + 1][0]) > cap
    left = _left(GROWS, states, fails)
    with Simulation(gpu_params(GROWS), seed=1, capacity=cap, device=0) as sim:
        for _ in range(2):
            sim.init()
            _run_to_failure(sim.run, pieces)
            assert sim.step_count == fails
            assert_state_equal(sim.state(), left, "failed")
            for mode in (0, 1):
                sim.set_sort(mode)
                assert_state_equal(sim.state(), left, f"sort {mode}")
                _run_to_failure(sim.run, [2])
            assert_state_equal(sim.state(), left, "run again")
        sim.init()
        assert np.array_equal(sim.run_array(fails), rows[1:fails + 1])
        assert_state_equal(sim.state(), states[fails], "up to the failure")


@pytest.mark.parametrize("pieces", [[1] * 20, [60]], ids=["stepped", "one run"])
@pytest.mark.parametrize("tile", TILES, ids=TILE_IDS)
def test_states_of_a_failed_batch(tile, pieces, monkeypatch):
    if tile:
        monkeypatch.setenv("PPHPC_TILE", tile)
    print(f"[case] states of a failed batch: {tile} {pieces[:2]}", flush=True)
    b, ids, ref = _failing_batch()
    with b:
        _run_to_failure(b.run, pieces)
        for _ in range(2):
            for rid, d, (states, _) in zip(ids, (GROWS, STAYS), ref):
                assert_state_equal(b.state(rid), _left(d, states, FAILS),
                                   f"replica {rid}")
            assert b.add(gpu_params(STAYS), 3, 300) is None
            b.set_sort(0)


@pytest.mark.parametrize("tile", [None, "0,16,8"], ids=["as laid out", "cut rows"])
def test_grass_when_the_failed_iteration_renews_its_ticks(tile, monkeypatch):
    """The tiles store the tick anew in live cells at every 32nd iteration:
    also of these the state before stays readable."""
    from pphpc_amd import Simulation
    if tile:
        monkeypatch.setenv("PPHPC_TILE", tile)
    print(f"[case] renewed grass: {tile}", flush=True)
    d = v2ref(60, iters=100)
    for fails in (31, 32, 33, 64):
        states, _ = _states(d, 17, fails + 1)
        cap = len(states[fails][0])
        assert max(len(s[0]) for s in states[:-1]) == cap < len(states[-1][0])
        with Simulation(gpu_params(d), seed=17, capacity=cap, device=0) as sim:
            sim.init()
            _run_to_failure(sim.run, [90])
            assert sim.step_count == fails
            assert_state_equal(sim.state(), _left(d, states, fails), f"{fails}")
