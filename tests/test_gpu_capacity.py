"""What is left after an iteration whose agents are more than the capacity:
the run ends with PP_OUT_OF_RESOURCES at that iteration, which does not count,
with the tiles laid out and forced (PPHPC_TILE=shape,columns,rows)."""
import numpy as np
import pytest

from helpers import gpu_params, v2ref, v2s

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
