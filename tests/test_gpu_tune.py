"""The tuner where the tiles it times stop short of a trial."""
import numpy as np
import pytest

from helpers import gpu_params, v2ref

pytestmark = pytest.mark.gpu

TRIAL, WARM = 40, 8


def test_a_trial_runs_whole_where_tiles_outgrow_their_limits(monkeypatch):
    """60 x 60 in one tile of 4096 agents, which this population passes some
    43 iterations on, in the first trial: every trial still runs all of its
    iterations, and those it ran are the oracle's."""
    from oracle.pp_oracle import simulate
    from pphpc_amd import Batch
    monkeypatch.setenv("PPHPC_TILE", "1,0,60")
    print("[case] tune: tiles that stop", flush=True)
    d = v2ref(60, iters=100000)
    room = 4 * d["grid_xy"]
    with Batch(room, d["grid_xy"], 2, 15, device=0) as b:
        rid = b.add(gpu_params(d), 17, room)
        best = b.tune(TRIAL)
        assert b.tick > 0 and b.tick % (TRIAL + WARM) == 0, b.tick
        assert best["sec_per_tick"] > 0
        n = b.replica(rid)["steps"]
        assert n == b.tick
        ref = simulate(dict(d, iters=n), seed=17, capacity=room)
        assert np.array_equal(b.rows_array(rid), ref)
