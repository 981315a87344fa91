"""Admissions while replicas hold their agents in tiles."""
import numpy as np
import pytest

from helpers import gpu_params, v1, v2s

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("short", ["agents", "cells", "slots"])
def test_a_refused_admission_leaves_the_tiles(short):
    """A batch without room for another replica stays in its tiles, and its
    replicas' rows are the oracle's."""
    from oracle.pp_oracle import simulate
    from pphpc_amd import Batch
    print(f"[case] refused admission: {short}", flush=True)
    ds = [(v2s(64, iters=60), 1), (v1(gx=50, gy=70, iters=50), 2)]
    room = [3 * d["grid_xy"] for d, _ in ds]
    cells = sum(d["grid_xy"] for d, _ in ds)
    more = v2s(32, iters=40)
    want = 3 * more["grid_xy"]
    with Batch(sum(room) + (want - 1 if short == "agents" else want),
               cells + (more["grid_xy"] - 1 if short == "cells" else 4096),
               2 if short == "slots" else 3, 15, device=0) as b:
        ids = [b.add(gpu_params(d), s, r) for (d, s), r in zip(ds, room)]
        for n in (7, 1, 12, 25, 60):
            b.run(n)
            if b.replica(ids[0])["state"] == b.replica(ids[1])["state"] == 1:
                assert b.add(gpu_params(more), 9, want) is None
                assert b.tiles()["in_use"] == 1
        for rid, (d, s), r in zip(ids, ds, room):
            assert np.array_equal(b.rows_array(rid), simulate(d, seed=s, capacity=r))
        rid = b.add(gpu_params(more), 9, want)
        b.run(40)
        assert np.array_equal(b.rows_array(rid), simulate(more, seed=9, capacity=want))


@pytest.mark.parametrize("sort", [1, 0])
def test_running_replicas_are_moved_by_one_launch(sort):
    """Twelve replicas of different sides in tiles, of which some end, then
    one more: one launch moves all agents for the iteration that sorts them."""
    from oracle.pp_oracle import simulate
    from pphpc_amd import Batch
    print(f"[case] one launch moves all: sort {sort}", flush=True)
    ds = [(v2s(gx=7 + 9 * i, gy=90 - 7 * i, iters=30 + 5 * (i % 4)), i) for i in range(12)]
    late = (v1(40, iters=30), 77)
    room = [3 * d["grid_xy"] + 8 for d, _ in ds + [late]]
    cells = sum(d["grid_xy"] for d, _ in ds + [late])
    with Batch(sum(room), cells, 13, 15, device=0) as b:
        ids = [b.add(gpu_params(d), s, r) for (d, s), r in zip(ds, room)]
        b.run(37)
        assert {b.replica(i)["state"] for i in ids} == {1, 2}
        assert b.tiles()["in_use"] == 1
        b.set_profiling(True)
        ids.append(b.add(gpu_params(late[0]), late[1], room[-1]))
        assert b.profile()["move0"][0] == 1
        b.set_profiling(False)
        b.set_sort(sort)
        b.run(40)
        for rid, (d, s), r in zip(ids, ds + [late], room):
            assert np.array_equal(b.rows_array(rid), simulate(d, seed=s, capacity=r)), s


def test_the_profile_names_what_is_launched():
    """Cells and agents are initialised by one kernel: one entry, no empty
    one."""
    from pphpc_amd import Simulation
    with Simulation(gpu_params(v2s(64)), seed=1, capacity=12000, device=0) as sim:
        sim.set_profiling(True)
        sim.init()
        p = {k: n for k, (n, _) in sim.profile().items() if k.startswith("init") or k == "move0"}
        assert p == {"init_reset": 2, "init": 1, "init_done": 1, "move0": 1}


def test_tables_larger_than_the_pinned_memory(monkeypatch):
    """24,000 tiles of one row: their table is copied in one piece, not from
    the handle's pinned memory; the next admission's tables are."""
    from oracle.pp_oracle import simulate
    from pphpc_amd import Batch
    monkeypatch.setenv("PPHPC_TILE", "0,0,1")
    print("[case] large tables", flush=True)
    ds = [(v2s(gx=4, gy=8000, iters=40), 1), (v1(gx=5, gy=16000, iters=60), 2),
          (v2s(gx=9, gy=70, iters=15), 3)]
    room = [2 * d["grid_xy"] for d, _ in ds]
    # (the tiles' tables lie in those of the cells' buckets)
    with Batch(sum(room), 1 << 23, 3, 15, device=0) as b:
        ids = [b.add(gpu_params(d), s, r) for (d, s), r in zip(ds[:2], room)]
        b.run(20)
        assert b.tiles()["tiles"] == 24000 and b.tiles()["in_use"] == 1
        ids.append(b.add(gpu_params(ds[2][0]), ds[2][1], room[2]))
        b.run(60)
        for rid, (d, s), r in zip(ids, ds, room):
            assert np.array_equal(b.rows_array(rid), simulate(d, seed=s, capacity=r)), s
