"""The tile step (pp_tile.h): statistics rows and the whole state equal the
oracle's at the sizes where its tiles, borders and buffers can go wrong, for
both tile shapes (forced with PPHPC_TILE=shape,columns,rows; columns 0: whole
rows), and where it hands over to the staged step and back."""
import sys

import numpy as np
import pytest

from helpers import assert_state_equal, gpu_params, v1, v2ref, v2s

pytestmark = pytest.mark.gpu

DENSE = dict(v2ref(60), init_sheep=6000, init_wolves=300)   # up to 5 a cell

CASES = [
    # name, PPHPC_TILE (None: as laid out), parameters, iterations
    ("one tile", "0,0,64", v2s(64), 70),
    ("two tiles, each both neighbours of the other", "1,0,32", v2s(64), 70),
    ("last tile of one row", "0,0,8", v2s(gx=100, gy=41), 70),
    ("tiles of one row", "0,0,1", v2s(gx=60, gy=33), 70),
    ("a grid of one row", None, v2s(gx=257, gy=1), 60),
    ("a grid of one column", None, v2s(gx=1, gy=300), 60),
    ("more tiles than threads sum in a round", "0,0,1", v2s(gx=16, gy=600), 50),
    ("grass by words (odd width)", "0,0,5", v1(gx=101, gy=47), 120),
    ("cut rows, one column in the last tile", "0,16,8", v2s(gx=97, gy=30), 70),
    ("cut rows, two tiles a row", "0,64,16", v2s(gx=100, gy=50), 70),
    ("cut rows, the larger shape", "1,256,32", v2s(gx=700, gy=90), 40),
    ("widest uncut rows", None, v2s(gx=2048, gy=24), 40),
    ("narrowest cut rows", None, v2s(gx=2049, gy=24), 40),
    ("two-byte grass", None, dict(v2s(90), grass_restart=300), 70),
    ("two-byte grass, cut rows", "0,32,16", dict(v2s(90), grass_restart=300), 70),
    ("four-byte grass", None, dict(v2s(60), grass_restart=70000), 40),
    ("cells of many agents", "0,0,4", DENSE, 40),
    ("tiles that outgrow their limits", "1,0,60", v2ref(60), 90),
    ("records in the spare part", "0,0,4", v2s(40), 40),
    ("crowded edge cells", "0,16,16", DENSE, 40),
]


def _capacity(name, d, iters):
    n0 = d["init_sheep"] + d["init_wolves"]
    if name.startswith("records"):
        # just what the run needs: slots for half of it
        from oracle.pp_oracle import simulate
        rows = simulate(dict(d, iters=iters + 3), seed=17, capacity=20 * n0)
        return int((rows[:, 0] + rows[:, 1]).max())
    return max(6 * n0, 3 * d["grid_x"] * d["grid_y"])


@pytest.mark.parametrize("name,tile,d,iters", CASES, ids=[c[0] for c in CASES])
def test_tiles_match_oracle(name, tile, d, iters, monkeypatch):
    from oracle.pp_oracle import Oracle
    from pphpc_amd import Simulation
    if tile:
        monkeypatch.setenv("PPHPC_TILE", tile)
    print(f"[case] tiles: {name}", flush=True)
    cap = _capacity(name, d, iters)
    o = Oracle(d, seed=17, capacity=cap)
    with Simulation(gpu_params(d), seed=17, capacity=cap, device=0) as sim:
        assert sim.init().as_tuple() == o.stats()
        rc, ref = o.run(iters)
        assert rc == 0
        rows = sim.run_array(iters)
        bad = np.nonzero((rows != ref).any(axis=1))[0]
        assert len(bad) == 0, (int(bad[0]), rows[bad[0]], ref[bad[0]])
        assert_state_equal(sim.state(), o.state(), name)
        for _ in range(3):                  # odd and even record buffers
            assert sim.step().as_tuple() == (o.step(), o.stats())[1]
        assert_state_equal(sim.state(), o.state(), name + ", stepped")
    o.close()


def test_handing_over_to_the_staged_step_and_back():
    """Tiles, then the radix sort, tiles, profiled (staged) launches, tiles,
    row buckets, tiles: every row and the state in between."""
    from oracle.pp_oracle import Oracle
    from pphpc_amd import Simulation
    d = v2s(gx=150, gy=70)
    cap = 3 * d["grid_xy"]
    o = Oracle(d, seed=4, capacity=cap)
    with Simulation(gpu_params(d), seed=4, capacity=cap, device=0) as sim:
        sim.init()
        for n, change in ((13, lambda: sim.set_sort(0)), (9, lambda: sim.set_sort(1)),
                          (34, lambda: sim.set_profiling(True)),
                          (5, lambda: sim.set_profiling(False)),
                          (11, lambda: sim.set_sort(9)), (12, lambda: sim.set_sort(1)),
                          (40, lambda: None), (1, lambda: None)):
            rows = sim.run_array(n)
            rc, ref = o.run(n)
            assert rc == 0 and np.array_equal(rows, ref), n
            assert_state_equal(sim.state(), o.state(), f"after {n}")
            change()
    o.close()


@pytest.mark.parametrize("tile", [None, "0,32,16"], ids=["whole rows", "cut rows"])
def test_batch_of_tiles_admits_and_retires(tile, monkeypatch):
    """Replicas that end at different ticks, one that fails its reservation,
    and one admitted while the others hold their agents in tiles."""
    from oracle.pp_oracle import Oracle, simulate
    from pphpc_amd import Batch
    if tile:
        monkeypatch.setenv("PPHPC_TILE", tile)
    ds = [(v2s(64, iters=90), 1), (v1(gx=33, gy=70, iters=41), 2),
          (v2s(gx=100, gy=20, iters=140), 3)]
    late = (v2s(48, iters=60), 5)
    bad = dict(v2s(32, iters=300), sheep_reproduce_prob=60, wolves_reproduce_prob=40)
    small = (bad["init_sheep"] + bad["init_wolves"]) * 5 // 4
    room = lambda d: 3 * d["grid_xy"]   # noqa: E731
    cells = sum(d["grid_xy"] for d, _ in ds + [late]) + bad["grid_xy"]
    with Batch(3 * cells, cells, 8, 10, device=0) as b:
        ids = [b.add(gpu_params(d), s, room(d)) for d, s in ds]
        rb = b.add(gpu_params(bad), 9, small)
        b.run(25)
        o = Oracle(ds[2][0], seed=3, capacity=room(ds[2][0]))
        assert o.run(25)[0] == 0
        assert_state_equal(b.state(ids[2]), o.state(), "running replica")
        o.close()
        ids.append(b.add(gpu_params(late[0]), late[1], room(late[0])))
        b.run(400)
        for rid, (d, s) in zip(ids, ds + [late]):
            ref = simulate(d, seed=s, capacity=room(d))
            assert np.array_equal(b.rows_array(rid), ref), s
        o = Oracle(bad, seed=9, capacity=small)
        rc, ref = o.run(300)
        st = b.replica(rb)
        assert rc == -8 and st["state"] == 3 and st["error"] == -8
        assert st["steps"] == o.step_count
        assert np.array_equal(b.rows_array(rb)[1:], ref[:o.step_count])
        o.close()
    sys.stdout.flush()


LARGEST = [
    ("every cell of the shape", "2,0,128", v2s(128), 40),
    ("one tile and a last tile of one row", "2,0,40", v2s(gx=150, gy=41), 40),
    ("most slots in use", "2,0,60", DENSE, 30),
    ("two-byte grass", "2,0,90", dict(v2s(90), grass_restart=300), 40),
    ("as laid out", None, v2s(gx=2000, gy=520), 12),
]


@pytest.mark.parametrize("name,tile,d,iters", LARGEST, ids=[c[0] for c in LARGEST])
def test_largest_shape_matches_oracle(name, tile, d, iters, monkeypatch):
    test_tiles_match_oracle(name, tile, d, iters, monkeypatch)


@pytest.mark.parametrize("per_cell", [0.25, 0.34, 0.6])
def test_cut_rows_by_density(per_cell, monkeypatch):
    """Cut rows in the smaller and, from the density that fills it, the larger
    shape, as laid out."""
    d = v2s(gx=2100, gy=40)
    n0 = int(per_cell * d["grid_x"] * d["grid_y"])
    d.update(init_wolves=n0 // 10, init_sheep=n0 - n0 // 10)
    test_tiles_match_oracle(f"density {per_cell}", None, d, 24, monkeypatch)
