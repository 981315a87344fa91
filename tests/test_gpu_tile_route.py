"""The runs of the tile tests take the tile step, in the tiles that they ask
for (results alone do not tell: the staged step's are the same), and the
tiles that are to outgrow their limits, or their slots, do."""
import numpy as np
import pytest

from helpers import gpu_params, v1, v2ref, v2s
from test_gpu_tiles import CASES, LARGEST, _capacity

pytestmark = pytest.mark.gpu

SHAPES = [(256, 4096), (512, 8192), (1024, 16384)]   # threads, cells


def _asked(tile, d):
    """Threads, cut rows, columns and rows of the tiles that PPHPC_TILE asks
    for."""
    shape, columns, rows = (int(x) for x in tile.split(","))
    threads, cells = SHAPES[shape]
    if columns:
        pitch = 16
        while pitch < columns:
            pitch *= 2
        most = min(64, cells // pitch)
    else:
        most = cells // d["grid_x"]
    return threads, columns > 0, columns or d["grid_x"], min(rows, most, d["grid_y"])


@pytest.mark.parametrize("name,tile,d,iters", CASES + LARGEST,
                         ids=[c[0] for c in CASES + LARGEST])
def test_tiles_as_asked_for(name, tile, d, iters, monkeypatch):
    from pphpc_amd import Simulation
    if tile:
        monkeypatch.setenv("PPHPC_TILE", tile)
    print(f"[case] tile route: {name}", flush=True)
    with Simulation(gpu_params(d), seed=17, capacity=_capacity(name, d, iters),
                    device=0) as sim:
        sim.init()
        sim.run(2)
        t = sim.tiles()
        assert t["in_use"] == 1 and t["stops"] == 0, t
        if tile:
            threads, cut, w, h = _asked(tile, d)
            n = -(-d["grid_x"] // w) * -(-d["grid_y"] // h)
            assert (t["threads"], t["cut"], t["tiles"]) == (threads, cut, n), t
        sim.run(iters - 2)
        t = sim.tiles()
        if "outgrow" in name:
            assert t["stops"] > 0, t
        if "spare" in name:
            cell = sim.state()[0] // d["grid_x"]     # (whole rows)
            assert np.bincount(cell // h).max() > t["slot"], t


def test_a_batch_stops_in_mid_run(monkeypatch):
    """A replica outgrows its tile while another's stays as it is: both go
    on, from the iteration reached."""
    from oracle.pp_oracle import simulate
    from pphpc_amd import Batch
    monkeypatch.setenv("PPHPC_TILE", "1,0,60")
    print("[case] tile route: a batch stops", flush=True)
    ds = [(v2ref(60, iters=90), 17), (v1(60, iters=120), 3)]
    room = 4 * 3600
    with Batch(2 * room, 2 * 3600, 2, 15, device=0) as b:
        ids = [b.add(gpu_params(d), s, room) for d, s in ds]
        b.run(20)
        assert b.tiles()["in_use"] == 1 and b.tiles()["stops"] == 0
        b.run(60)
        assert b.tiles()["stops"] > 0
        b.run(40)
        for rid, (d, s) in zip(ids, ds):
            assert np.array_equal(b.rows_array(rid), simulate(d, seed=s, capacity=room))


def test_dense_populations_are_staged():
    from pphpc_amd import Simulation
    d = dict(v2s(100), init_sheep=300000, init_wolves=100)
    with Simulation(gpu_params(d), seed=1, capacity=2000000, device=0) as sim:
        sim.init()
        sim.run(3)
        assert sim.tiles() == dict(in_use=0, threads=0, cut=0, tiles=0, slot=0,
                                   stops=0)


@pytest.mark.parametrize("noalloc", [False, True], ids=["run", "without allocating"])
def test_runs_in_pieces_after_stops(noalloc):
    """A population that grows through several stops within one run: the
    iterations after each are enqueued piece by piece, to the last."""
    from oracle.pp_oracle import simulate
    from pphpc_amd import Simulation, simulate_noalloc
    d = v2ref(70, iters=500)
    room = 4 * d["grid_xy"]
    ref = simulate(d, seed=6, capacity=room)
    print(f"[case] tile route: pieces {noalloc}", flush=True)
    if noalloc:
        assert np.array_equal(simulate_noalloc(gpu_params(d), 6, room, device=0), ref)
        return
    with Simulation(gpu_params(d), seed=6, capacity=room, device=0) as sim:
        for _ in range(2):
            assert sim.init().as_tuple() == tuple(ref[0])
            assert np.array_equal(sim.run_array(500), ref[1:])
            assert sim.tiles()["stops"] > 1
