"""The work that programs have this framework do, as cases that can be timed.

A case is one pass through the public entry points: a whole simulation from
its seeded initial state (``Simulation.init`` + ``run`` or ``step``,
``simulate_noalloc``), or a batch of replicas from admission to its last row
(``Batch.add`` / ``run`` / ``rows_array``). ``prepare`` creates the handle,
which a program keeps over its runs; every pass starts again from iteration 0,
so passes on one state give the same outputs. Outputs are statistics rows
(sheep, wolves, live grass, energy sums, countdown sum per iteration) and, for
the cases that read the state back, every agent and cell: whole numbers
throughout.

The parameter sets are v1 (the reference's configs/config100v1.txt: sparse,
slow grass) and v2s (the dense set of the 1600 x 1600 benchmark), scaled with
the grid as pphpc_amd/workloads.py scales them.
"""
import math
import random

import numpy as np

from pphpc_amd import Batch, Params, Simulation, simulate_noalloc
from pphpc_amd.workloads import params_of, reserve_for, v1, v2s

# Grid sides of a heterogeneous batch (those of the batched workload up to
# 1600) and the iterations a pass of it runs.
MIXED_SIDES = (100, 200, 400, 800, 1600)


def listed():
    return [
        # An interactive program or a coupled model: the reference's 100 x 100
        # grid advanced one iteration per call, each row looked at.
        dict(name="step_100_v1", kind="step", set="v1", gx=100, gy=100, iters=64),
        # The reference's own configuration, whole: 4000 iterations.
        dict(name="plain_100_v1", kind="plain", set="v1", gx=100, gy=100,
             iters=4000),
        # A short run inside a loop that must not allocate (parameter search).
        dict(name="noalloc_200_v2s", kind="noalloc", set="v2s", gx=200, gy=200,
             iters=200),
        # Slow, rich grass (two-byte regrow ticks), odd sides, the state read
        # back at the end: a run that is checkpointed.
        dict(name="state_301x257_slow", kind="state", set="v1", gx=301, gy=257,
             iters=300, restart=200, gain=40),
        # An ordinary study grid.
        dict(name="plain_400_v2s", kind="plain", set="v2s", gx=400, gy=400,
             iters=1000),
        # Odd sides, sparse set, wider than high.
        dict(name="plain_1013x487_v1", kind="plain", set="v1", gx=1013, gy=487,
             iters=500),
        # The benchmark's grid and set.
        dict(name="plain_1600_v2s", kind="plain", set="v2s", gx=1600, gy=1600,
             iters=1000),
        # A wide grid (rows longer than 2048 cells), with every iteration
        # sorted by the radix sort, as the benchmark's bandwidth leg runs it.
        dict(name="radix_2400x1200_v2s", kind="plain", set="v2s", gx=2400,
             gy=1200, iters=60, sort=0),
        # Large and odd, sparse.
        dict(name="plain_4001x2999_v1", kind="plain", set="v1", gx=4001,
             gy=2999, iters=100),
        # The largest grid of the benchmark.
        dict(name="plain_12800_v2s", kind="plain", set="v2s", gx=12800,
             gy=12800, iters=24),
        # A study of many configurations: 48 replicas of mixed sides and sets
        # as one batch.
        dict(name="batch_48_mixed", kind="batch", n=48, side=0, iters=200,
             key=4),
        # Replicas for statistics: 30 of the benchmark's configuration.
        dict(name="batch_30x1600_v2s", kind="batch", n=30, side=1600,
             iters=60, key=0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges: sides over their logarithm from 64 to
    6400, both sets, iterations so that a pass stays below the largest listed
    one; batches of 2 to 40 replicas."""
    kind = rng.choice(["step", "plain", "plain", "plain", "state", "noalloc",
                       "batch"])
    pset = rng.choice(["v1", "v2s"])
    if kind == "batch":
        side = rng.choice([0, 0, _log_int(rng, 64, 1600)])
        n = rng.randint(2, 40)
        return dict(kind="batch", n=n, side=side, iters=rng.randint(20, 120),
                    key=rng.randint(5, 1 << 20), set=pset)
    if kind == "noalloc":
        gx, gy = _log_int(rng, 64, 500), _log_int(rng, 64, 500)
        return dict(kind=kind, set="v2s", gx=gx, gy=gy,
                    iters=rng.randint(20, 300))
    hi = {"step": 1600, "state": 1200, "plain": 6400}[kind]
    gx, gy = _log_int(rng, 64, hi), _log_int(rng, 64, hi)
    if kind == "step":
        return dict(kind=kind, set=pset, gx=gx, gy=gy, iters=rng.randint(8, 64))
    most = max(10, min(2000, 10 ** 9 // (gx * gy)))
    case = dict(kind=kind, set=pset, gx=gx, gy=gy,
                iters=rng.randint(max(5, most // 4), most))
    if kind == "state":
        case.update(rng.choice([{"restart": 5}, {"restart": 10}, {"restart": 30},
                                {"set": "v1", "restart": 200, "gain": 40}]))
    elif rng.random() < 0.15:
        case["sort"] = 0
    return case


def _params(case):
    make = v1 if case["set"] == "v1" else v2s
    d = make(iters=case["iters"], gx=case["gx"], gy=case["gy"])
    if case.get("restart"):
        d["grass_restart"] = case["restart"]
    if case.get("gain"):
        d["sheep_gain_from_food"] = case["gain"]
    return d


def _replicas(case):
    """(parameters, seed offset) of a batch's replicas."""
    rng = random.Random(case["key"])
    out = []
    for i in range(case["n"]):
        if case["side"]:
            kind, side = case.get("set", "v2s"), case["side"]
        else:
            kind, side = rng.choice(("v1", "v2s")), rng.choice(MIXED_SIDES)
        out.append((params_of(kind, side, case["iters"]), i))
    return out


def prepare(case, seed):
    if case["kind"] == "batch":
        reps = _replicas(case)
        agents = sum(reserve_for(d) for d, _ in reps)
        cells = sum(d["grid_xy"] for d, _ in reps)
        return {"kind": "batch", "iters": case["iters"],
                "batch": Batch(agents, cells, len(reps), 10, device=0),
                "reps": [(Params.from_values(**d), seed * 1000 + i,
                          reserve_for(d)) for d, i in reps]}
    d = _params(case)
    p = Params.from_values(**d)
    if case["kind"] == "noalloc":
        # (the fixed scratch holds 262,144 agents)
        cap = min(reserve_for(d), 1 << 18)
        return {"kind": "noalloc", "params": p, "seed": seed, "capacity": cap}
    sim = Simulation(p, seed=seed, capacity=reserve_for(d), device=0)
    if "sort" in case:
        sim.set_sort(case["sort"])
    return {"kind": case["kind"], "iters": case["iters"], "sim": sim,
            "capacity": reserve_for(d)}


def run(state):
    kind = state["kind"]
    if kind == "noalloc":
        return simulate_noalloc(state["params"], state["seed"],
                                state["capacity"], device=0)
    if kind == "batch":
        b = state["batch"]
        ids = [b.add(p, s, r) for p, s, r in state["reps"]]
        b.run(state["iters"])
        rows = [b.rows_array(rid) for rid in ids]
        for rid in ids:
            b.release(rid)
        return np.stack(rows)
    sim = state["sim"]
    row0 = sim.init()
    if kind == "step":
        rows = [row0] + [sim.step() for _ in range(state["iters"])]
        return np.array([r.as_tuple() for r in rows], np.uint64)
    rows = sim.run_array(state["iters"])
    if kind == "state":
        # a checkpoint of fixed size: the agents in arrays of the capacity
        cell, energy, typ, grass = sim.state()
        ck = np.zeros((3, state["capacity"]), np.int64)
        ck[0, :len(cell)], ck[1, :len(cell)], ck[2, :len(cell)] = \
            cell, energy, typ
        return rows, len(cell), ck, grass
    return rows


# Agents per cell that the two sets settle at (they start at 0.06 and 0.24).
_DENSITY = {"v1": 0.15, "v2s": 0.23}


def work(case):
    """Per iteration every agent's 8-byte record is read and its successor
    written, and the grass of its cell (one byte) read; about 100 integer
    operations per agent (the move's Philox block, the bounded draws, the
    action). Once per pass the initial agents and cells are drawn."""
    if case["kind"] == "batch":
        cells = {"v1": 0, "v2s": 0}
        for d, _ in _replicas(case):
            cells["v1" if d["grass_restart"] == 10 else "v2s"] += d["grid_xy"]
    else:
        cells = {case["set"]: case["gx"] * case["gy"]}
    n = sum(_DENSITY[k] * c for k, c in cells.items())
    c = sum(cells.values())
    it = case["iters"]
    return {"bytes": it * 17.0 * n + 8.0 * n + c, "flops": it * 100.0 * n + 80.0 * (n + c)}


def exact(case, seed):
    """Every output is a whole number, equal from version to version; none has
    a 64-bit value beside it."""
    return None
