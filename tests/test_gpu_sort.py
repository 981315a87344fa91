"""The radix sort of every iteration (sort mode 0): rows and state equal the
oracle's with one pass, two and three, digits of up to 8 bits and of up to 11
(whose pairs lie side by side between the passes), both tile sizes, a part of
one tile and many."""
import pytest

from helpers import assert_state_equal, gpu_params, v2ref, v2s

pytestmark = pytest.mark.gpu

CASES = [
    # parameters, iterations: key bits
    (v2s(gx=9, gy=7), 20),                                 # 6: one pass
    (dict(v2ref(30), init_sheep=9000, init_wolves=90), 8),  # 10: one of 11 bits
    (v2s(gx=230, gy=190), 12),                             # 16: two of 8
    (v2s(gx=1100, gy=1000), 6),                            # 21: two of 11
    (v2s(gx=2100, gy=2050), 4),                            # 23: three of 8
]


@pytest.mark.parametrize("kpt", ["8", "16"])
@pytest.mark.parametrize("d,iters", CASES,
                         ids=["%dx%d" % (c[0]["grid_x"], c[0]["grid_y"]) for c in CASES])
def test_radix_matches_oracle(d, iters, kpt, monkeypatch):
    from oracle.pp_oracle import Oracle
    from pphpc_amd import Simulation
    monkeypatch.setenv("PPHPC_SORT_KPT", kpt)
    n0 = d["init_sheep"] + d["init_wolves"]
    cap = max(4 * n0, d["grid_x"] * d["grid_y"])
    print(f"[case] radix: {d['grid_x']} x {d['grid_y']}, {kpt}", flush=True)
    o = Oracle(d, seed=11, capacity=cap)
    with Simulation(gpu_params(d), seed=11, capacity=cap, device=0) as sim:
        sim.set_sort(0)
        assert sim.init().as_tuple() == o.stats()
        rc, ref = o.run(iters)
        assert rc == 0
        assert (sim.run_array(iters) == ref).all()
        assert_state_equal(sim.state(), o.state(), "radix")
    o.close()
