"""A lattice handle initialised again before its first step behaves as after one initialisation: its buffers are
given back as a whole, and every pointer into them is set again (cylinders with a free surface get theirs late)."""
import numpy as np
import pytest

from helpers import fixture_config, load_case

pytestmark = pytest.mark.gpu


def test_second_initialisation_of_a_lattice():
    from hybird_amd import runtime

    cfg, rec, _ = load_case("net")
    views = []
    for again in (False, True):
        print(f"[gpu reinit] net, initialised {'twice' if again else 'once'}", flush=True)
        sim = runtime.Simulation(fixture_config(cfg), rec)
        if again:
            assert runtime.load().hyb_lb_init(sim._lb, sim._dem) == 0
        sim.cycle(5)
        views.append({k: sim.get(k).copy() for k in ("types", "f", "mass", "e_x", "e_forces")})
        sim.close()
    for k, v in views[0].items():
        assert np.array_equal(v, views[1][k], equal_nan=v.dtype != np.uint8), k
