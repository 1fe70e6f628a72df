"""Several threads reading one handle (an IO thread and a plot) each get their own values.

The views of a handle are packed into one device buffer, which grows with the largest one asked for; ctypes releases
the interpreter lock during a call, so the readers here really overlap.
"""
import threading

import numpy as np
import pytest

from helpers import fixture_config, load_case

pytestmark = pytest.mark.gpu

DEM_VIEWS = ("e_x", "e_w", "e_q", "e_forces", "p_data", "energy")
# sizes that make the buffer grow under the other readers
LB_VIEWS = ("pflag", "solidIndex", "mass", "visc", "u", "f", "n", "types")
ROUNDS = 60


def _read_together(make, names):
    alone = make()
    want = {n: alone.get(n) for n in names}
    alone.close()
    sim = make()
    wrong, gate = [], threading.Barrier(len(names))

    def reader(name):
        v = want[name]
        gate.wait()
        for k in range(ROUNDS):
            if not np.array_equal(sim.get(name), v, equal_nan=v.dtype == np.float64):
                wrong.append((name, k))
                return

    threads = [threading.Thread(target=reader, args=(n,)) for n in names]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    sim.close()
    assert not wrong, wrong


@pytest.mark.parametrize("names", [DEM_VIEWS, LB_VIEWS], ids=["elements", "lattice"])
def test_readers_of_one_handle(names):
    from hybird_amd import runtime

    cfg, rec, _ = load_case("dense")
    print(f"[gpu view threads] {names}", flush=True)

    def make():
        sim = runtime.Simulation(fixture_config(cfg), rec)
        sim.cycle(3)
        return sim

    _read_together(make, names)
