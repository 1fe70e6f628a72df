"""DRUM has two y walls beside the six box planes: all eight are near-wall candidates, each with its own plane."""
import numpy as np
import pytest

from helpers import fixture_config, load_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wait", [0, -1], ids=["one launch", "launches of a sub-step"])
@pytest.mark.parametrize("copies", [1, 60])
def test_near_walls_of_the_drum(copies, wait):
    from hybird_amd import runtime

    cfg, rec, _ = load_case("drum")
    rec = np.tile(rec, (copies, 1))
    rng = np.random.default_rng(2)
    rec[:, 0] = np.arange(len(rec))
    rec[:, 3] = rng.uniform(0.4, 1.4, len(rec))
    rec[:, 4] = rng.uniform(0.06, 0.7, len(rec))
    rec[:, 5] = rng.uniform(0.3, 2.0, len(rec))
    conf = fixture_config(dict(cfg, wallContacts="ALL"))
    conf.demStepWait = wait
    conf.pairCapacity = 100_000
    print(f"[gpu drum walls] {len(rec)} elements, wait {wait}", flush=True)
    sim = runtime.Simulation(conf, rec)
    walls, reach = sim.get("walls"), sim.get("dem_scalars")[1]
    assert len(walls) == 8
    x = rec[:, 3:6]
    near = np.array([(x - w[:3]) @ w[3:6] < reach for w in walls]).T
    want = np.argwhere(near)
    assert (want[:, 1] >= 6).any()
    assert np.array_equal(sim.get("nearWallTable").reshape(-1, 2), want)
    sim.close()
