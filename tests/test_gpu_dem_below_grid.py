"""A particle below the cell grid near its first corner: its cell number falls among the particle slots, in front of the
cells. Every form of the neighbour rebuild reports it and touches no other memory."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wait", [0, -1, 1], ids=["one launch", "launches of a sub-step", "one workgroup"])
def test_particle_in_front_of_the_cells(wait):
    from hybird_amd import runtime
    from hybird_amd.cfg import base_config
    from hybird_amd._abi import config_from_cfg, element_records

    print(f"[gpu dem below grid] wait {wait}", flush=True)
    n = 150
    g = np.stack(np.meshgrid(np.arange(6), np.arange(5), np.arange(5), indexing="ij"), -1).reshape(-1, 3)
    x = 3.0 + 4.2 * g
    # cells of 5 x 0.4 x 2 = 4 units: 8 per axis and two more; floor(z / 4) = -1 and floor(y / 4) = 0 give cell
    # 10 (0 + 1 + 10 * -1 + 1) + 1 = -79, and with 150 slots in front of the cells the entry 71
    x[0] = (1.0, 1.0, -1.0)
    cfg = base_config(lbSolve=0, lbSizeX=32, lbSizeY=32, lbSizeZ=32, boundary0=7, boundary1=7, boundary2=7, boundary3=7,
                      boundary4=7, boundary5=7, density=2.5)
    conf = config_from_cfg(cfg)
    conf.demStepWait = wait
    sim = runtime.Simulation(conf, element_records(x, np.full(n, 0.8)))
    with pytest.raises(runtime.HybError, match="DEM device error 2") as e:
        sim.sync()
    assert e.value.code == -4
    sim.close()
