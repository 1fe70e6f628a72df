"""Free surface against walls whose links the mass pass takes one at a time: slip and moving slip walls beside plain
ones, on sizes that fill no wavefront of the interface list, compared with the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CYCLES = 40


@pytest.mark.parametrize("sides", [(6, 7), (7, 5), (6, 8), (5, 6)], ids=lambda s: f"x{s[0]}y{s[1]}")
def test_surface_between_slip_walls(sides):
    from hybird_amd import runtime
    from hybird_amd.cfg import base_config
    from hybird_amd._abi import config_from_cfg, element_records
    from oracle.oracle import OracleSim
    print(f"[gpu slip surface] boundaries {sides}", flush=True)
    x, y = sides
    cfg = base_config(problemName="LIQUID_BOX", freeSurfaceSolve=1, lbSizeX=23, lbSizeY=13, lbSizeZ=19, initVisc=0.05,
                      lbFX=2.0e-4, lbFY=1.0e-4, lbFZ=-4.0e-4, boundary0=x, boundary1=x, boundary2=y, boundary3=y,
                      boundary4=7, boundary5=7, density=2.5, slipCoefficient=0.4)
    conf = config_from_cfg(cfg, liquid_box=(1, 12, 1, 11, 1, 11))
    rec = element_records(np.array([[6.0, 6.0, 5.0]]), np.array([2.2]))
    gpu, orc = runtime.Simulation(conf, rec), OracleSim(conf, rec)
    start = gpu.get("types").copy()
    gpu.cycle(CYCLES)
    orc.cycle(CYCLES)
    types = gpu.get("types").reshape(-1)
    assert (types != start.reshape(-1)).any(), "the interface must move"
    assert np.array_equal(types, np.asarray(orc.get("types")).reshape(-1))
    itf = types == 3
    a, b = gpu.get("mass").reshape(-1)[itf], np.asarray(orc.get("mass")).reshape(-1)[itf]
    # the oracle adds the surplus in list order, the device exactly: a few hundred roundings of 2^-53 a pass
    assert np.linalg.norm(a - b) <= 1.0e-9 * np.linalg.norm(b)
    gpu.close()
