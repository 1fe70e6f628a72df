"""Free surface over a lattice of several list-building workgroups.

The interface list is put in lattice order by workgroups of 4,096 nodes, 16 of
them per lane, every 16 passes, and regrouped by every pass: a lattice of 17 *
31 * 33 nodes (no multiple of either) is run past three orderings, in the plain form of the mass
pass and, with a slip wall, in the general one, and compared with the oracle.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CYCLES = 60


@pytest.mark.parametrize("side", [7, 5])
def test_interface_survives_its_orderings(side):
    from hybird_amd import runtime
    from hybird_amd.cfg import base_config
    from hybird_amd._abi import config_from_cfg, element_records
    from oracle.oracle import OracleSim
    print(f"[gpu interface list] boundary {side}", flush=True)
    cfg = base_config(problemName="LIQUID_BOX", freeSurfaceSolve=1, lbSizeX=17, lbSizeY=31, lbSizeZ=33, initVisc=0.05,
                      lbFX=2.0e-4, lbFZ=-4.0e-4, boundary0=side, boundary1=side, boundary2=side, boundary3=side,
                      boundary4=7, boundary5=7, density=2.5, slipCoefficient=0.4)
    conf = config_from_cfg(cfg, liquid_box=(1, 9, 1, 29, 1, 20))
    rec = element_records(np.array([[5.0, 15.0, 10.0]]), np.array([2.5]))
    gpu, orc = runtime.Simulation(conf, rec), OracleSim(conf, rec)
    start = gpu.get("types").copy()
    gpu.cycle(CYCLES)
    orc.cycle(CYCLES)
    types = gpu.get("types").reshape(-1)
    assert (types != start.reshape(-1)).sum() > 50, "the interface must move"
    assert np.array_equal(types, np.asarray(orc.get("types")).reshape(-1))
    itf = types == 3
    a, b = gpu.get("mass").reshape(-1)[itf], np.asarray(orc.get("mass")).reshape(-1)[itf]
    # the oracle adds the surplus in list order, the device exactly: a few hundred roundings of 2^-53 a pass
    assert np.linalg.norm(a - b) <= 1.0e-9 * np.linalg.norm(b)
    gpu.close()
