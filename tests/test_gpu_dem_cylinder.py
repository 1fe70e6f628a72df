"""Multi-sphere elements of several workgroups in a cylinder: the DEM step in one launch against the launches of a
sub-step, bit for bit, while elements touch the cylinder and each other."""
import numpy as np
import pytest

from test_gpu_dem_step import NEVER, _same, _views

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spring", [False, True], ids=["viscous", "spring"])
def test_clumps_in_a_cylinder(spring):
    from hybird_amd import runtime
    from hybird_amd.cfg import base_config
    from hybird_amd._abi import config_from_cfg, element_records

    rng = np.random.default_rng(9)
    # the cylinder lies along x through (4, 4) with radius 4
    gx, gy, gz = np.meshgrid(np.arange(12), np.arange(3), np.arange(3), indexing="ij")
    x = np.stack([2.0 + 1.5 * gx, 2.5 + 1.5 * gy, 2.5 + 1.5 * gz], -1).reshape(-1, 3)
    n = len(x)
    v = rng.normal(0.0, 0.05, (n, 3)) + 0.3 * (x - [11.0, 4.0, 4.0]) * [0.0, 1.0, 1.0]
    q = rng.normal(size=(n, 4))
    q /= np.linalg.norm(q, axis=1)[:, None]
    cfg = base_config(problemName="NET", lbSolve=0, freeSurfaceSolve=1, unitLength=0.5, unitTime=0.05, lbSizeX=22.0,
                      lbSizeY=9.0, lbSizeZ=9.0, boundary0=7, boundary1=7, boundary2=7, boundary3=7, boundary4=7,
                      boundary5=7, density=2.5, youngMod=2.0e3, restitution=0.8, multiStep=10,
                      tangentialModel="SPRING" if spring else "VISCOUS")
    conf = config_from_cfg(cfg)
    rec = element_records(x, rng.uniform(0.28, 0.32, n), v=v, size=rng.integers(1, 5, n), q=q)
    print(f"[gpu dem cylinder] {n} elements, spring {spring}", flush=True)
    whole, steps = runtime.Simulation(conf, rec), runtime.Simulation(conf, rec)
    steps.set_save_count(NEVER)
    wall = 0.0
    for k in (1, 40, 80):
        whole.cycle(k)
        steps.cycle(k)
        a = _views(whole)
        _same(a, _views(steps), k)
        wall = max(wall, np.abs(a["e_forces"][:, 4]).max())
    assert wall > 0.0
    assert whole.get("alone_steps")[0] == 0.0
    whole.close()
    steps.close()
