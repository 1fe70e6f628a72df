"""The differentiated forward run leaves the element forces of its last step, as the same steps one by one do."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("steps,every", [(1, 1), (7, 3)])
def test_element_forces_after_the_forward_run(steps, every):
    from hybird_amd import runtime
    from hybird_amd.cfg import base_config
    from hybird_amd._abi import config_from_cfg, element_records

    cfg = base_config(lbSizeX=21, lbSizeY=19, lbSizeZ=17, initVisc=0.1, lbFX=1.0e-5, boundary0=4, boundary1=4,
                      boundary2=4, boundary3=4, boundary4=7, boundary5=7, density=2.5)
    # the first sphere has periodic copies, the second touches the bottom wall
    x, v = np.array([[1.5, 9.0, 8.0], [12.0, 9.0, 3.0]]), np.array([[0.01, 0.0, 0.002], [0.0, -0.01, 0.0]])
    out = []
    for forward in (True, False):
        print(f"[gpu adjoint forward] {steps} steps, forward run: {forward}", flush=True)
        sim = runtime.Simulation(config_from_cfg(cfg, precision="FP64"), element_records(x, np.array([2.5, 2.0]), v=v))
        if forward:
            sim.adj_forward(steps, every)
        else:
            sim.step_lb(steps)
        out.append({k: sim.get(k).copy() for k in ("e_forces", "f")})
        sim.close()
    assert np.abs(out[0]["e_forces"][:, 0]).max() > 0.0
    for k, a in out[0].items():
        assert np.array_equal(a, out[1][k], equal_nan=True), k
