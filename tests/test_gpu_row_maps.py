"""Node-to-lane maps of the lattice kernels against a plain float64 step.

Which nodes a wavefront and a workgroup take depends on X: several rows of a
workgroup up to X = 64 and 128, one above, and another order of the workgroups
where rows do not end on 128-byte lines (multiples of 32 nodes in FP32, 16 in
FP64). Sizes lie on both sides of each of these, with rows and workgroups left
over, and the sphere lies across x = 64 where there is one.
"""
import numpy as np
import pytest
import torch

from adjoint_reference import Lattice

pytestmark = pytest.mark.gpu

TAU, MAGIC, STEPS = 0.8, 0.25, 3


@pytest.mark.parametrize("precision", ["FP64", "FP32"])
@pytest.mark.parametrize("X", [12, 31, 32, 48, 63, 64, 65, 96, 100, 128, 130, 192, 257, 320, 385])
def test_steps_match_the_reference_for_every_row_length(X, precision):
    from hybird_amd import runtime
    from hybird_amd.cfg import base_config
    from hybird_amd._abi import config_from_cfg, element_records
    size = (X, 11, 10)
    print(f"[gpu rows] {precision} {size}", flush=True)
    cfg = base_config(lbSizeX=X, lbSizeY=size[1], lbSizeZ=size[2], initVisc=(TAU - 0.5) / 3.0, lbFX=1.0e-5, lbFZ=0.0,
                      boundary0=4, boundary1=4, boundary2=4, boundary3=4, boundary4=7, boundary5=7, density=2.5)
    rec = element_records(np.array([[64.0 if X > 70 else X / 2.0, 5.3, 4.8]]), np.array([2.6]))
    sim = runtime.Simulation(config_from_cfg(cfg, collision="TRT", precision=precision, trt_magic=MAGIC), rec)
    types = sim.get("types").reshape(-1)
    act = (types == 0) | (types == 3)
    lat = Lattice(types, sim.get("pflag").reshape(-1).astype(bool) & act, size, (True, True, False))
    assert lat.pmask.sum() > 30, "the case must contain particle nodes"
    rng = np.random.default_rng(X)
    w = lat.w.numpy()[:, 0]
    f0 = w * (1.0 + 1.0e-3 * rng.standard_normal((act.size, 19)))
    sim.set_populations(f0)
    sim.step_lb(STEPS)
    F = torch.tensor([1.0e-5, 0.0, 0.0], dtype=torch.float64)[:, None].expand(3, lat.active.size)
    tau = torch.tensor(TAU, dtype=torch.float64)
    g = lat.to_active(f0)
    for _ in range(STEPS):
        before = g
        g = lat.stream(lat.collide(g, F, tau, MAGIC))
    n = before.sum(0)
    u = (lat.c @ before) / n
    force = (lat.pmask / n * u).sum(1).numpy()  # on the sphere at rest, node mass 1
    # the same operations up to their order: a few dozen roundings of 2^-53, or of 2^-24 on deviations of 1e-3 w
    tol = 1.0e-13 if precision == "FP64" else 1.0e-7
    got = lat.to_active(sim.get("f")).numpy()
    assert np.linalg.norm(got - g.numpy()) <= tol * np.linalg.norm(g.numpy())
    assert np.abs(sim.get("e_forces").reshape(-1)[:3] - force).max() <= tol * lat.pmask.sum()
    sim.close()
