"""The device memory of a gradient: the states and gradients that it holds, and no slab that is left empty."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(128, 128, 112), (40, 40, 40)])  # a state larger than a slab, several states in one
def test_memory_of_the_forward_run(size):
    from hybird_amd import runtime
    from hybird_amd.cfg import base_config
    from hybird_amd._abi import config_from_cfg

    print(f"[gpu adjoint memory] {size}", flush=True)
    X, Y, Z = size
    cfg = base_config(lbSizeX=X, lbSizeY=Y, lbSizeZ=Z, initVisc=0.1, lbFX=1.0e-6)
    steps, every = 4, 2
    free = []
    sim = runtime.Simulation(config_from_cfg(cfg), np.zeros((0, 20)))
    for _ in range(2):  # the second run gives the first one's memory back
        sim.sync()
        free.append(torch.cuda.mem_get_info()[0])
        sim.adj_forward(steps, every)
        used = free[0] - torch.cuda.mem_get_info()[0]
        # two checkpoints, one interval's two states, two adjoint states, the force gradient; one partial sum of tau
        # per workgroup of at least 64 nodes; planes are padded by up to 511 nodes, allocations to 2 MiB
        n = X * Y * Z
        held = 6 * 19 * 8 * n + 3 * 8 * n
        spare = 6 * 19 * 8 * 511 + 8 * n // 32 + 8 * (2 << 20)
        assert held <= used + (8 << 20) and used <= held + spare, (used, held)
        sim.close()
        sim = runtime.Simulation(config_from_cfg(cfg), np.zeros((0, 20)))
    sim.close()
