"""Steps of one, two and three sub-steps, where the form of a DEM step (one launch, or three per sub-step) depends on
their number, the elements and the springs: every view bit for bit that of the per-sub-step launches."""
import numpy as np
import pytest

from test_gpu_dem_step import NEVER, _case, _same, _views

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("multi", [1, 2, 3])
@pytest.mark.parametrize("case", [dict(count=64), dict(count=65), dict(count=64, spring=True),
                                  dict(count=200, spring=True), dict(count=65, clumps=True, spring=True)],
                         ids=lambda c: "-".join(f"{k}{v}" for k, v in c.items()))
def test_few_sub_steps(case, multi):
    from hybird_amd import runtime

    conf, rec, _ = _case(seed=7, **case)
    conf.unitTime *= multi / conf.multiStep  # the sub-step's length of that case
    conf.multiStep = multi
    print(f"[gpu dem few sub-steps] {case} {multi}", flush=True)
    sim, steps = runtime.Simulation(conf, rec), runtime.Simulation(conf, rec)
    steps.set_save_count(NEVER)
    for n in (1, 300 // multi):
        sim.cycle(n)
        steps.cycle(n)
        _same(_views(sim), _views(steps), n)
    assert float(sim.get("rebuilds")[0]) > 1.0
    assert np.abs(sim.get("e_forces")[:, 2:6]).max() > 0.0
    sim.close()
    steps.close()
