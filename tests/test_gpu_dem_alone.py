"""A DEM step whose workgroups are not on the device together is done by one of them, with the same results.

With demStepWait below the clock's tick nobody counts as present, so every launch over several workgroups takes that
way; the per-sub-step launches (a save count that is never reached) are the oracle. After the first such steps the
handle takes those launches itself for a while, so a run holds both forms and the change between them.
"""
import numpy as np
import pytest

from test_gpu_dem_step import NEVER, _case, _same, _views

pytestmark = pytest.mark.gpu

CASES = [dict(count=129), dict(count=300, spring=True), dict(count=65, clumps=True, spring=True),
         dict(count=150, clumps=True, periodic=False, walls="ALL"), dict(count=200, periodic=False, walls="ALL"),
         dict(count=1000)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(f"{k}{v}" for k, v in c.items()))
def test_one_workgroup_does_the_step(case):
    from hybird_amd import runtime

    conf, rec, objects = _case(seed=11, **case)
    conf.demStepWait = 1
    print(f"[gpu dem alone] {case}", flush=True)
    contact = 0.0
    # one step alone, then the other launches; several steps in the queue before the host hears of the first
    for counts in ((1, 3), (20,)):
        alone = runtime.Simulation(conf, rec, objects)
        steps = runtime.Simulation(conf, rec, objects)
        steps.set_save_count(NEVER)
        if len(counts) > 1:
            _same(_views(alone), _views(steps), "after initialisation")
        for n in counts:
            alone.cycle(n)
            steps.cycle(n)
            a = _views(alone)
            _same(a, _views(steps), n)
            contact = max(contact, np.abs(a["e_forces"][:, 2:6]).max())
        print(f"[gpu dem alone] {alone.get('alone_steps')[0]:.0f} steps alone", flush=True)
        assert alone.get("alone_steps")[0] >= 1.0
        rebuilds = float(alone.get("rebuilds")[0])
        alone.close()
        steps.close()
    assert contact > 0.0 and rebuilds > 2.0


def test_steps_alone_follow_each_other_and_whole_ones(tmp_path):
    """Many steps in the queue before the host looks, then a restart of their state where everybody is present."""
    from hybird_amd import runtime

    conf, rec, _ = _case(seed=3, count=300, spring=True)
    print("[gpu dem alone] queue of steps", flush=True)
    whole = runtime.Simulation(conf, rec)
    conf.demStepWait = 1
    alone = runtime.Simulation(conf, rec)
    path = str(tmp_path / "state")
    for k in range(3):
        whole.save_state(path)
        alone.load_state(path)
        whole.cycle(4)
        alone.cycle(4)
        a, b = _views(alone), _views(whole)
        _same(a, b, k)
        alone.save_state(path)
        whole.load_state(path)
        whole.cycle(2)
        alone.cycle(2)
        _same(_views(alone), _views(whole), (k, "after loading"))
    assert whole.get("alone_steps")[0] == 0.0
    whole.close()
    alone.close()


def test_negative_wait_takes_the_launches_of_a_sub_step():
    from hybird_amd import runtime

    conf, rec, _ = _case(seed=5, count=300)
    whole = runtime.Simulation(conf, rec)
    conf.demStepWait = -1
    apart = runtime.Simulation(conf, rec)
    print("[gpu dem alone] negative wait", flush=True)
    for s in (whole, apart):
        s.cycle(12)
    _same(_views(apart), _views(whole), "negative wait")
    assert apart.get("alone_steps")[0] == 0.0 and whole.get("alone_steps")[0] == 0.0
    whole.close()
    apart.close()
