"""The DEM step in one launch against the per-sub-step kernels.

Without MercuryDPM saving a DEM step is one launch with the neighbour rebuilds
inside (dem_run.hip); with a save count set it is three launches per sub-step
(dem.hip), so a save count that is never reached selects those. Both do the
same operations in the same order: every view must agree bit for bit. Element
counts lie on both sides of the sizes where the launch changes (64 elements
per workgroup, one workgroup up to 128, or 64 with multi-sphere elements),
with more than 32 neighbours per element, rebuilds inside the run, and every
kind of contact partner.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NEVER = 10 ** 6
VIEWS = ("e_x", "e_xp", "e_q", "e_w", "e_forces", "e_misc", "p_data", "p_idx", "neighborTable", "nearWallTable",
         "ghostIndex", "ghostVec", "nearObjectTable", "objectForces", "walls", "dem_scalars", "rebuilds", "energy")


def _case(count, seed, periodic=True, spring=False, clumps=False, walls="FIRST"):
    from hybird_amd.cfg import base_config
    from hybird_amd._abi import config_from_cfg, element_records

    rng = np.random.default_rng(seed)
    small, big = 1.7, 2.0
    # a grid whose larger spheres overlap a little, in a box that grows with the count
    per_axis = int(np.ceil(count ** (1.0 / 3.0)))
    step = 3.8 * (1.7 if clumps else 1.0)
    X, Y, Z = (max(s, np.ceil(step * per_axis) + 5.0) for s in (18.0, 17.0, 21.0))
    grid = np.stack(np.meshgrid(*[np.arange(per_axis)] * 3, indexing="ij"), -1).reshape(-1, 3)[:count]
    x = 3.0 + (grid + 0.5) * step
    r = rng.uniform(small, big, count)
    v = rng.normal(0.0, 0.1, (count, 3))
    w = rng.normal(0.0, 0.05, (count, 3))
    n = rng.integers(1, 5, count) if clumps else None
    q = rng.normal(size=(count, 4))
    q = q / np.linalg.norm(q, axis=1)[:, None] if clumps else None
    side = 4 if periodic else 7
    cfg = base_config(lbSolve=0, lbSizeX=X, lbSizeY=Y, lbSizeZ=Z, lbFZ=-2.0e-4, lbFX=1.0e-4, boundary0=side,
                      boundary1=side, boundary2=side, boundary3=side, boundary4=7, boundary5=7, density=2.5,
                      youngMod=2.0e3, restitution=0.8, multiStep=13, wallContacts=walls,
                      tangentialModel="SPRING" if spring else "VISCOUS")
    objects = None
    if not periodic:
        from hybird_amd.particles import object_records
        # in the gaps between the spheres
        objects = object_records([[0.3 if clumps else 1.2, *[3.0 + k * step] * 3, 0.0, 0.0, 0.0] for k in (1, 2)])
    return config_from_cfg(cfg), element_records(x, r, v=v, size=n, w=w, q=q), objects


def _views(sim):
    return {k: sim.get(k).copy() for k in VIEWS}


def _same(a, b, what):
    for k in VIEWS:
        assert a[k].shape == b[k].shape and np.array_equal(a[k], b[k]), (what, k)


CASES = [dict(count=1), dict(count=17, spring=True), dict(count=64, periodic=False, walls="ALL"),
         dict(count=65), dict(count=128, spring=True, walls="ALL", periodic=False), dict(count=129),
         dict(count=300, spring=True), dict(count=64, clumps=True), dict(count=65, clumps=True, spring=True),
         dict(count=150, clumps=True, periodic=False, walls="ALL"), dict(count=1000)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(f"{k}{v}" for k, v in c.items()))
def test_one_launch_matches_the_sub_step_kernels(case):
    from hybird_amd import runtime

    conf, rec, objects = _case(seed=11, **case)
    print(f"[gpu dem step] {case}", flush=True)
    whole = runtime.Simulation(conf, rec, objects)
    steps = runtime.Simulation(conf, rec, objects)
    steps.set_save_count(NEVER)
    _same(_views(whole), _views(steps), "after initialisation")
    contact = 0.0
    for n in (1, 24):
        whole.cycle(n)
        steps.cycle(n)
        a = _views(whole)
        _same(a, _views(steps), n)
        contact = max(contact, np.abs(a["e_forces"][:, 2:6]).max())
    if case["count"] > 1:
        assert contact > 0.0
        assert float(whole.get("rebuilds")[0]) > 2.0
    # the two forms can follow each other on one handle
    whole.set_save_count(NEVER)
    steps.set_save_count(0)
    whole.cycle(3)
    steps.cycle(3)
    whole.set_save_count(0)
    whole.cycle(2)
    steps.cycle(2)
    _same(_views(whole), _views(steps), "after changing the form")
    whole.close()
    steps.close()


def test_many_neighbours_per_element():
    """More than 32 pairs of one element: the part of its list that is not kept on chip."""
    from hybird_amd import runtime
    from hybird_amd.cfg import base_config
    from hybird_amd._abi import config_from_cfg, element_records

    rng = np.random.default_rng(5)
    g = np.stack(np.meshgrid(*[np.arange(6)] * 3, indexing="ij"), -1).reshape(-1, 3)
    x = 2.0 + 1.6 * g
    r = np.full(len(x), 0.75)
    x = np.concatenate([x, [[6.0, 6.0, 16.0]]])
    r = np.concatenate([r, [2.5]])
    v = np.concatenate([rng.normal(0.0, 0.05, (len(g), 3)), [[0.0, 0.0, -0.2]]])
    for spring in ("VISCOUS", "SPRING"):
        cfg = base_config(lbSolve=0, lbSizeX=13, lbSizeY=13, lbSizeZ=24, boundary0=4, boundary1=4, boundary2=4,
                          boundary3=4, boundary4=7, boundary5=7, density=2.5, youngMod=2.0e2, multiStep=10,
                          tangentialModel=spring)
        conf, rec = config_from_cfg(cfg), element_records(x, r, v=v)
        conf.pairCapacity = 100_000
        print(f"[gpu dem step] many neighbours, {spring}", flush=True)
        whole, steps = runtime.Simulation(conf, rec), runtime.Simulation(conf, rec)
        steps.set_save_count(NEVER)
        whole.cycle(15)
        steps.cycle(15)
        a = _views(whole)
        t = a["neighborTable"].reshape(-1, 2)
        assert np.bincount(t.ravel()).max() > 64
        _same(a, _views(steps), spring)
        whole.close()
        steps.close()
