"""Handles initialised again, from another DEM handle or unsuccessfully.

An initialisation gives the buffers of the one before back as a whole. What the next one does not set must be
gone as well: it would point into memory that is no longer the handle's.
"""
import ctypes as C

import numpy as np
import pytest

from helpers import fixture_config, load_case

pytestmark = pytest.mark.gpu

VIEWS = {"types": np.uint8, "f": np.float64, "n": np.float64, "mass": np.float64}


def _views(L, lb):
    out = {}
    for name, dtype in VIEWS.items():
        need = C.c_size_t(0)
        assert L.hyb_lb_get(lb, name.encode(), None, 0, C.byref(need)) == 0
        out[name] = np.empty(need.value // np.dtype(dtype).itemsize, dtype=dtype)
        assert L.hyb_lb_get(lb, name.encode(), out[name].ctypes.data, need.value, C.byref(need)) == 0
    return out


@pytest.mark.parametrize("precision", ["FP64", "FP32"])
def test_lattice_with_a_cylinder_initialised_again_without_one(precision):
    """The curved-wall rule belongs to the cylinder of the DEM handle: without that handle the lattice is the one
    of a new handle initialised without."""
    from hybird_amd import runtime

    L = runtime.load()
    cfg, rec, _ = load_case("net")
    conf = fixture_config(cfg, precision=precision)
    got = []
    for again in (True, False):
        print(f"[gpu reinit handles] net {precision}, cylinder first: {again}", flush=True)
        sim = runtime.Simulation(conf, rec) if again else None
        lb = sim._lb if again else C.c_void_p()
        if not again:
            assert L.hyb_lb_create(C.byref(conf), C.byref(lb)) == 0
        assert L.hyb_lb_init(lb, None) == 0
        for _ in range(4):
            assert L.hyb_lb_fs_step(lb) == 0 and L.hyb_lb_step(lb, None) == 0
        assert L.hyb_sync(lb) == 0
        got.append(_views(L, lb))
        if again:
            sim.close()
        else:
            assert L.hyb_lb_destroy(lb) == 0
    assert (got[0]["types"] == 3).any()
    for name, v in got[1].items():
        assert np.array_equal(got[0][name], v, equal_nan=v.dtype != np.uint8), name


def _bed_of_wide_spheres(L, runtime, conf, lb):
    """A DEM handle whose run-sum lists no device can hold: 300 spheres, the largest of radius 2,000."""
    from hybird_amd._abi import element_records

    rng = np.random.default_rng(3)
    r = np.full(300, 2.0)
    r[0] = 2000.0
    rec = element_records(rng.uniform(3.0, 7.0, (300, 3)), r)
    wide = type(conf)()
    C.memmove(C.byref(wide), C.byref(conf), C.sizeof(conf))
    wide.pairCapacity = 50_000
    dem = C.c_void_p()
    assert L.hyb_dem_create(C.byref(wide), len(rec), rec.ctypes.data, C.byref(dem)) == 0
    assert L.hyb_dem_init(dem, lb) == 0
    return dem


def test_lattice_whose_second_initialisation_fails():
    """The lattice is as before its first initialisation: every call on its state is refused, and it can be
    initialised again."""
    from hybird_amd import runtime
    from hybird_amd._abi import config_from_cfg, element_records
    from hybird_amd.cfg import base_config

    L = runtime.load()
    conf = config_from_cfg(base_config(lbSizeX=12, lbSizeY=11, lbSizeZ=13, boundary0=7, boundary1=7, boundary2=7,
                                       boundary3=7, lbFX=1.0e-5))
    rec = element_records(np.array([[5.0, 5.0, 6.0]]), np.array([2.2]))
    sim, new = runtime.Simulation(conf, rec), runtime.Simulation(conf, rec)
    print("[gpu reinit handles] lattice, second initialisation fails", flush=True)
    wide = _bed_of_wide_spheres(L, runtime, conf, sim._lb)
    assert L.hyb_lb_init(sim._lb, wide) == -2  # HYB_E_HIP
    new.step_lb(1)  # another handle's launch doesn't report the failed allocation again
    need = C.c_size_t(0)
    buf = np.zeros(8 * 19 * 12 * 11 * 13, dtype=np.uint8)
    state = -3  # HYB_E_STATE
    assert L.hyb_lb_step(sim._lb, sim._dem) == state
    assert L.hyb_lb_fs_step(sim._lb) == state
    assert L.hyb_lb_couple(sim._lb, sim._dem, None) == state
    assert L.hyb_lb_get(sim._lb, b"f", buf.ctypes.data, buf.nbytes, C.byref(need)) == state
    assert L.hyb_lb_set_force_field(sim._lb, buf.ctypes.data) == state
    assert L.hyb_lb_set_populations(sim._lb, buf.ctypes.data) == state
    assert L.hyb_adj_forward(sim._lb, sim._dem, 2, 1) == state
    assert L.hyb_state_save(sim._lb, None, b"/dev/null") == state
    assert L.hyb_lb_wall_fhydro_into(sim._lb, buf.ctypes.data, 18) == state
    assert L.hyb_lb_init(sim._lb, sim._dem) == 0
    sim.step_lb(3)
    new.step_lb(2)
    for name in ("types", "f", "u", "pflag"):
        v = new.get(name)
        assert np.array_equal(sim.get(name), v, equal_nan=v.dtype == np.float64), name
    assert L.hyb_dem_destroy(wide) == 0
    sim.close()
    new.close()


def test_dem_handle_whose_second_initialisation_fails():
    """Every call on the handle is refused, also from the lattice it is coupled to, and it can be initialised again."""
    from hybird_amd import runtime

    L = runtime.load()
    cfg, rec, _ = load_case("drum")
    conf = fixture_config(cfg)
    sim, new = runtime.Simulation(conf, rec), runtime.Simulation(conf, rec)
    print("[gpu reinit handles] DEM handle, second initialisation fails", flush=True)
    size = (C.c_int32 * 3)(*[int(np.floor(conf.lbSize[k] / conf.unitLength + 0.5)) for k in range(3)])
    rotating = (C.c_int32 * 6)(*conf.boundary)
    rotating[2] = 6  # the drum's rotating y walls are not supported
    init_args = [size, C.c_double(conf.unitLength), C.c_double(1.0e-4), C.c_double(conf.unitDensity), (C.c_double * 3)()]
    assert L.hyb_dem_init_lattice(sim._dem, rotating, *init_args) == -5  # HYB_E_UNSUPPORTED
    need = C.c_size_t(0)
    buf = np.zeros(1 << 20, dtype=np.uint8)
    state = -3  # HYB_E_STATE
    assert L.hyb_dem_step(sim._dem) == state
    assert L.hyb_dem_set_save_count(sim._dem, 1) == state
    assert L.hyb_dem_get(sim._dem, b"e_x", buf.ctypes.data, buf.nbytes, C.byref(need)) == state
    assert L.hyb_state_save(None, sim._dem, b"/dev/null") == state
    assert L.hyb_lb_init(sim._lb, sim._dem) == state
    assert L.hyb_lb_couple(sim._lb, sim._dem, None) == state
    assert L.hyb_lb_step(sim._lb, sim._dem) == state
    assert L.hyb_cycle(sim._lb, sim._dem, 1) == state
    assert L.hyb_dem_init(sim._dem, sim._lb) == 0 and L.hyb_lb_init(sim._lb, sim._dem) == 0
    for s in (sim, new):
        s.cycle(5)
    for name in ("types", "f", "e_x", "e_forces"):
        v = new.get(name)
        assert np.array_equal(sim.get(name), v, equal_nan=v.dtype == np.float64), name
    sim.close()
    new.close()
