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
