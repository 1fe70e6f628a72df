"""Host views and inputs larger than one packing range.

Views are packed and inputs unpacked on the device in ranges of up to 64 MiB:
the lattices here take several ranges (populations: 13 for FP64, 2 for FP32;
forces: 2), with odd sizes, so that the ranges end inside rows, and inactive
nodes, which read NaN.
"""
import numpy as np
import pytest

from adjoint_reference import W

pytestmark = pytest.mark.gpu


def _sim(size, precision):
    from hybird_amd import runtime
    from hybird_amd.cfg import base_config
    from hybird_amd._abi import config_from_cfg, element_records
    X, Y, Z = size
    cfg = base_config(lbSizeX=X, lbSizeY=Y, lbSizeZ=Z, initVisc=0.1, lbFX=0.0, lbFY=0.0, lbFZ=0.0, boundary0=4,
                      boundary1=4, boundary2=4, boundary3=4, boundary4=7, boundary5=7, density=2.5)
    rec = element_records(np.array([[30.0, 31.0, 20.0]]), np.array([3.0]))
    return runtime.Simulation(config_from_cfg(cfg, precision=precision), rec)


@pytest.mark.parametrize("precision,size", [("FP64", (181, 179, 175)), ("FP32", (97, 83, 71))])
def test_populations_and_forces_over_several_ranges(precision, size):
    print(f"[gpu views] {precision} {size}", flush=True)
    rng = np.random.default_rng(5)
    sim = _sim(size, precision)
    n = int(np.prod(size))
    types = sim.get("types").reshape(-1)
    act = (types == 0) | (types == 3)
    w = np.asarray(W, dtype=np.float64)
    f0 = w * (1.0 + 1.0e-3 * rng.standard_normal((n, 19), dtype=np.float32))
    sim.set_populations(f0)
    f = sim.get("f").reshape(-1, 19)
    # FP32 stores the deviation from the weights, rounded once
    want = f0 if precision == "FP64" else (f0 - w).astype(np.float32).astype(np.float64) + w
    assert np.array_equal(f[act], want[act])
    assert not act.all() and np.isnan(f[~act]).all()

    # from rest a collision sees u = F / 2: sum w = 1 and sum c w = 0 up to rounding of 19 terms below 1/3, and F
    # enters as float32 exactly; FP32 rounds F / 2 and a few operations of that size besides
    F = (1.0e-3 * rng.standard_normal((n, 3), dtype=np.float32)).astype(np.float32)
    sim.set_populations(np.broadcast_to(w, (n, 19)))
    sim.set_force_field(F)
    sim.step_lb(1)
    free = act & (sim.get("pflag").reshape(-1) == 0)
    u = sim.get("u").reshape(-1, 3)
    tol = 1.0e-14 if precision == "FP64" else 4 * 2.0 ** -24 * float(np.abs(F).max())
    assert np.abs(u[free] - 0.5 * F[free].astype(np.float64)).max() <= tol
    assert np.isnan(u[~act]).all()
    sim.close()


def test_views_into_unaligned_buffers():
    """A large view (whose pages are made present beforehand) writes its own bytes only, wherever the buffer starts."""
    import ctypes as C

    from hybird_amd import runtime
    size = (97, 83, 71)
    sim = _sim(size, "FP64")
    want = sim.get("u")
    n = want.nbytes
    assert n > 8 << 20
    for shift in (8, 4096 - 8, 4096):
        print(f"[gpu views] unaligned by {shift}", flush=True)
        raw = np.full(n + 3 * 4096, 0xA5, dtype=np.uint8)
        off = -raw.ctypes.data % 4096 + shift
        need = C.c_size_t(0)
        rc = runtime.load().hyb_lb_get(sim._lb, b"u", raw.ctypes.data + off, n, C.byref(need))
        assert rc == 0 and need.value == n
        assert np.array_equal(raw[off:off + n], want.reshape(-1).view(np.uint8))
        assert (raw[:off] == 0xA5).all() and (raw[off + n:] == 0xA5).all()
    sim.close()
