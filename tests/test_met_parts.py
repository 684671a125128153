"""A met window's way through the staging buffer's two halves, the third part
and later waiting for a half to be free: every step has the values of a window of
that step alone, in FP64 as in mixed precision, with and without the optional
variables; and the buffer stays small beside the window."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

START = (0.0, 172, 6, 2001)


def _met(n, steps, optional, seed):
    rng = np.random.default_rng(seed)
    f32 = lambda lo, hi: rng.uniform(lo, hi, (steps, n)).astype(np.float32)  # noqa: E731
    met = {"swdown": f32(0, 900), "tair": f32(250, 310), "qair": f32(0.001, 0.02), "wind": f32(0.5, 9),
           "rainf": f32(0, 1e-3), "tair_offset": 0.0, "psurf_scale": 0.01, "rainf_scale": 1800.0}
    if "lwdown" in optional:
        met["lwdown"] = f32(200, 400)
    if "wind_e" in optional:
        met["wind_e"] = f32(-5, 5)
    if "psurf" in optional:
        met["psurf"] = f32(9e4, 1e5)
    elevation = None if "psurf" in optional else rng.uniform(0, 3000, n)
    return met, rng.uniform(-80, 80, n), elevation, rng.permutation(n)


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("optional", [(), ("lwdown", "wind_e", "psurf")], ids=["required", "all"])
@pytest.mark.parametrize("n,steps", [(30011, 65), (300007, 9), (2100001, 4)])
def test_a_window_in_halves(n, steps, optional, precision):
    from cable_amd import gpu
    if n > 1000000 and precision == 0:
        n = 1100001                                  # two steps a part would not fit: one
    print(f"[met parts] {n} tiles x {steps}, precision {precision}, {optional}", flush=True)
    met, lat, elevation, order = _met(n, steps, optional, n)
    vars_ = sum(isinstance(v, np.ndarray) for v in met.values())
    assert vars_ * 4 * n * steps > 2 * (8 << 20), "three parts"
    g = gpu.CableGPU(n, precision)
    g.set_tile_order(order)
    g.set_met(0, steps, 1800.0, met, lat, elevation=elevation, start=START)
    ks = sorted({0, 1, steps // 2, steps - 2, steps - 1})
    whole = {k: g.download_forcing(k) for k in ks}
    for k in ks:
        one = {q: v[k:k + 1].copy() if isinstance(v, np.ndarray) else v for q, v in met.items()}
        g.set_met(k, 1, 1800.0, one, lat, elevation=elevation, start=START)
        for name, x in g.download_forcing(k).items():
            np.testing.assert_array_equal(x, whole[k][name], err_msg=f"{name} step {k}")
    g.close()


def _free_device_memory():
    from cable_amd import gpu
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert gpu.lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0   # the runtime it is linked with
    return free.value


def test_a_window_takes_little_staging_memory():
    from cable_amd import gpu
    print("[met parts] staging memory", flush=True)
    n, steps = 131072, 64
    met, lat, _, _ = _met(n, steps, ("lwdown", "psurf"), 1)
    g = gpu.CableGPU(n, 1)
    g.sync()
    free = _free_device_memory()
    g.set_met(0, steps, 1800.0, met, lat, start=START)
    taken = free - _free_device_memory() - 8 * 4 * n * steps
    g.close()
    # two halves, the latitudes and the allocator's rounding of nine buffers
    assert taken <= 2 * (8 << 20) + 8 * n + 9 * (2 << 20), taken
