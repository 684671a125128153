"""A met window larger than the staging buffer goes up in parts: its steps have
the values that a window of each step alone gives, in any tile order."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("mp,steps", [(150001, 18), (2600000, 2)])
def test_a_window_in_parts(mp, steps, precision):
    from cable_amd import gpu
    print(f"[met window] {mp} tiles x {steps}, precision {precision}", flush=True)
    rng = np.random.default_rng(mp)
    f32 = lambda lo, hi: rng.uniform(lo, hi, (steps, mp)).astype(np.float32)  # noqa: E731
    met = {"swdown": f32(0, 900), "lwdown": f32(200, 400), "tair": f32(250, 310), "qair": f32(0.001, 0.02),
           "wind": f32(0.5, 9), "psurf": f32(9e4, 1e5), "rainf": f32(0, 1e-3),
           "tair_offset": 0.0, "psurf_scale": 0.01, "rainf_scale": 1800.0}
    lat = rng.uniform(-80, 80, mp)
    g = gpu.CableGPU(mp if precision else min(mp, 150001), precision)
    n = g.mp
    if n != mp:
        met = {k: v[:, :n].copy() if isinstance(v, np.ndarray) else v for k, v in met.items()}
        lat = lat[:n].copy()
    g.set_tile_order(rng.permutation(n))
    start = (0.0, 172, 6, 2001)
    g.set_met(0, steps, 1800.0, met, lat, start=start)
    ks = sorted({0, steps // 2, steps - 1})
    whole = {k: g.download_forcing(k) for k in ks}
    for k in ks:
        one = {q: v[k:k + 1].copy() if isinstance(v, np.ndarray) else v for q, v in met.items()}
        g.set_met(k, 1, 1800.0, one, lat, start=start)
        for name, x in g.download_forcing(k).items():
            np.testing.assert_array_equal(x, whole[k][name], err_msg=f"{name} step {k}")
    g.close()
