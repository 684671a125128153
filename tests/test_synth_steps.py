"""The forcing generator at the tile counts where a thread changes from one
step to several: the values of a step do not depend on the count or on the
window, so any tile's row equals a window of that step alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("mp,steps", [(32767, 9), (32768, 9), (33001, 8)])
def test_a_step_is_the_same_in_any_window(mp, steps, precision):
    from cable_amd import gpu
    print(f"[synth steps] {mp} tiles, precision {precision}", flush=True)
    rng = np.random.default_rng(mp)
    t0, lat = rng.uniform(250.0, 305.0, mp), rng.uniform(-80.0, 80.0, mp)
    # a context of few tiles takes one step per thread; draws are keyed by the tile
    few = 300
    g, h = gpu.CableGPU(mp, precision), gpu.CableGPU(few, precision)
    g.set_tile_order(rng.permutation(mp))
    g.synth_forcing(3, steps, 11, t0, lat)
    h.synth_forcing(0, 20, 11, t0[:few], lat[:few])
    for k in (3, 2 + steps):
        a, b = g.download_forcing(k), h.download_forcing(k)
        for x, y in zip(a.values() if isinstance(a, dict) else a, b.values() if isinstance(b, dict) else b):
            np.testing.assert_array_equal(np.asarray(x)[:few], y)
    g.close()
    h.close()
