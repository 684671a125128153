"""The resident run's launches of several steps: the same bits as one launch
per step and as the consistency check's kernels, across a launch's largest
number of steps, at the edges of waves and workgroups."""
import numpy as np
import pytest

from cable_amd.fields import FIELDS

pytestmark = pytest.mark.gpu

NAMES = [f.name for f in FIELDS if f.role == "STATE"] + ["canopy%rnet", "canopy%fe", "canopy%fh", "canopy%fgpp",
                                                         "ssnow%runoff", "rad%trad"]


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("tiles,steps", [(1, 49), (64, 48), (65, 50), (257, 97), (1025, 47)])
def test_steps_of_one_launch_equal_single_steps(tiles, steps, precision):
    from cable_amd import gpu
    from cable_amd.workload import Workload, add_snow
    print(f"[run steps] {tiles} tiles x {steps}, precision {precision}", flush=True)
    wl = add_snow(Workload(tiles, 1, seed=tiles, forcing=False))
    out = []
    for how in ("run", "single", "checked", "split"):
        g = gpu.from_workload(wl, precision=precision, full=False)
        g.synth_forcing(0, steps, 5, wl.t0, wl.lat, dels=wl.dels)
        if how == "checked":
            g.consistency_check(True)
        if how == "single":
            for k in range(steps):
                g.run(k, 1, wl.dels)
        elif how == "split":
            g.run(0, 7, wl.dels)
            g.run(7, steps - 7, wl.dels)
        else:
            g.run(0, steps, wl.dels)
        out.append(g.download_fields(NAMES))
        g.close()
    for other in out[1:]:
        for n in NAMES:
            np.testing.assert_array_equal(out[0][n], other[n], err_msg=n)
